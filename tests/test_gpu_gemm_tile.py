"""GPU parity of the prompt-bucket product (solort_gemm_tile) and of the launch that adds its k shares
(solort_add_parts_rmsnorm).

Bar of the products as in test_gpu_gemm_rows.py: within four bf16 ulps (2^-6 relative) plus 2e-3 of the
fp64 value on the same bf16 inputs, mean relative error <= 2e-3; the fp32 shares, which are not rounded,
sum to within 1e-5 of the product of the absolute values (k 2^-24 at most, usually sqrt(k) 2^-24)."""
from __future__ import annotations

import pytest
import torch

from solort_amd import ops

from test_gpu_gemm_rows import _close, _lin, _wide

pytestmark = pytest.mark.gpu


def _inputs(m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    return (torch.randn(m, k, generator=g).to(torch.bfloat16), (torch.randn(n, k, generator=g) * 0.02).to(torch.bfloat16))


# m: one row, the edges of the 32, 64, 128 and 256 row tiles; n: below one tile, ragged, more tiles than CUs; k: the
# smallest, step counts of every remainder by the buffers
SHAPES = [(1, 4, 512), (17, 68, 640), (32, 1004, 768), (33, 8224, 512), (64, 100, 2560), (65, 36, 896), (100, 6144, 2560),
          (128, 196, 1024), (129, 68, 1152), (256, 4096, 1024), (257, 132, 640), (1000, 260, 512)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_gemm_tile_plain_and_parts(gpu, m, n, k):
    print(f"[gemm_tile m={m} n={n} k={k}]", flush=True)
    x, w = _inputs(m, n, k)
    xd, wd = _wide(x, gpu, 8), _wide(w, gpu, 16)
    out = _wide(torch.zeros(m, n, dtype=torch.bfloat16), gpu, 4)
    ops.gemm_tile(wd, xd, out)
    _close(out, _lin(x, w))
    assert (out._base[:, n:] == 7).all()
    exact = x.double() @ w.double().t()
    bound = x.double().abs() @ w.double().abs().t() * 1e-5
    for s in {1, ops.gemm_tile_parts(m, n, k), k // 256}:
        parts = torch.full((s, m, n), 9.0, device=gpu)
        ops.gemm_tile(wd, xd, parts, mode=ops.TILE_PARTS)
        assert ((parts.double().sum(0).cpu() - exact).abs() <= bound).all()


@pytest.mark.parametrize("m,n,inter,k", [(17, 20, 24, 512), (64, 3072, 3072, 1024), (128, 9728, 9728, 512), (32, 9728, 9728, 512),
                                         (50, 6200, 6208, 640), (100, 52, 52, 768), (200, 6148, 6160, 512), (300, 40, 40, 640),
                                         (1000, 164, 168, 896), (513, 480, 480, 512)])
def test_gemm_tile_swiglu(gpu, m, n, inter, k):
    print(f"[gemm_tile swiglu m={m} n={n} k={k}]", flush=True)
    x, w = _inputs(m, inter + n, k)
    gate, up = _lin(x, w[:n]).double(), _lin(x, w[inter:]).double()
    out = torch.empty(m, n, dtype=torch.bfloat16, device=gpu)
    ops.gemm_tile(w.to(gpu), x.to(gpu), out, mode=ops.TILE_SWIGLU, inter=inter)
    _close(out, (gate * torch.sigmoid(gate)).to(torch.bfloat16).double() * up)


@pytest.mark.parametrize("m,k,n_parts", [(1, 8, 1), (5, 2560, 6), (33, 4096, 3), (3, 4104, 5), (2, 8192, 16)])
@pytest.mark.parametrize("norm", [False, True], ids=["sum", "norm"])
def test_add_parts_rmsnorm(gpu, m, k, n_parts, norm):
    """The sum of the shares in order, rounded, then solort_add_rmsnorm: equal bits for x, and for h the bar
    of test_gpu_rows.py (half a bf16 ulp plus the fp32 arithmetic)."""
    print(f"[add_parts_rmsnorm m={m} k={k} n_parts={n_parts} norm={norm}]", flush=True)
    g = torch.Generator().manual_seed(m + k)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    parts = torch.randn(n_parts, m, k, generator=g)
    w = torch.randn(k, generator=g).to(torch.bfloat16)
    y = torch.zeros(m, k)
    for p in parts:
        y = y + p
    total = (x.float() + y.to(torch.bfloat16).float()).to(torch.bfloat16)
    xd = _wide(x, gpu, 8)
    h = _wide(torch.zeros_like(x), gpu, 16) if norm else None
    ops.add_parts_rmsnorm(xd, parts.to(gpu), w.to(gpu) if norm else None, 1e-6, xd, h)
    assert torch.equal(xd.cpu(), total)
    assert (xd._base[:, k:] == 7).all()
    if norm:
        t = total.double()
        want = t * torch.rsqrt(t.square().mean(-1, keepdim=True) + 1e-6) * w.double()
        assert ((h.double().cpu() - want).abs() <= want.abs() * 2 ** -8 + 1e-30).all()


def test_gemm_tile_rejects_bad_arguments(gpu):
    x, w = (torch.zeros(40, 640, dtype=torch.bfloat16, device=gpu) for _ in range(2))
    out = torch.zeros(40, 40, dtype=torch.bfloat16, device=gpu)
    assert ops.gemm_tile_parts(40, 42, 640) == 0 and ops.gemm_tile_parts(40, 40, 576) == 0
    with pytest.raises(RuntimeError):
        ops.gemm_tile(w[:, :576], x[:, :576], out)
    with pytest.raises(RuntimeError):
        ops.gemm_tile(w, x, out[:, :38])
    with pytest.raises(RuntimeError):
        ops.gemm_tile(w, x, torch.zeros(3, 40, 40, device=gpu), mode=ops.TILE_PARTS)


@pytest.mark.parametrize("m,n,k", [(17, 68, 640), (64, 100, 2560), (100, 196, 1024), (200, 6148, 512), (300, 132, 640),
                                   (1000, 260, 512)])
@pytest.mark.parametrize("mode", [ops.TILE_PLAIN, ops.TILE_PARTS, ops.TILE_SWIGLU], ids=["plain", "parts", "swiglu"])
def test_gemm_tile_nan_and_infinity_stay_in_their_row(gpu, m, n, k, mode):
    """A NaN or an infinity in a row of x or of w reaches its own row of results only, and what lies behind the rows
    (NaN here) none: the others keep their bits."""
    print(f"[gemm_tile nan m={m} n={n} k={k} mode={mode}]", flush=True)
    x, w = _inputs(m, 2 * n if mode == ops.TILE_SWIGLU else n, k)
    s = ops.gemm_tile_parts(m, n, k)

    def run(x, w):
        xd, wd = _wide(x, gpu, 8), _wide(w, gpu, 16)
        xd._base[:, k:] = float("nan")
        wd._base[:, k:] = float("nan")
        if mode == ops.TILE_PARTS:
            out = torch.empty(s, m, n, device=gpu)
        else:
            out = torch.empty(m, n, dtype=torch.bfloat16, device=gpu)
        ops.gemm_tile(wd, xd, out, mode=mode, inter=n)
        return out if out.dim() == 3 else out[None]

    clean = run(x, w)
    assert torch.isfinite(clean).all()
    bad_x, bad_w = {m // 2: "nan", m - 1: "inf"}, {1: "inf", n - 1: "nan"}
    for row, v in bad_x.items():
        x[row, (7 * row + 3) % k] = float(v)
    for row, v in bad_w.items():
        w[row, (11 * row + k - 1) % k] = float(v)
    got = run(x, w)
    rows = [r for r in range(m) if r not in bad_x]
    cols = [c for c in range(n) if c not in bad_w]
    assert torch.equal(got[:, rows][:, :, cols], clean[:, rows][:, :, cols])
    assert not torch.isfinite(got[:, m // 2]).all(0).any() and not torch.isfinite(got[:, :, n - 1]).all(0).any()
