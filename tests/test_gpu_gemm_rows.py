"""GPU parity of the few-row matrix product (solort_gemm_rows) with its fused RMSNorm, residual and SwiGLU.

Bar as in test_gpu_gemv.py: within four bf16 ulps (2^-6 relative) plus 2e-3 of the fp64 value of the
same computation on the same bf16 inputs (the fused roundings are the reference's bf16 tensors'),
mean relative error <= 2e-3."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import ref
from solort_amd import ops

pytestmark = pytest.mark.gpu


def _close(got: torch.Tensor, want: torch.Tensor, part: torch.Tensor | None = None) -> None:
    """part: a bf16 summand of want; its rounding may fall one bf16 ulp (at most 2^-7 relative) away, which a sum
    that cancels does not scale down."""
    got, want = got.double().cpu().numpy(), want.double().numpy()
    err = np.abs(got - want)
    slack = 0.0 if part is None else np.abs(part.double().numpy()) * 2 ** -7
    assert (err <= np.abs(want) * 2 ** -6 + 2e-3 + slack).all(), err.max()
    assert (err / (np.abs(want) + 1e-2)).mean() <= 2e-3


def _lin(x, w):
    return (x.double() @ w.double().t()).to(torch.bfloat16)


def _wide(t: torch.Tensor, gpu, pad: int) -> torch.Tensor:
    buf = torch.full((t.shape[0], t.shape[1] + pad), 7.0, dtype=t.dtype, device=gpu)
    buf[:, : t.shape[1]] = t.to(gpu)
    return buf[:, : t.shape[1]]


# k: ragged (less than a step, some wavefronts without a share, a tail chunk), then shares of 1, 2, 4, 5, 6, 8, 9,
# 19, 24 and 25 whole steps per wavefront; n: below one tile, ragged, uneven over the CUs, many tiles per workgroup
SHAPES = [(1, 7, 24), (5, 33, 136), (16, 100, 520), (3, 4099, 8 * 700), (9, 40, 512), (5, 17000, 1024),
          (8, 9001, 2048), (5, 6144, 2560), (12, 6144, 2560), (5, 1024, 3072), (5, 2560, 4096), (16, 2560, 4096),
          (2, 70, 4608), (8, 2563, 9728), (11, 2560, 9728), (5, 4096, 12288), (5, 130, 12800)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("norm", [False, True], ids=["plain", "norm"])
def test_gemm_rows_plain_and_residual(gpu, m, n, k, norm):
    print(f"[gemm_rows m={m} n={n} k={k} norm={norm}]", flush=True)
    g = torch.Generator().manual_seed(m + n + k)
    w = (torch.randn(n, k, generator=g) * 0.02).to(torch.bfloat16)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    nw = (torch.randn(k, generator=g) * 0.1 + 1).to(torch.bfloat16)
    res = torch.randn(m, n, generator=g).to(torch.bfloat16)
    h = ref.rmsnorm(x, nw, 1e-6) if norm else x
    lin = _lin(h, w)
    xd, wd, nwd = _wide(x, gpu, 8), _wide(w, gpu, 16), nw.to(gpu) if norm else None
    out = _wide(torch.zeros(m, n, dtype=torch.bfloat16), gpu, 3)
    ops.gemm_rows(wd, xd, out, nwd, 1e-6)
    _close(out, lin)
    assert (out._base[:, n:] == 7).all()
    buf = res.to(gpu)
    ops.gemm_rows(wd, xd, buf, nwd, 1e-6, res=buf, mode=ops.GEMV_RESID)  # in place
    _close(buf, res.double() + lin.double(), lin)


@pytest.mark.parametrize("m,n,inter,k", [(5, 9728, 9728, 2560), (16, 9, 12, 72), (1, 3072, 3072, 1024),
                                         (2, 70, 100, 4096 + 512)])
def test_gemm_rows_swiglu(gpu, m, n, inter, k):
    print(f"[gemm_rows swiglu m={m} n={n} k={k}]", flush=True)
    g = torch.Generator().manual_seed(m + n)
    w = (torch.randn(inter + n, k, generator=g) * 0.02).to(torch.bfloat16)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    nw = (torch.randn(k, generator=g) * 0.1 + 1).to(torch.bfloat16)
    h = ref.rmsnorm(x, nw, 1e-6)
    gate, up = _lin(h, w[:n]).double(), _lin(h, w[inter:]).double()
    out = torch.empty(m, n, dtype=torch.bfloat16, device=gpu)
    ops.gemm_rows(w.to(gpu), x.to(gpu), out, nw.to(gpu), 1e-6, mode=ops.GEMV_SWIGLU, inter=inter)
    _close(out, (gate * torch.sigmoid(gate)).to(torch.bfloat16).double() * up)


def test_gemm_rows_rejects_bad_arguments(gpu):
    w = torch.zeros(32, 64, dtype=torch.bfloat16, device=gpu)
    with pytest.raises(RuntimeError):
        ops.gemm_rows(w, torch.zeros(ops.GEMM_ROWS_MAX + 1, 64, dtype=torch.bfloat16, device=gpu),
                      torch.zeros(ops.GEMM_ROWS_MAX + 1, 32, dtype=torch.bfloat16, device=gpu))
    with pytest.raises(RuntimeError):
        ops.gemm_rows(w, w[:2], torch.zeros(2, 33, dtype=torch.bfloat16, device=gpu))


# Several tiles per workgroup (more than 16 outputs a CU) in each form that keeps x resident in several batches: the
# next tile's first batches load during this one, the sums alternate between two LDS buffers; last, two to four tiles
# of a one-batch form with 9-16 rows
@pytest.mark.parametrize("m,n,k", [(16, 6144, 4096), (9, 12301, 4096), (5, 4200, 9728), (8, 9001, 9728), (5, 4200, 12288),
                                   (3, 8403, 12288), (16, 6144, 2560), (13, 17001, 1024), (11, 9728, 9728)])
@pytest.mark.parametrize("norm", [False, True], ids=["plain", "norm"])
def test_gemm_rows_several_tiles_per_workgroup(gpu, m, n, k, norm):
    test_gemm_rows_plain_and_residual(gpu, m, n, k, norm)


# the gate/up products of 9-16 rows at the three served widths (x resident, two row groups), and one row group
@pytest.mark.parametrize("m,inter,k", [(16, 9728, 2560), (12, 3072, 1024), (16, 12288, 4096), (8, 12288, 4096)])
@pytest.mark.parametrize("norm", [False, True], ids=["plain", "norm"])
def test_gemm_rows_swiglu_widths(gpu, m, inter, k, norm):
    print(f"[gemm_rows swiglu m={m} inter={inter} k={k} norm={norm}]", flush=True)
    g = torch.Generator().manual_seed(m + inter)
    w = (torch.randn(2 * inter, k, generator=g) * 0.02).to(torch.bfloat16)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    nw = (torch.randn(k, generator=g) * 0.1 + 1).to(torch.bfloat16)
    h = ref.rmsnorm(x, nw, 1e-6) if norm else x
    gate, up = _lin(h, w).double().split(inter, -1)
    out = torch.empty(m, inter, dtype=torch.bfloat16, device=gpu)
    ops.gemm_rows(w.to(gpu), x.to(gpu), out, nw.to(gpu) if norm else None, 1e-6, mode=ops.GEMV_SWIGLU, inter=inter)
    _close(out, (gate * torch.sigmoid(gate)).to(torch.bfloat16).double() * up)


@pytest.mark.parametrize("m,n,k", [(5, 70, 136), (16, 6144, 2560), (16, 2560, 4096), (5, 4200, 9728), (11, 2560, 9728)])
@pytest.mark.parametrize("mode", [ops.GEMV_PLAIN, ops.GEMV_RESID, ops.GEMV_SWIGLU], ids=["plain", "resid", "swiglu"])
def test_gemm_rows_nan_and_infinity_stay_in_their_row(gpu, m, n, k, mode):
    """A NaN or an infinity in a row of x or of w reaches its own row of results only, and what lies behind the rows
    (NaN here) none: the others keep their bits."""
    print(f"[gemm_rows nan m={m} n={n} k={k} mode={mode}]", flush=True)
    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(2 * n if mode == ops.GEMV_SWIGLU else n, k, generator=g) * 0.02).to(torch.bfloat16)
    nw = torch.ones(k, dtype=torch.bfloat16, device=gpu)
    res = torch.randn(m, n, generator=g).to(torch.bfloat16).to(gpu)

    def run(x, w):
        xd, wd = _wide(x, gpu, 8), _wide(w, gpu, 16)
        xd._base[:, k:] = float("nan")
        wd._base[:, k:] = float("nan")
        out = torch.empty(m, n, dtype=torch.bfloat16, device=gpu)
        ops.gemm_rows(wd, xd, out, nw, 1e-6, res=res if mode == ops.GEMV_RESID else None, mode=mode, inter=n)
        return out

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
    assert torch.equal(got[rows][:, cols], clean[rows][:, cols])
    # the norm spreads a bad x over its row
    assert not torch.isfinite(got[m // 2]).any() and not torch.isfinite(got[m - 1]).any()
    assert not torch.isfinite(got[:, n - 1]).any()
