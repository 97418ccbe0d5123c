"""GPU parity of the row-wise kernels of a multi-row layer (solort_add_rmsnorm, solort_swiglu_rows).

The residual sum is one bf16 rounding of an exact fp32 sum: equal bits.  The norm and the SwiGLU are
compared with fp64 values of the same rounded inputs: the fp32 arithmetic before the one rounding to
bf16 adds a few 2^-24, so an element is within half a bf16 ulp (2^-9 relative) plus that (bar: 2^-8;
silu(gate) is rounded to bf16 before the product, a second half ulp: 2^-7)."""
from __future__ import annotations

import pytest
import torch

from solort_amd import ops

pytestmark = pytest.mark.gpu


def _randn(g, *dims):
    return torch.randn(*dims, generator=g).to(torch.bfloat16)


def _padded(t: torch.Tensor, gpu, pad: int) -> torch.Tensor:
    """t on the device as a view of wider rows."""
    buf = torch.full((t.shape[0], t.shape[1] + pad), 7.0, dtype=t.dtype, device=gpu)
    buf[:, : t.shape[1]] = t.to(gpu)
    return buf[:, : t.shape[1]]


@pytest.mark.parametrize("m,k,pad", [(1, 8, 0), (5, 2560, 0), (17, 2048, 8), (3, 8192, 0), (2, 8200, 16),
                                     (1024, 1024, 0), (2, 65536, 0)])
@pytest.mark.parametrize("add", [False, True], ids=["norm", "add_norm"])
def test_add_rmsnorm(gpu, m, k, pad, add):
    print(f"[add_rmsnorm m={m} k={k} pad={pad} add={add}]", flush=True)
    g = torch.Generator().manual_seed(m + k)
    x, y, w = _randn(g, m, k), _randn(g, m, k), _randn(g, k)
    xd, h = _padded(x, gpu, pad), _padded(torch.zeros_like(x), gpu, pad)
    total = x
    if add:
        total = (x.float() + y.float()).to(torch.bfloat16)
        ops.add_rmsnorm(xd, _padded(y, gpu, pad), w.to(gpu), 1e-6, xd, h)
        assert torch.equal(xd.cpu(), total)
    else:
        ops.add_rmsnorm(xd, None, w.to(gpu), 1e-6, None, h)
        assert torch.equal(xd.cpu(), x)
    t = total.double()
    want = t * torch.rsqrt(t.square().mean(-1, keepdim=True) + 1e-6) * w.double()
    assert ((h.double().cpu() - want).abs() <= want.abs() * 2 ** -8 + 1e-30).all()
    if pad:
        assert (h._base[:, k:] == 7).all()


@pytest.mark.parametrize("m,inter,pad", [(1, 8, 0), (5, 9728, 0), (33, 2056, 8), (300, 3072, 0)])
def test_swiglu_rows(gpu, m, inter, pad):
    print(f"[swiglu_rows m={m} inter={inter} pad={pad}]", flush=True)
    g = torch.Generator().manual_seed(m + inter)
    gu = _randn(g, m, 2 * inter) * 3
    out = _padded(torch.zeros(m, inter, dtype=torch.bfloat16), gpu, pad)
    ops.swiglu_rows(_padded(gu, gpu, pad), out)
    gate, up = gu.double().split(inter, -1)
    want = gate * torch.sigmoid(gate) * up
    assert ((out.double().cpu() - want).abs() <= want.abs() * 2 ** -7 + 1e-30).all()


def test_rows_reject_bad_arguments(gpu):
    x = torch.zeros(2, 16, dtype=torch.bfloat16, device=gpu)
    w = torch.ones(16, dtype=torch.bfloat16, device=gpu)
    with pytest.raises(RuntimeError):
        ops.add_rmsnorm(x, x.clone(), w, 1e-6, None, x.clone())
    with pytest.raises(RuntimeError):
        ops.swiglu_rows(x, torch.zeros(2, 16, dtype=torch.bfloat16, device=gpu))


def test_nan_and_infinity_stay_in_their_row(gpu):
    """A row that holds a NaN or an infinity leaves the other rows' bits alone, in each of the three launches."""
    g = torch.Generator().manual_seed(5)
    m, k = 7, 2568
    x, y, gu, nw = _randn(g, m, k), _randn(g, m, k), _randn(g, m, 2 * k), _randn(g, k)
    parts = torch.randn(3, m, k, generator=g)

    def run():
        outs = [torch.empty(m, k, dtype=torch.bfloat16, device=gpu) for _ in range(5)]
        ops.add_rmsnorm(x.to(gpu), y.to(gpu), nw.to(gpu), 1e-6, outs[0], outs[1])
        ops.add_parts_rmsnorm(x.to(gpu), parts.to(gpu), nw.to(gpu), 1e-6, outs[2], outs[3])
        ops.swiglu_rows(gu.to(gpu), outs[4])
        return outs

    clean = run()
    for t in (y, gu, parts[1]):
        t[2, 11], t[5, k - 1] = float("nan"), float("inf")
    got = run()
    rows = [0, 1, 3, 4, 6]
    for a, b in zip(got, clean):
        assert torch.equal(a[rows], b[rows]) and torch.isfinite(b).all()
        assert not torch.isfinite(a[2, 11]) and not torch.isfinite(a[5]).all()


def test_swiglu_rows_silu_of_every_gate(gpu):
    """silu of each bf16 value, infinities included, rounds to the bits of torch's (up = 1)."""
    gate = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).to(gpu)
    out = torch.empty(1, 65536, dtype=torch.bfloat16, device=gpu)
    ops.swiglu_rows(torch.cat([gate, torch.ones_like(gate)])[None], out)
    want = torch.nn.functional.silu(gate)[None]
    assert torch.equal(out.isnan(), want.isnan())
    ok = ~want.isnan()
    assert torch.equal(out[ok].view(torch.int16), want[ok].view(torch.int16))
