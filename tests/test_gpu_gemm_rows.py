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
