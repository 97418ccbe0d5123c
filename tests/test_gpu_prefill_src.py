"""GPU parity of the prefill layer over rows found through a record in device memory
(solort_set_qkv_src, solort_prefill_layer_src) and of the runner's prefill, which uses it from
FUSED_PREFILL_MIN rows on: the bits of solort_prefill_layer over the same rows padded with zeros, cache
padding rows included."""
from __future__ import annotations

import pytest
import torch

from solort_amd import ops, runner

pytestmark = pytest.mark.gpu
EPS, THETA, HD = 1e-6, 1e6, 128


def _want(qkv, bound, nh, nkv, qn, kn):
    """ctx [L, plen, nh*128] and the K/V rows 0..bound-1 by solort_prefill_layer."""
    L, plen, width = qkv.shape
    pad = torch.zeros(L, bound, width, dtype=torch.bfloat16, device=qkv.device)
    pad[:, :plen] = qkv
    kc = torch.full((L, bound, nkv, HD), 7.0, dtype=torch.bfloat16, device=qkv.device)
    vc, ctx = kc.clone(), torch.empty(L, bound, nh * HD, dtype=torch.bfloat16, device=qkv.device)
    cs = torch.empty(2, bound, HD // 2, dtype=torch.bfloat16, device=qkv.device)
    ops.rope_rows(ops.inv_freq(HD, THETA, qkv.device), torch.zeros(1, dtype=torch.long, device=qkv.device), bound, cs)
    for li in range(L):
        ops.prefill_layer(pad[li], qn[li], kn[li], EPS, cs, kc[li], vc[li], HD ** -0.5, ctx[li], nh, nkv)
    return ctx[:, :plen], kc, vc


# the first length of a bucket, its ends, lengths inside a tile; every query group
CASES = [(129, 16, 8), (255, 32, 8), (256, 8, 8), (257, 32, 8), (500, 32, 4), (513, 16, 8), (700, 32, 8), (1000, 8, 8),
         (1024, 32, 8)]


@pytest.mark.parametrize("plen,nh,nkv", CASES)
@pytest.mark.parametrize("form", ["rows", "wide_rows", "layers_inside", "fp32", "host"])
def test_runner_prefill_forms(gpu, plen, nh, nkv, form):
    print(f"[prefill_src plen={plen} nh={nh} nkv={nkv} form={form}]", flush=True)
    L, width = 2, (nh + 2 * nkv) * HD
    g = torch.Generator().manual_seed(plen + nh)
    base = torch.randn(L, plen, width, generator=g).to(torch.bfloat16)
    qn, kn = ((torch.randn(L, HD, generator=g) * 0.1 + 1).to(torch.bfloat16).to(gpu) for _ in range(2))
    dev = base.to(gpu)
    if form == "wide_rows":
        given = torch.full((L, plen, width + 8), 9.0, dtype=torch.bfloat16, device=gpu)
        given[..., :width] = dev
        given = given[..., :width]
    elif form == "layers_inside":
        given = dev.transpose(0, 1).contiguous().transpose(0, 1)
    else:
        given = {"rows": dev, "fp32": dev.float(), "host": base}[form]
    r = runner.GraphQwen3Attention(nh, nkv, L, 1024, qn, kn, EPS, THETA, gpu, 5, 1000)
    bound = next(b for b in r.pre_buckets if b >= plen)
    want, kc, vc = _want(dev, bound, nh, nkv, qn, kn)
    for again in range(3):
        r.kc.fill_(5.0)
        r.vc.fill_(5.0)
        got = r.prefill(given)
        assert torch.equal(got, want), again
        assert torch.equal(r.kc[:, :bound], kc) and torch.equal(r.vc[:, :bound], vc)
        assert (r.kc[:, bound:] == 5).all() and (r.vc[:, bound:] == 5).all()
    assert r.src_pre[0].item() == r.qkv_pre.data_ptr()  # nothing refers to the caller's rows after the call
    other = torch.randn(L, plen - 1, width, generator=g).to(torch.bfloat16).to(gpu)  # other rows, the same graph
    assert torch.equal(r.prefill(other), _want(other, bound if plen - 1 > bound // 2 else bound // 2, nh, nkv, qn, kn)[0])


def test_set_qkv_src_rejects(gpu):
    src = ops.qkv_src(gpu)
    rows = torch.zeros(2, 300, 1024, dtype=torch.bfloat16, device=gpu)
    for bad in (rows[:, :, 4:], rows[:, ::1, ::2], rows.float(), rows[0], rows[:, :0]):
        with pytest.raises(RuntimeError):
            ops.set_qkv_src(src, bad)


# full buckets, the ends of the two rules (256: 64 padding rows, 65 and 63), padding of most of a bucket
@pytest.mark.parametrize("plen", [129, 191, 192, 193, 256, 448, 449, 512, 700, 961, 1024])
@pytest.mark.parametrize("form", ["fp32", "own", "rows"])
def test_runner_prefill_over_own_buffer(gpu, plen, form):
    """A prompt in the runner's buffer (copied there, or put there by the caller) that nearly fills its bucket
    replays a graph over the buffer itself, every other one the graph over the record; the two alternate on one runner
    without touching each other's rows."""
    print(f"[prefill own buffer plen={plen} form={form}]", flush=True)
    L, nh, nkv = 2, 16, 8
    g = torch.Generator().manual_seed(plen)
    qn, kn = ((torch.randn(L, HD, generator=g) * 0.1 + 1).to(torch.bfloat16).to(gpu) for _ in range(2))
    r = runner.GraphQwen3Attention(nh, nkv, L, 1024, qn, kn, EPS, THETA, gpu, 5, 1000)
    bound = next(b for b in r.pre_buckets if b >= plen)
    for again in range(3):
        rows = torch.randn(L, plen, r.width, generator=g).to(torch.bfloat16).to(gpu)
        want, kc, vc = _want(rows, bound, nh, nkv, qn, kn)
        if form == "own":
            r.qkv_pre.fill_(3.0)  # rows past the prompt are not the caller's to clear
            r.qkv_pre[:, :plen].copy_(rows)
        got = r.prefill({"fp32": lambda: rows.float(), "own": lambda: r.qkv_pre[:, :plen], "rows": lambda: rows}[form]())
        assert torch.equal(got, want), again
        assert torch.equal(r.kc[:, :bound], kc) and torch.equal(r.vc[:, :bound], vc)
        other = torch.randn(L, bound - 100, r.width, generator=g).to(torch.bfloat16).to(gpu)  # over the record
        assert torch.equal(r.prefill(other), _want(other, bound, nh, nkv, qn, kn)[0])
        assert r.src_pre[0].item() == r.qkv_pre.data_ptr()
    assert sorted(r._pre_own) == ([bound] if form != "rows" and bound - plen < 64 else [])
    assert sorted(r._pre_src) == [bound]


@pytest.mark.parametrize("plen,bound,nh,nkv", [(130, 256, 8, 8), (250, 256, 16, 8), (300, 512, 32, 8), (512, 512, 8, 1)])
def test_prefill_layer_src_fp32_output(gpu, plen, bound, nh, nkv):
    """The fp32 output over a record: the bits of solort_prefill_layer's over the padded rows."""
    print(f"[prefill_layer_src fp32 plen={plen} bound={bound} nh={nh} nkv={nkv}]", flush=True)
    g = torch.Generator().manual_seed(plen)
    width = (nh + 2 * nkv) * HD
    rows = torch.randn(2, plen, width, generator=g).to(torch.bfloat16).to(gpu)
    qn, kn = ((torch.randn(HD, generator=g) * 0.1 + 1).to(torch.bfloat16).to(gpu) for _ in range(2))
    cs = ops.rope_rows(ops.inv_freq(HD, THETA, gpu), torch.zeros(1, dtype=torch.long, device=gpu), bound)
    src = ops.qkv_src(gpu)
    ops.set_qkv_src(src, rows)
    pad = torch.zeros(bound, width, dtype=torch.bfloat16, device=gpu)
    for layer in range(2):
        kc, vc, kc2, vc2 = (torch.full((bound, nkv, HD), 7.0, dtype=torch.bfloat16, device=gpu) for _ in range(4))
        out, out2 = (torch.empty(bound, nh * HD, device=gpu) for _ in range(2))
        ops.prefill_layer_src(src, layer, qn, kn, EPS, cs, kc, vc, HD ** -0.5, out, nh, nkv)
        pad[:plen] = rows[layer]
        ops.prefill_layer(pad, qn, kn, EPS, cs, kc2, vc2, HD ** -0.5, out2, nh, nkv)
        assert torch.equal(out[:plen], out2[:plen]) and torch.equal(kc, kc2) and torch.equal(vc, vc2)
