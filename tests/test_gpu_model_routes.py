"""The products a prompt's rows (GraphQwen3Decode.prefill) and a verify's tokens take by bucket, width and weight
layout: each combination against the fp32 evaluation of the same model (oracle/ref.py) on the CPU.

Bar: the logits and the K/V rows within 0.03 of the fp32 model's (2-norm of the difference over the 2-norm).  Two
layers of bf16 roundings leave 0.004 to 0.013 whatever the order of the sums; a neighbouring layer's norm weight, a
stale row or a residual left out moves them by 0.1 and more.  Each case states the products it means to run, so that
it fails when a rule sends it elsewhere."""
from __future__ import annotations

import pytest
import torch

from oracle import ref
from solort_amd import model as mdl

pytestmark = pytest.mark.gpu
SMALL = mdl.ModelShape("small", hidden=512, inter=1024, nh=8, nkv=2, layers=2, vocab=4096, tie_embeddings=False)


def _f32(w) -> dict:
    return {k: (v.float().cpu() if torch.is_tensor(v) else [t.float().cpu() for t in v]) for k, v in vars(w).items()
            if k != "shape"}


def _near(got: torch.Tensor, want: torch.Tensor, what: str) -> None:
    rel = ((got.float().cpu() - want).norm() / want.norm()).item()
    print(f"  {what}: {rel:.4f} of the fp32 model", flush=True)
    assert rel <= 0.03, what


def _route(monkeypatch) -> list:
    """The _RowBuffers that the calls after this make."""
    made = []

    class Recorded(mdl._RowBuffers):
        def __init__(self, *args) -> None:
            super().__init__(*args)
            made.append(self)

    monkeypatch.setattr(mdl, "_RowBuffers", Recorded)
    return made


def _prefill_near(w, plen: int, max_len: int, seed: int) -> mdl.GraphQwen3Decode:
    s = w.shape
    m = mdl.GraphQwen3Decode(w, max_len)
    ids = torch.randint(0, s.vocab, (plen,), generator=torch.Generator().manual_seed(seed)).tolist()
    m.prefill(ids)
    kc, vc = (torch.zeros(s.layers, max_len, s.nkv, 128) for _ in range(2))
    want = ref.prefill_model(_f32(w), ids, kc, vc, s.nh, s.nkv)
    _near(m.logits.view(-1), want, "logits")
    _near(m.kc[:, :plen], kc[:, :plen], "K rows")
    _near(m.vc[:, :plen], vc[:, :plen], "V rows")
    first = m.logits.clone()
    m.prefill(ids)  # the captured graph again: the same bits
    assert torch.equal(m.logits, first)
    return m


def _verify_near(w, p0: int, seed: int) -> mdl.GraphQwen3Decode:
    s = w.shape
    m = mdl.GraphQwen3Decode(w, 256)
    g = torch.Generator().manual_seed(seed)
    for c in (m.kc, m.vc):
        c[:, :p0].copy_(torch.randn(s.layers, p0, s.nkv, 128, generator=g))
    kc, vc = m.kc.float().cpu(), m.vc.float().cpu()
    toks = torch.randint(0, s.vocab, (m.k1,), generator=g).tolist()
    m.vtok.copy_(torch.tensor(toks, device=m.dev))
    got = m.verify(p0)
    want = ref.verify_model(_f32(w), toks, p0, kc, vc, s.nh, s.nkv)
    _near(got, want, "logits")
    _near(m.kc[:, p0:p0 + m.k1], kc[:, p0:p0 + m.k1], "K rows")
    _near(m.vc[:, p0:p0 + m.k1], vc[:, p0:p0 + m.k1], "V rows")
    first = got.clone()
    assert torch.equal(m.verify(p0), first)
    return m


def _spread(weights: list[torch.Tensor], stride: int) -> list[torch.Tensor]:
    """The same rows, stride elements apart (in one buffer, side by side)."""
    n, k = weights[0].shape
    buf = torch.empty(n * stride, dtype=torch.bfloat16, device=weights[0].device)
    out = [buf.as_strided((n, k), (stride, 1), i * k) for i in range(len(weights))]
    for o, t in zip(out, weights):
        o.copy_(t)
    return out


@pytest.mark.parametrize("plen", [40, 300])
def test_prefill_takes_weights_past_32_bit_offsets(gpu, monkeypatch, plen):
    """Weights of 2 GiB and more are the library's (solort_gemm_tile has 32-bit offsets)."""
    print(f"[prefill of {plen} rows, weights past 2 GiB]", flush=True)
    w = mdl.RandomQwen3(SMALL, gpu, seed=101)
    for name in ("wqkv", "wo", "wgu", "wd"):
        t = getattr(w, name)
        setattr(w, name, _spread(t, ((1 << 30) // t[0].shape[0] // 8 + 1) * 8))
    made = _route(monkeypatch)
    _prefill_near(w, plen, 512, plen)
    assert all(not b.tile_qkv and not b.tile_gu and b.o_parts is None and b.d_parts is None for b in made) and made


def _weights(gpu, form: str, seed: int):
    odd = dict(hidden=100) if form == "hidden 100" else dict(inter=100) if form == "inter 100" else {}
    shape = mdl.ModelShape(**{**vars(SMALL), **odd})
    w = mdl.RandomQwen3(shape, gpu, seed=seed)
    if form == "columns":  # stored as their transposes
        for name in ("wqkv", "wo", "wgu", "wd"):
            setattr(w, name, [t.t().contiguous().t() for t in getattr(w, name)])
    elif form == "unaligned rows":
        w.wgu = _spread(w.wgu, 2 * shape.hidden + 4)
    elif form == "fp32 norms":
        w.in_ln, w.post_ln = w.in_ln.float(), w.post_ln.float()
    elif form == "head":
        w.lm_head, w.final_norm = w.lm_head.t().contiguous().t(), w.final_norm.float()
    return w


# prefill ends with gemv_argmax, which needs hidden a multiple of 8 and takes the head's rows as they lie
@pytest.mark.parametrize("form", ["inter 100", "columns", "unaligned rows", "fp32 norms"])
@pytest.mark.parametrize("plen", [9, 40, 300])
def test_prefill_takes_weights_the_kernels_do_not_read(gpu, monkeypatch, form, plen):
    print(f"[prefill of {plen} rows, {form}]", flush=True)
    made = _route(monkeypatch)
    _prefill_near(_weights(gpu, form, 102), plen, 512, plen)
    assert made and all(b.general for b in made)


@pytest.mark.parametrize("form", ["hidden 100", "inter 100", "columns", "unaligned rows", "fp32 norms", "head"])
def test_verify_takes_weights_the_kernels_do_not_read(gpu, monkeypatch, form):
    print(f"[verify, {form}]", flush=True)
    made = _route(monkeypatch)
    _verify_near(_weights(gpu, form, 103), 60, 104)
    assert made and all(b.general == (form != "head") for b in made)


def test_start_takes_any_embedding_layout(gpu):
    """The separate-ops tail gathers the embedding row with torch, so it and start() take any strides."""
    w = mdl.RandomQwen3(SMALL, gpu, seed=105)
    want = mdl.GraphQwen3Decode(w, 256, fused_tail=False).generate(7, 0, 6)
    w.embed = w.embed.t().contiguous().t()
    m = mdl.GraphQwen3Decode(w, 256, fused_tail=False)
    m.start(9, 3)
    assert torch.equal(m.x, w.embed[9:10]) and [m.tok.item(), m.pos.item(), m.step.item()] == [9, 3, 0]
    assert m.generate(7, 0, 6) == want
    with pytest.raises(RuntimeError, match="outside the vocabulary"):
        m.start(SMALL.vocab, 3)


# The served widths with two layers and a small vocabulary: what _RowBuffers chooses for the bucket of plen rows.
WIDTHS = {"0.6b": (1024, 3072, 16), "4b": (2560, 9728, 32), "8b": (4096, 12288, 32)}
ROUTES = [("4b", 1, "few"), ("4b", 12, "few"), ("8b", 16, "few"), ("0.6b", 9, "few"),
          ("0.6b", 100, "qkv gu parts"), ("4b", 200, "qkv gu parts"),
          ("0.6b", 300, ""), ("0.6b", 1000, ""),             # library products: add_rmsnorm, and x.add_ in the last layer
          ("4b", 500, "parts"), ("8b", 400, "parts"), ("4b", 1000, "gu parts")]  # at 1024 rows: one round of tiles


@pytest.mark.parametrize("width,plen,route", ROUTES)
def test_prefill_routes_at_served_widths(gpu, monkeypatch, width, plen, route):
    print(f"[prefill of {plen} rows, {width} widths, {route or 'library'}]", flush=True)
    hidden, inter, nh = WIDTHS[width]
    made = _route(monkeypatch)
    w = mdl.RandomQwen3(mdl.ModelShape(width, hidden, inter, nh, 8, 2, 4096, False), gpu, seed=106)
    _prefill_near(w, plen, 1024, plen)
    for b in made:
        if route == "few":
            assert b.few
            continue
        took = [n for n, on in (("qkv", b.tile_qkv), ("gu", b.tile_gu), ("parts", b.o_parts is not None)) if on]
        assert not b.few and not b.general and " ".join(took) == route
        assert (b.o_parts is None) == (b.d_parts is None)
    assert made


@pytest.mark.parametrize("width", list(WIDTHS))
def test_verify_at_served_widths(gpu, monkeypatch, width):
    print(f"[verify, {width} widths]", flush=True)
    hidden, inter, nh = WIDTHS[width]
    made = _route(monkeypatch)
    _verify_near(mdl.RandomQwen3(mdl.ModelShape(width, hidden, inter, nh, 8, 2, 4096, False), gpu, seed=107), 60, 108)
    assert made and all(b.few for b in made)
