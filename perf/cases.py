"""The work that is timed and compared when a kernel changes: one token, a speculative round's verify
and a prompt, through the attention runner (GraphQwen3Attention), the whole-model runner
(GraphQwen3Decode) and the tensor front end (ops), at the Qwen3-0.6B / 4B / 8B shapes of this
repository.

Kinds of case (dict key "kind"):
  attn_decode   runner.decode_argmax: one token through every layer's attention block, then the
                greedy argmax of its logits
  attn_verify   runner.verify: the spec_k + 1 tokens of a speculative round, argmax, acceptance
  attn_prefill  runner.prefill: a prompt through every layer's attention block
  paged_decode  ops.paged_decode_layer over every layer's page arena, in a captured graph
  mlp_decode    ops.gemv twice per layer: norm + gate/up + SwiGLU, then down + residual
  model_decode  GraphQwen3Decode.generate of one token: start, one replay, the token read back
  model_prefill GraphQwen3Decode.prefill: a prompt up to its first token's logits
  model_verify  GraphQwen3Decode.verify: the logits of a speculative round's tokens

The whole-model cases run at the real widths with the layer count cut down ("layers"): rounding in a
bf16 layer travels through all that follow, and a few layers already exceed the 256 MB cache.
"""
from __future__ import annotations

import math
import random

import torch

from solort_amd import model as mdl
from solort_amd import ops, runner
from solort_amd.workloads import EPS, HD, THETA, VOCAB

DEV = "cuda"
SHAPES = {"0.6b": mdl.QWEN3_0_6B, "4b": mdl.QWEN3_4B, "8b": mdl.QWEN3_8B}
VERIFY = 5  # spec_k = 4 drafts and the last accepted token


def listed() -> list[dict]:
    return [
        # The draft model in a short chat turn: launch latency is most of it.
        {"name": "attn_decode_0.6b_97", "kind": "attn_decode", "shape": "0.6b", "layers": 28, "max_len": 1024,
         "pos": 96},
        # The step that the benchmark quotes: the last token of a 1024-token context.
        {"name": "attn_decode_4b_1024", "kind": "attn_decode", "shape": "4b", "layers": 36, "max_len": 1024,
         "pos": 1023},
        # A long document: 32K keys, with the few outsized key rows that long contexts show.
        {"name": "attn_decode_8b_32768", "kind": "attn_decode", "shape": "8b", "layers": 8, "max_len": 32768,
         "pos": 32767},
        # The same decode over a paged cache (16-row pages, shuffled), as a server with many sequences keeps it.
        {"name": "paged_decode_4b_1900", "kind": "paged_decode", "shape": "4b", "layers": 36, "max_len": 2048,
         "pos": 1899, "page": 16},
        # A speculative round's check: five tokens after 2048 live keys.
        {"name": "attn_verify_4b_2048", "kind": "attn_verify", "shape": "4b", "layers": 36, "max_len": 4096,
         "pos": 2048},
        # A short question: 100 prompt rows, padded to the 128-row bucket.
        {"name": "attn_prefill_4b_100", "kind": "attn_prefill", "shape": "4b", "layers": 36, "max_len": 1024,
         "rows": 100},
        # A prompt that fills the largest bucket.
        {"name": "attn_prefill_4b_1024", "kind": "attn_prefill", "shape": "4b", "layers": 36, "max_len": 1024,
         "rows": 1024},
        # The MLP half of a decode step on its own.
        {"name": "mlp_decode_4b", "kind": "mlp_decode", "shape": "4b", "layers": 12},
        # One greedy token of the model, host call to host result, in the 1024-key bucket.
        {"name": "model_decode_4b_1000", "kind": "model_decode", "shape": "4b", "layers": 8, "max_len": 1024,
         "pos": 1000},
        # Time to first token of a short ragged prompt.
        {"name": "model_prefill_4b_100", "kind": "model_prefill", "shape": "4b", "layers": 8, "max_len": 1024,
         "rows": 100},
        # Time to first token of a prompt that all but fills the largest bucket.
        {"name": "model_prefill_4b_1000", "kind": "model_prefill", "shape": "4b", "layers": 4, "max_len": 1024,
         "rows": 1000},
        # A speculative round's scoring through the model.
        {"name": "model_verify_4b_1500", "kind": "model_verify", "shape": "4b", "layers": 8, "max_len": 2048,
         "pos": 1500},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["attn_decode", "attn_decode", "attn_verify", "attn_prefill", "paged_decode", "mlp_decode",
                       "model_decode", "model_prefill", "model_verify"])
    shape = rng.choice(["0.6b", "4b", "8b"])
    full = SHAPES[shape].layers
    case: dict = {"kind": kind, "shape": shape}
    if kind in ("attn_decode", "paged_decode", "attn_verify"):
        pos = _log_int(rng, 16, 32000 if kind == "attn_decode" else 8000)
        max_len = 1024
        while max_len < pos + VERIFY:
            max_len *= 2
        # the layers' caches stay under about 1 GB
        case.update(layers=max(4, min(full, 8 * 32768 // max_len)), max_len=max_len, pos=pos)
        if kind == "paged_decode":
            case["page"] = rng.choice([16, 64, 256])
    elif kind in ("attn_prefill", "model_prefill"):
        rows = _log_int(rng, 5, 1024)
        layers = full if kind == "attn_prefill" else rng.choice([2, 3, 4])
        case.update(layers=layers, max_len=1024, rows=rows)
    elif kind == "mlp_decode":
        case.update(layers=rng.randint(6, 12))
    else:
        pos = _log_int(rng, 16, 4000)
        case.update(layers=rng.choice([2, 4, 6]), max_len=1024 if pos + VERIFY < 1024 else 4096, pos=pos)
    return case


# ---------------------------------------------------------------- inputs

def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g: torch.Generator, *dims: int, std: float = 1.0, mean: float = 0.0) -> torch.Tensor:
    return (torch.randn(*dims, generator=g, device=DEV) * std + mean).to(torch.bfloat16)


def _attn_inputs(case: dict, seed: int) -> dict:
    """Norm weights, raw qkv rows, the filled cache rows and (decode, verify) logits of an attention case:
    normed keys and values of unit scale, at 32K keys 1 % of the key rows eight times as large."""
    s, layers, kind = SHAPES[case["shape"]], case["layers"], case["kind"]
    g = _gen(seed)
    t = {"qn": _randn(g, layers, HD, std=0.1, mean=1.0), "kn": _randn(g, layers, HD, std=0.1, mean=1.0)}
    nq = case["rows"] if kind == "attn_prefill" else (VERIFY if kind == "attn_verify" else 1)
    t["qkv"] = _randn(g, layers, nq, s.qkv_width)
    if kind != "attn_prefill":
        pos = case["pos"]
        t["k"] = _randn(g, layers, pos, s.nkv, HD)
        t["v"] = _randn(g, layers, pos, s.nkv, HD)
        if pos > 16384:
            heavy = torch.randperm(pos, generator=g, device=DEV)[: pos // 100]
            t["k"][:, heavy] *= 8.0
    if kind in ("attn_decode", "attn_verify"):
        t["logits"] = _randn(g, nq, VOCAB, std=3.0).float()
    if kind == "attn_verify":
        # the first drafts agree with the target, as most accepted ones do
        draft = t["logits"].argmax(-1)[: VERIFY - 1].clone()
        draft[2:] = (draft[2:] + 1) % VOCAB
        t["draft"] = draft
    return t


def _model_shape(case: dict) -> mdl.ModelShape:
    s = SHAPES[case["shape"]]
    return mdl.ModelShape(s.name, s.hidden, s.inter, s.nh, s.nkv, case["layers"], s.vocab, s.tie_embeddings)


def _model_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed + 1)
    t: dict = {"weights": mdl.RandomQwen3(_model_shape(case), DEV, seed=seed)}
    s = t["weights"].shape
    if case["kind"] == "model_prefill":
        t["ids"] = torch.randint(0, s.vocab, (case["rows"],), generator=g, device=DEV)
    else:
        t["k"] = _randn(g, s.layers, case["pos"], s.nkv, HD)
        t["v"] = _randn(g, s.layers, case["pos"], s.nkv, HD)
        t["ids"] = torch.randint(0, s.vocab, (VERIFY,), generator=g, device=DEV)
    return t


def _mlp_inputs(case: dict, seed: int) -> list[dict]:
    s, g = SHAPES[case["shape"]], _gen(seed)
    return [{"x": _randn(g, s.hidden), "norm": _randn(g, s.hidden, std=0.1, mean=1.0),
             "gu": _randn(g, 2 * s.inter, s.hidden, std=0.02), "down": _randn(g, s.hidden, s.inter, std=0.02)}
            for _ in range(case["layers"])]


def prepare(case: dict, seed: int) -> dict:
    kind, s = case["kind"], SHAPES[case["shape"]]
    st: dict = {"case": case}
    if kind.startswith("attn"):
        t = _attn_inputs(case, seed)
        r = runner.GraphQwen3Attention(s.nh, s.nkv, case["layers"], case["max_len"], t["qn"], t["kn"], EPS, THETA, DEV,
                                       VERIFY, VOCAB)
        if kind != "attn_prefill":
            r.kc[:, : case["pos"]].copy_(t.pop("k"))
            r.vc[:, : case["pos"]].copy_(t.pop("v"))
        st.update(t, r=r)
    elif kind == "paged_decode":
        st.update(_prepare_paged(case, seed))
    elif kind == "mlp_decode":
        st["layers"] = _mlp_inputs(case, seed)
        for w in st["layers"]:
            w["act"] = torch.empty(s.inter, dtype=torch.bfloat16, device=DEV)
            w["out"] = torch.empty(s.hidden, dtype=torch.bfloat16, device=DEV)
    else:
        t = _model_inputs(case, seed)
        m = mdl.GraphQwen3Decode(t["weights"], case["max_len"], EPS, THETA, max_tokens=64, spec_k=VERIFY - 1)
        if kind != "model_prefill":
            m.kc[:, : case["pos"]].copy_(t["k"])
            m.vc[:, : case["pos"]].copy_(t["v"])
        st.update(m=m, ids=t["ids"].tolist())
        if kind == "model_verify":
            m.vtok.copy_(t["ids"])
    return st


def _prepare_paged(case: dict, seed: int) -> dict:
    """One layer-major arena of shuffled pages and the step's captured graph, as a serving loop holds them."""
    s, layers, page, bound = SHAPES[case["shape"]], case["layers"], case["page"], case["max_len"]
    t = _attn_inputs(case, seed)
    n_pages = bound // page
    g = _gen(seed + 1)
    table = torch.randperm(n_pages, generator=g, device=DEV)
    arena = torch.zeros(layers, n_pages, 2, page, s.nkv, HD, dtype=torch.bfloat16, device=DEV)
    full = torch.zeros(layers, bound, s.nkv, HD, dtype=torch.bfloat16, device=DEV)
    for i, name in enumerate(("k", "v")):
        full[:, : case["pos"]].copy_(t.pop(name))
        arena[:, table, i] = full.view(layers, n_pages, page, s.nkv, HD)
    pos = torch.tensor([case["pos"]], dtype=torch.long, device=DEV)
    ns = runner.decode_splits(bound, s.nkv)
    st = dict(t, arena=arena, table=table.to(torch.int32), pos=pos, inv=ops.inv_freq(HD, THETA, DEV), ns=ns,
              cs=torch.zeros(2, 1, HD // 2, dtype=torch.bfloat16, device=DEV),
              ws=ops.attn_workspace(1, s.nh, s.nkv, ns, DEV),
              ctx=torch.zeros(layers, 1, s.nh * HD, dtype=torch.bfloat16, device=DEV))

    def step() -> None:
        ops.rope_rows(st["inv"], pos, 1, st["cs"])
        for li in range(layers):
            ops.paged_decode_layer(st["qkv"][li], st["qn"][li], st["kn"][li], EPS, st["cs"], pos, arena[li],
                                   st["table"], bound, HD ** -0.5, st["ws"], ns, st["ctx"][li], s.nh, s.nkv)

    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    p, slot = int(table[case["pos"] // page]), case["pos"] % page
    st.update(graph=graph, new_k=arena[:, p, 0, slot], new_v=arena[:, p, 1, slot])
    return st


def run(state: dict) -> dict:
    case = state["case"]
    kind = case["kind"]
    if kind == "attn_decode":
        r, pos = state["r"], case["pos"]
        tok = r.decode_argmax(state["qkv"], pos, state["logits"])
        return {"ctx": r.ctx_dec, "k": r.kc[:, pos], "v": r.vc[:, pos], "tok": tok}
    if kind == "attn_verify":
        r, pos = state["r"], case["pos"]
        ctx = r.verify(state["qkv"], pos, state["logits"], state["draft"])
        return {"ctx": ctx, "k": r.kc[:, pos:pos + VERIFY], "v": r.vc[:, pos:pos + VERIFY], "tok": r.tok_ver,
                "accepted": r.acc_ver}
    if kind == "attn_prefill":
        r, rows = state["r"], case["rows"]
        return {"ctx": r.prefill(state["qkv"]), "k": r.kc[:, :rows], "v": r.vc[:, :rows]}
    if kind == "paged_decode":
        state["graph"].replay()
        return {"ctx": state["ctx"], "k": state["new_k"], "v": state["new_v"]}
    if kind == "mlp_decode":
        for w in state["layers"]:
            ops.gemv(w["gu"], w["x"], w["act"], w["norm"], EPS, mode=ops.GEMV_SWIGLU, inter=w["act"].numel())
            ops.gemv(w["down"], w["act"], w["out"], res=w["x"], mode=ops.GEMV_RESID)
        return {"act": [w["act"] for w in state["layers"]], "out": [w["out"] for w in state["layers"]]}
    m = state["m"]
    if kind == "model_prefill":
        rows = case["rows"]
        m.prefill(state["ids"])
        return {"logits": m.logits, "k": m.kc[:, :rows], "v": m.vc[:, :rows]}
    pos = case["pos"]
    if kind == "model_decode":
        m.generate(state["ids"][0], pos, 1)
        return {"logits": m.logits, "k": m.kc[:, pos], "v": m.vc[:, pos]}
    return {"logits": m.verify(pos), "k": m.kc[:, pos:pos + VERIFY], "v": m.vc[:, pos:pos + VERIFY]}


# ---------------------------------------------------------------- what a pass cannot do without

def _attn_work(s, layers: int, live: int, nq: int, causal: bool) -> tuple[int, int]:
    """Bytes and operations of the attention blocks: qkv in, new K/V out, live K/V in, ctx out."""
    pairs = nq * (nq + 1) // 2 + (0 if causal else nq * live)
    nbytes = 2 * (nq * s.qkv_width + nq * s.nh * HD + 2 * nq * s.nkv * HD + 2 * live * s.nkv * HD)
    return layers * nbytes, layers * 4 * s.nh * HD * pairs


def work(case: dict) -> dict:
    kind, s, layers = case["kind"], SHAPES[case["shape"]], case["layers"]
    if kind == "mlp_decode":
        weights = layers * 3 * s.hidden * s.inter
        return {"bytes": 2 * weights + layers * 2 * (3 * s.hidden + s.inter), "flops": 2 * weights}
    prefill = kind.endswith("prefill")
    nq = case["rows"] if prefill else (VERIFY if kind.endswith("verify") else 1)
    live = 0 if prefill else case["pos"]
    nbytes, flops = _attn_work(s, layers, live, nq, prefill)
    if kind in ("attn_decode", "attn_verify"):
        nbytes += 4 * nq * VOCAB
    if kind.startswith("model"):
        block = s.hidden * (s.qkv_width + s.nh * HD + 3 * s.inter)
        scored = 1 if prefill else nq  # rows through the head
        nbytes = layers * 2 * (block + 2 * live * s.nkv * HD + 2 * nq * s.nkv * HD)
        nbytes += 2 * s.hidden * (s.vocab + nq) + 2 * scored * s.vocab
        flops += 2 * (layers * nq * block + scored * s.hidden * s.vocab)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case: dict) -> dict:
    """Two correct bf16 implementations lie as far apart as their roundings, at most about sqrt(2) times
    their distance from the 64-bit result.  Measured against exact(): 0.0031-0.0044 in a single attention
    block or MLP (0.0092 at 32K keys, nearly all of it the rounding of q and k to bf16, which every
    implementation shares), 0.014-0.022 in the logits and caches of a few whole layers, where each
    layer's roundings travel on."""
    if case["kind"].startswith("model"):
        return {"rel": 0.03, "max": 0.3}
    return {"rel": 0.01, "max": 0.1}


# ---------------------------------------------------------------- the same in 64 bits

def _norm64(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x: torch.Tensor, pos0: int) -> torch.Tensor:
    """x [T, heads, 128] rotated to positions pos0.. (half-split pairs)."""
    half = HD // 2
    f = THETA ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
    a = torch.arange(pos0, pos0 + x.shape[0], device=x.device, dtype=torch.float64)[:, None, None] * f
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat([lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin()], -1)


def _attn64(s, qkv, qn, kn, pos0: int, k_old, v_old):
    """One layer's attention block: (ctx [T, nh*128], new K rows, new V rows [T, nkv, 128])."""
    T, G = qkv.shape[0], s.nh // s.nkv
    q, k, v = qkv.view(T, s.nh + 2 * s.nkv, HD).split([s.nh, s.nkv, s.nkv], 1)
    q, k = _rope64(_norm64(q, qn), pos0), _rope64(_norm64(k, kn), pos0)
    keys = k if k_old is None else torch.cat([k_old.double(), k])
    vals = v if v_old is None else torch.cat([v_old.double(), v])
    mask = torch.arange(keys.shape[0], device=q.device)[None] > pos0 + torch.arange(T, device=q.device)[:, None]
    ctx = torch.empty(T, s.nh, HD, dtype=torch.float64, device=q.device)
    for h in range(s.nkv):
        kt, vh = keys[:, h].t().contiguous(), vals[:, h].contiguous()
        for g in range(G):
            p = (q[:, h * G + g].contiguous() @ kt) * HD ** -0.5
            ctx[:, h * G + g] = torch.softmax(p.masked_fill(mask, -math.inf), -1) @ vh
    return ctx.view(T, s.nh * HD), k, v


def _mm64(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x @ w.T, the weight widened in row blocks."""
    return torch.cat([x @ b.double().t().contiguous() for b in w.split(16384)], -1)


def exact(case: dict, seed: int):
    kind, s, layers = case["kind"], SHAPES[case["shape"]], case["layers"]
    if kind == "mlp_decode":
        act, out = [], []
        for w in _mlp_inputs(case, seed):
            x = w["x"].double()[None]
            gate, up = _mm64(_norm64(x, w["norm"]), w["gu"]).split(s.inter, -1)
            a = gate * torch.sigmoid(gate) * up
            act.append(a.view(-1))
            out.append((x + _mm64(a, w["down"])).view(-1))
        return {"act": act, "out": out}
    if kind.startswith("model"):
        return _exact_model(case, seed)
    t = _attn_inputs(case, seed)
    pos = 0 if kind == "attn_prefill" else case["pos"]
    ctx, ks, vs = [], [], []
    for li in range(layers):
        c, k, v = _attn64(s, t["qkv"][li].double(), t["qn"][li], t["kn"][li], pos, t["k"][li] if "k" in t else None,
                          t["v"][li] if "v" in t else None)
        ctx.append(c)
        ks.append(k)
        vs.append(v)
    one = kind in ("attn_decode", "paged_decode")
    ans = {"ctx": torch.stack(ctx), "k": torch.stack([k[0] for k in ks] if one else ks),
           "v": torch.stack([v[0] for v in vs] if one else vs)}
    if kind in ("attn_decode", "attn_verify"):
        top = t["logits"].max(-1, keepdim=True).values
        ans["tok"] = (t["logits"] == top).int().argmax(-1)  # the lowest index of equal maxima
    if kind == "attn_verify":
        tok, draft = ans["tok"].tolist(), t["draft"].tolist()
        n = next((i for i, d in enumerate(draft) if d != tok[i]), len(draft))
        ans["accepted"] = torch.tensor([n, tok[n]], device=DEV)
    return ans


def _exact_model(case: dict, seed: int) -> dict:
    kind = case["kind"]
    t = _model_inputs(case, seed)
    w, s = t["weights"], t["weights"].shape
    ids = t["ids"] if kind != "model_decode" else t["ids"][:1]
    pos = 0 if kind == "model_prefill" else case["pos"]
    x = w.embed[ids].double()
    ks, vs = [], []
    for li in range(s.layers):
        qkv = _mm64(_norm64(x, w.in_ln[li]), w.wqkv[li])
        ctx, k, v = _attn64(s, qkv, w.qn[li], w.kn[li], pos, t["k"][li] if "k" in t else None,
                            t["v"][li] if "v" in t else None)
        x = x + _mm64(ctx, w.wo[li])
        gate, up = _mm64(_norm64(x, w.post_ln[li]), w.wgu[li]).split(s.inter, -1)
        x = x + _mm64(gate * torch.sigmoid(gate) * up, w.wd[li])
        ks.append(k)
        vs.append(v)
    if kind == "model_prefill":
        x = x[-1:]
    logits = _mm64(_norm64(x, w.final_norm), w.lm_head)
    one = kind == "model_decode"
    return {"logits": logits, "k": torch.stack([k[0] for k in ks] if one else ks),
            "v": torch.stack([v[0] for v in vs] if one else vs)}
