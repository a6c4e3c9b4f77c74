"""What is measured: the work a user of this library has it do, through its public entry points.

A case is a dict of plain values; its "kind" names the path:

  step    one decode token over the layers of a plan (attn_step_run): a stack whose queries are ready together, or one layer
  pair    a token of both head_dims with KV sharing (attn_step_run_pair)
  batch   one layer of a continuous batch: every sequence's step prepared and run each token (attn_step)
  block   layers in the engine's order with their projections, captured once in a HIP graph and replayed
  engine  one layer through the drop-in dispatches, kernel for kernel as the engine issues them
  prefill a prompt's chunked prep and causal prefill (attn_prompt_prep_many, then attn_prefill or a kept plan)
  head    the sampling head: the fused pass, or the engine's three dispatches

Inputs: raw projections and hidden states N(0, 1); norm weights near 1 (q) and near 1/8 (k), which give scores of a few
nats at scale 1 as trained models have them; cached K rows normalised and weighted the same way, V rows of unit RMS.
"""
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "gemma4-webgpu_amd"))

from g4attn import abi, e2b, ops  # noqa: E402

NQH, NKH, HIDDEN, EPS = 8, 1, 1536, 1e-6
GLOBAL_LAYERS = e2b.GLOBAL_LAYERS


# ---- the cases -----------------------------------------------------------------------

def listed():
    return [
        # One local layer at position 512: the smallest decode call, all latency and launches.
        dict(name="step_local_512", kind="step", layers=1, globals=0, head_dim=256, pos=512, window=512),
        # The 35-layer stack at 8K context, head_dim 256 everywhere: an ordinary chat turn's token.
        dict(name="step_stack_8k", kind="step", layers=35, globals=7, head_dim=256, pos=8192, window=512),
        # A token of the real model's shapes (head_dim 512 on global layers, shared caches) at 32K context.
        dict(name="pair_32k", kind="pair", pos=32768, window=512),
        # A serving batch: 64 sequences of 1K to 32K rows on a global layer, planned anew each token.
        dict(name="batch_64", kind="batch", sequences=64, lo=1024, hi=32768, head_dim=256, window=0),
        # One period of layers (four local, one global of head_dim 512) with their f16 projections at 8K.
        dict(name="block_f16_8k", kind="block", format="f16", locals=4, globals=1, pos=8192, window=512),
        # The same with 4-bit weights in a short chat.
        dict(name="block_q4k_1k", kind="block", format="q4k", locals=4, globals=1, pos=1023, window=512),
        # The engine's own dispatches on a global layer at the end of its default 2048-token context.
        dict(name="engine_global_2k", kind="engine", format="f16", head_dim=512, pos=2047, window=0),
        # A short chat prompt (77 tokens), one local and one global layer, planned for this prompt.
        dict(name="prompt_77", kind="prefill", head_dim=256, tokens=77, start=0, chunk=512, locals=1, globals=1,
             window=512, vt=True, keep_plan=False),
        # A 4096-token prompt as 512-token chunks, one local and one global layer, the plan kept.
        dict(name="prefill_4k", kind="prefill", head_dim=256, tokens=4096, start=0, chunk=512, locals=1, globals=1,
             window=512, vt=True, keep_plan=True),
        # A follow-up turn: 1900 tokens after 3001 cached ones on a global layer of head_dim 512, no V^T kept.
        dict(name="prefill_turn_512", kind="prefill", head_dim=512, tokens=1900, start=3001, chunk=1900, locals=0,
             globals=1, window=512, vt=False, keep_plan=False),
        # The sampling head of every token: the tied embedding's GEMV, softcap and top-1.
        dict(name="head_fused", kind="head", fused=True, vocab=262144, hidden=1536, cap=30.0),
        # The same through the engine's three dispatches.
        dict(name="head_engine", kind="head", fused=False, vocab=262144, hidden=1536, cap=30.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["step", "step", "pair", "batch", "block", "block", "engine", "engine", "prefill", "prefill",
                       "prefill", "head"])
    window = rng.choice([512, 512, 512, 1024])
    if kind == "step":
        layers = rng.choice([1, 1, 5, 14, 35])
        globals_ = max(rng.choice([0, 1]), layers // 5)
        return dict(kind=kind, layers=layers, globals=globals_, head_dim=rng.choice([256, 256, 512]),
                    pos=_log_int(rng, 64, 131071 if layers < 5 else 32768 if layers < 35 else 16384), window=window)
    if kind == "pair":
        return dict(kind=kind, pos=_log_int(rng, 300, 32768), window=window)
    if kind == "batch":
        lo = _log_int(rng, 16, 4096)
        return dict(kind=kind, sequences=rng.randint(2, 64), lo=lo, hi=lo + _log_int(rng, 16, 24000),
                    head_dim=rng.choice([256, 256, 512]), window=rng.choice([0, 0, window]))
    if kind == "block":
        return dict(kind=kind, format=rng.choice(["f16", "f16", "q8", "q4k"]), locals=rng.randint(1, 4),
                    globals=rng.randint(0, 1), pos=_log_int(rng, 40, 32768), window=window)
    if kind == "engine":
        hd = rng.choice([256, 512])
        return dict(kind=kind, format=rng.choice(["f16", "q8", "q4k"]), head_dim=hd,
                    pos=_log_int(rng, 20, 2047), window=0 if hd == 512 else window)
    if kind == "prefill":
        hd = rng.choice([256, 256, 512])
        tokens = _log_int(rng, 5, 4096 if hd == 256 else 2048)
        return dict(kind=kind, head_dim=hd, tokens=tokens, start=rng.choice([0, 0, rng.randint(1, 4000)]),
                    chunk=rng.choice([512, 512, 4096]), locals=rng.randint(0, 1) if hd == 256 else 0, globals=1,
                    window=window, vt=rng.random() < 0.6, keep_plan=rng.random() < 0.4)
    return dict(kind="head", fused=rng.random() < 0.7, vocab=_log_int(rng, 4000, 262144),
                hidden=256 * rng.randint(4, 10), cap=rng.choice([0.0, 30.0]))


# ---- inputs --------------------------------------------------------------------------

class _Inputs:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.gen = torch.Generator(device=self.dev)
        self.gen.manual_seed(1_000_003 * seed + 17)

    def normal(self, *shape, scale=1.0):
        return torch.randn(*shape, generator=self.gen, device=self.dev) * scale

    def norm_weight(self, n, around):
        return (around * (1.0 + 0.1 * self.normal(n))).half()

    def rows(self, n, hd, weight=None):
        """n cache rows of unit RMS, times the norm weight, f16."""
        out = torch.empty(n, hd, dtype=torch.float16, device=self.dev)
        for a in range(0, n, 1 << 18):
            x = self.normal(min(1 << 18, n - a), hd)
            x /= (x.square().mean(dim=1, keepdim=True) + EPS).sqrt()
            out[a:a + x.shape[0]] = x if weight is None else x * weight.float()
        return out

    def weight(self, fmt, rows, n):
        """One projection matrix in its format, as linear_f16 / linear_quant / matmul_* take it."""
        if fmt == "f16":
            return (self.normal(rows, n, scale=0.03).half(),)
        if fmt == "q8":
            q = self.normal(rows, n, scale=40.0).round().clamp(-127, 127).to(torch.int8)
            return q, (0.0007 * (1.0 + 0.2 * torch.rand(rows, n // 32, generator=self.gen, device=self.dev))).half()
        q = torch.randint(-2**31, 2**31, (rows, n // 8), generator=self.gen, device=self.dev, dtype=torch.int64)
        meta = torch.empty(rows, n // 256, 16, device=self.dev)
        scale = 0.006 * (1.0 + 0.2 * torch.rand(rows, n // 256, 8, generator=self.gen, device=self.dev))
        meta[..., :8], meta[..., 8:] = scale, -7.5 * scale
        return q.to(torch.int32), meta.half()

    def rope_freqs(self):
        return torch.tensor(e2b.rope_freqs_f16_bits(256), dtype=torch.int32, device=self.dev).to(torch.int16).view(
            torch.float16)


def _theta(window):
    return (1e4, 0) if window else (1e6, 1)


def _inv_host(window, hd):
    import numpy as np

    theta, div = _theta(window)
    return ops.rope_inv_freq_host(theta, hd, div, np.array(e2b.rope_freqs_f16_bits(256), dtype=np.uint16))


def _step_layers(case):
    """(head_dim, window, producer) of the layers of a step or pair case; producer: the layer whose cache is read."""
    if case["kind"] == "pair":
        cfg = e2b.AttnConfig(num_layers=35)
        pmap = e2b.compute_kv_producer_map(cfg)
        return [(e2b.head_dim(i, cfg), 0 if i in GLOBAL_LAYERS else case["window"], pmap[i]) for i in range(35)]
    n, g = case["layers"], case["globals"]
    every = n // g if g else n + 1
    return [(case["head_dim"], 0 if (i + 1) % every == 0 else case["window"], i) for i in range(n)]


def _lengths(case):
    """The batch's sequence lengths: fixed by the case, so that every state of it is the same work."""
    n, lo, hi = case["sequences"], case["lo"], case["hi"]
    return [lo + (hi - lo) * ((i * 37 + 11) % n) // max(1, n - 1) + (i * 7) % 13 for i in range(n)]


def _entry(x, hd, window, pos, pool_k, pool_v, k_weight, inv, out, rope, producer=None):
    """A step entry on its cache rows; producer: the entry whose raw k/v and cache it shares (KV sharing)."""
    theta, div = _theta(window)
    it = dict(q=x.normal(NQH * hd), q_weight=x.norm_weight(hd, 1.0), rope_freqs=rope, rope_inv_freq_host=inv, out=out,
              seq_len=pos + 1, position=pos, sliding_window=window, theta=theta, apply_divisor=div, scale=1.0, eps=EPS)
    if producer is None:
        it.update(k=x.normal(NKH * hd), v=x.normal(NKH * hd), k_weight=k_weight, k_cache=pool_k, v_cache=pool_v,
                  store_kv=True)
    else:
        it.update({n: producer[n] for n in ("k", "v", "k_weight", "k_cache", "v_cache")}, store_kv=False)
    return it


def prepare(case, seed):
    abi.load()
    return globals()["_prepare_" + case["kind"]](case, _Inputs(seed))


def _prepare_step(case, x):
    layers, pos = _step_layers(case), case["pos"]
    rope, items, caches, outs = x.rope_freqs(), [], {}, {}
    inv = {(w, hd): _inv_host(w, hd) for hd, w, _ in layers}
    for hd in sorted({hd for hd, _, _ in layers}):
        idx = [i for i, L in enumerate(layers) if L[0] == hd]
        outs[hd] = torch.zeros(len(idx), NQH * hd, device=x.dev)
        own = [i for i in idx if layers[i][2] == i]
        kw = {i: x.norm_weight(hd, 0.125) for i in own}
        caches[hd] = (torch.stack([x.rows(pos + 1, hd, kw[i]) for i in own]),
                      x.rows(len(own) * (pos + 1), hd).view(len(own), pos + 1, hd), own, kw, idx)
    for i, (hd, w, p) in enumerate(layers):
        k, v, own, kw, idx = caches[hd]
        j = own.index(p)
        items.append(_entry(x, hd, w, pos, k[j], v[j], kw[p], inv[w, hd], outs[hd][idx.index(i)], rope,
                            None if p == i else items[p]))
    plans, keep = [], []
    for hd in sorted(outs, reverse=True):
        idx = caches[hd][4]
        arr = ops.make_step_entries([items[i] for i in idx], NQH, NKH, hd)
        ws = torch.empty(ops.step_workspace_bytes(len(idx), NQH, NKH, hd), dtype=torch.uint8, device=x.dev)
        plans.append(ops.attn_step_prepare(arr, NQH, NKH, hd, ws))
        keep.append((arr, ws))
    result = {"out%d" % hd: outs[hd] for hd in outs}
    for hd in outs:
        result["k%d" % hd], result["v%d" % hd] = caches[hd][:2]
    return dict(kind=case["kind"], plans=plans, keep=keep, items=items, layers=layers, caches=caches, result=result)


_prepare_pair = _prepare_step


def _prepare_batch(case, x):
    hd, w, lens = case["head_dim"], case["window"], _lengths(case)
    rope, inv, kw = x.rope_freqs(), _inv_host(w, hd), x.norm_weight(hd, 0.125)
    total = sum(lens)
    k, v = x.rows(total, hd, kw), x.rows(total, hd)
    out = torch.zeros(len(lens), NQH * hd, device=x.dev)
    items, at = [], 0
    for i, n in enumerate(lens):
        items.append(_entry(x, hd, w, n - 1, k[at:at + n], v[at:at + n], kw, inv, out[i], rope))
        at += n
    arr = ops.make_step_entries(items, NQH, NKH, hd)
    ws = torch.empty(ops.step_workspace_bytes(len(lens), NQH, NKH, hd), dtype=torch.uint8, device=x.dev)
    return dict(kind="batch", arr=arr, ws=ws, hd=hd, items=items, result={"out": out, "k": k, "v": v})


def _block_layers(case):
    return [(256, case["window"])] * case["locals"] + [(512, 0)] * case["globals"]


def _project(fmt, x, n, mats):
    """One launch over the matrices: mats (weight tensors, out, rows)."""
    segs = [(*w, out, rows) for w, out, rows in mats]
    if fmt == "f16":
        ops.linear_f16(x, n, segs)
    else:
        ops.linear_quant(x, n, fmt, segs)


def _prepare_block(case, x):
    fmt, pos, rope = case["format"], case["pos"], x.rope_freqs()
    layers, result = [], {}
    by_hd = {}
    for i, (hd, w) in enumerate(_block_layers(case)):
        kw = x.norm_weight(hd, 0.125)
        k, v = x.rows(pos + 1, hd, kw), x.rows(pos + 1, hd)
        out, y = torch.zeros(NQH * hd, device=x.dev), torch.zeros(HIDDEN, device=x.dev)
        it = _entry(x, hd, w, pos, k, v, kw, _inv_host(w, hd), out, rope)
        mats = [(x.weight(fmt, rows, HIDDEN), it[t], rows) for t, rows in (("q", NQH * hd), ("k", NKH * hd),
                                                                         ("v", NKH * hd))]
        layers.append(dict(hd=hd, window=w, x=x.normal(HIDDEN), item=it, qkv=mats,
                           o=x.weight(fmt, HIDDEN, NQH * hd), y=y))
        by_hd.setdefault(hd, []).append(i)
        result["%d" % i] = {"y": y, "attn": out, "k": k, "v": v}
    keep = []
    for hd, idx in by_hd.items():
        arr = ops.make_step_entries([layers[i]["item"] for i in idx], NQH, NKH, hd)
        ws = torch.empty(ops.step_layers_workspace_bytes(len(idx), NQH, NKH, hd), dtype=torch.uint8, device=x.dev)
        for i, plan in zip(idx, ops.attn_step_prepare_layers(arr, NQH, NKH, hd, ws)):
            layers[i]["plan"] = plan
        keep.append((arr, ws))

    def token():
        for L in layers:
            n = NQH * L["hd"]
            _project(fmt, L["x"], HIDDEN, L["qkv"])
            if fmt == "f16":
                ops.attn_step_run_attention(L["plan"])
                ops.attn_step_run_out(L["plan"], n, [(L["o"][0], L["y"], HIDDEN)])
            else:
                ops.attn_step_run(L["plan"])
                _project(fmt, L["item"]["out"], n, [(L["o"], L["y"], HIDDEN)])

    token()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        token()
    return dict(kind="block", graph=graph, layers=layers, keep=keep, result=result)


def _prepare_engine(case, x):
    hd, w, pos, fmt = case["head_dim"], case["window"], case["pos"], case["format"]
    theta, div = _theta(w)
    kw = x.norm_weight(hd, 0.125)
    zeros = lambda n: torch.zeros(n, device=x.dev)  # noqa: E731
    s = dict(kind="engine", fmt=fmt, hd=hd, pos=pos, window=w, theta=theta, div=div, x=x.normal(HIDDEN),
             wq=x.weight(fmt, NQH * hd, HIDDEN), wk=x.weight(fmt, NKH * hd, HIDDEN), wv=x.weight(fmt, NKH * hd, HIDDEN),
             wo=x.weight(fmt, HIDDEN, NQH * hd), q_weight=x.norm_weight(hd, 1.0), k_weight=kw, rope=x.rope_freqs(),
             q=zeros(NQH * hd), k=zeros(NKH * hd), v=zeros(NKH * hd), scores=zeros(NQH * (pos + 1)),
             attn=zeros(NQH * hd), y=zeros(HIDDEN), k_cache=x.rows(pos + 1, hd, kw), v_cache=x.rows(pos + 1, hd))
    return s


def _prepare_prefill(case, x):
    hd, T, s0 = case["head_dim"], case["tokens"], case["start"]
    rows, rope = s0 + T, x.rope_freqs()
    preps, entries, result, layers = [], [], {}, []
    for li, w in enumerate([0] * case["globals"] + [case["window"]] * case["locals"]):
        theta, div = _theta(w)
        kw, qw = x.norm_weight(hd, 0.125), x.norm_weight(hd, 1.0)
        kc, vc = x.rows(rows, hd, kw), x.rows(rows, hd)
        q16 = torch.zeros(T, NQH * hd, dtype=torch.float16, device=x.dev)
        out = torch.zeros(T, NQH * hd, device=x.dev)
        vt = torch.zeros(ops.vt_cache_elems(rows, NKH, hd), dtype=torch.float16, device=x.dev) if case["vt"] else None
        raw = dict(q=x.normal(T, NQH * hd), k=x.normal(T, NKH * hd), v=x.normal(T, NKH * hd), q_weight=qw, k_weight=kw)
        common = dict(num_q_heads=NQH, num_kv_heads=NKH, head_dim=hd, theta=theta, apply_divisor=div, rope_freqs=rope,
                      rope_inv_freq=ops.rope_inv_freq(theta, hd, div, rope), k_cache=kc, v_cache=vc, vt_cache=vt,
                      max_seq_len=rows, eps=EPS)
        if vt is not None and s0:  # earlier turns' rows went through the prep too
            first = dict(raw, q=x.normal(s0, NQH * hd), k=x.normal(s0, NKH * hd), v=x.normal(s0, NKH * hd))
            ops.attn_prompt_prep(q_out=torch.empty(s0, NQH * hd, dtype=torch.float16, device=x.dev), n_tokens=s0,
                                 start=0, **first, **common)
        preps.append(dict(q_out=q16, n_tokens=T, start=s0, **raw, **common))
        for c0 in range(0, T, case["chunk"]):
            n = min(case["chunk"], T - c0)
            e = dict(q=q16[c0:], k_cache=kc, v_cache=vc, out=out[c0:], n_tokens=n, start=s0 + c0, sliding_window=w,
                     scale=1.0)
            entries.append(dict(e, vt_cache=vt, vt_rows=rows) if vt is not None else e)
        layers.append(dict(raw, window=w, k_cache=kc, v_cache=vc))
        result["%d" % li] = {"attn": out, "q": q16, "k": kc, "v": vc}
    arr = ops.make_prefill_entries(entries, NQH, NKH, hd)
    ws = torch.empty(ops.prefill_workspace_bytes(arr, NQH, NKH, hd), dtype=torch.uint8, device=x.dev)
    plan = ops.attn_prefill_prepare(arr, NQH, NKH, hd, ws) if case["keep_plan"] else None
    return dict(kind="prefill", preps=preps, arr=arr, ws=ws, plan=plan, hd=hd, layers=layers, result=result)


def _prepare_head(case, x):
    V, H = case["vocab"], case["hidden"]
    w = torch.empty(V, H, dtype=torch.float16, device=x.dev)
    for a in range(0, V, 1 << 16):
        w[a:a + (1 << 16)] = x.normal(min(1 << 16, V - a), H, scale=0.05)
    s = dict(kind="head", fused=case["fused"], V=V, H=H, cap=case["cap"], w=w, x=x.normal(H),
             logits=torch.zeros(V, device=x.dev), top=torch.zeros(1, dtype=torch.int32, device=x.dev))
    if case["fused"]:
        s["ws"] = torch.empty(ops.lm_head_workspace_bytes(V, H, case["cap"]), dtype=torch.uint8, device=x.dev)
    return s


# ---- one pass --------------------------------------------------------------------------

def run(s):
    return globals()["_run_" + s["kind"]](s)


def _run_step(s):
    ops.attn_step_run(s["plans"][0])
    return s["result"]


def _run_pair(s):
    ops.attn_step_run_pair(*s["plans"])
    return s["result"]


def _run_batch(s):
    ops.attn_step(s["arr"], NQH, NKH, s["hd"], s["ws"])
    return s["result"]


def _run_block(s):
    s["graph"].replay()
    return s["result"]


def _matmul(fmt, x, w, out, M, N):
    {"f16": ops.matmul_quant_f16, "q8": ops.matmul_q8, "q4k": ops.matmul_q4k}[fmt](x, *w, out, M, N)


def _run_engine(s):
    hd, pos, n, fmt = s["hd"], s["pos"], s["pos"] + 1, s["fmt"]
    _matmul(fmt, s["x"], s["wq"], s["q"], NQH * hd, HIDDEN)
    _matmul(fmt, s["x"], s["wk"], s["k"], NKH * hd, HIDDEN)
    _matmul(fmt, s["x"], s["wv"], s["v"], NKH * hd, HIDDEN)
    ops.per_head_rms_norm_no_weight(s["v"], NKH, hd, EPS)
    ops.fused_per_head_norm_rope(s["q"], s["q_weight"], s["rope"], NQH, hd, EPS, pos, s["theta"], s["div"])
    ops.fused_per_head_norm_rope(s["k"], s["k_weight"], s["rope"], NKH, hd, EPS, pos, s["theta"], s["div"])
    ops.kv_cache_store(s["k"], s["v"], s["k_cache"], s["v_cache"], NKH, hd, pos, n)
    ops.attn_score(s["q"], s["k_cache"], s["scores"], NQH, NKH, hd, n, 1.0, s["window"])
    ops.softmax(s["scores"], NQH, n)
    ops.attn_output(s["scores"], s["v_cache"], s["attn"], NQH, NKH, hd, n)
    _matmul(fmt, s["attn"], s["wo"], s["y"], HIDDEN, NQH * hd)
    return {t: s[t] for t in ("q", "k", "v", "k_cache", "v_cache", "scores", "attn", "y")}


def _run_prefill(s):
    ops.attn_prompt_prep_many(s["preps"])
    if s["plan"] is not None:
        ops.attn_prefill_run(s["plan"])
    else:
        ops.attn_prefill(s["arr"], NQH, NKH, s["hd"], s["ws"])
    return s["result"]


def _run_head(s):
    if s["fused"]:
        ops.lm_head_argmax(s["x"], s["w"], s["logits"], s["top"], s["ws"], s["V"], s["H"], s["cap"])
    else:
        ops.matmul_quant_f16(s["x"], s["w"], s["logits"], s["V"], s["H"])
        if s["cap"] > 0:
            ops.logit_softcap(s["logits"], s["V"], s["cap"])
        ops.argmax(s["logits"], s["top"], s["V"])
    return {"logits": s["logits"], "top": s["top"]}


# ---- what a pass cannot do without ---------------------------------------------------------

def _attended(seq, window):
    return min(seq, window) if window else seq


def _attention_work(seq, window, hd):
    """Bytes and flops of one entry: attended K and V rows (f16) once, q and attnOut (f32)."""
    n = _attended(seq, window)
    return 2 * n * NKH * hd * 2 + 2 * NQH * hd * 4, 4 * n * NQH * hd


def _weight_bytes(fmt, rows, n):
    return {"f16": 2 * rows * n, "q8": rows * n + rows * n // 16, "q4k": rows * n // 2 + rows * n // 8}[fmt]


def _projection_work(fmt, hd):
    qkv = (NQH + 2 * NKH) * hd
    b = _weight_bytes(fmt, qkv, HIDDEN) + _weight_bytes(fmt, HIDDEN, NQH * hd) + 4 * (2 * HIDDEN + qkv + NQH * hd)
    return b, 2 * (qkv * HIDDEN + HIDDEN * NQH * hd)


def work(case):
    kind = case["kind"]
    parts = []
    if kind in ("step", "pair"):
        seen = set()
        for hd, w, p in _step_layers(case):
            b, f = _attention_work(case["pos"] + 1, w, hd)
            if p in seen:  # a shared cache's rows are read once
                b -= 2 * _attended(case["pos"] + 1, w) * NKH * hd * 2
            seen.add(p)
            parts.append((b, f))
    elif kind == "batch":
        parts = [_attention_work(n, case["window"], case["head_dim"]) for n in _lengths(case)]
    elif kind == "block":
        for hd, w in _block_layers(case):
            parts += [_attention_work(case["pos"] + 1, w, hd), _projection_work(case["format"], hd)]
    elif kind == "engine":  # the six kernels' buffers in between are outputs too: scores written once
        hd, n = case["head_dim"], case["pos"] + 1
        parts = [_attention_work(n, case["window"], hd), _projection_work(case["format"], hd), (4 * NQH * n, 0)]
    elif kind == "prefill":
        hd, T, s0 = case["head_dim"], case["tokens"], case["start"]
        for w in [0] * case["globals"] + [case["window"]] * case["locals"]:
            pairs = sum(_attended(s0 + t + 1, w) for t in range(T))
            rows = s0 + T - (max(0, s0 + 1 - w) if w else 0)
            b = T * (NQH + 2 * NKH) * hd * 4 + T * NQH * hd * 2 + 2 * T * NKH * hd * 2  # prep: raw in, f16 out
            b += 2 * (rows - T) * NKH * hd * 2 + T * NQH * hd * 4                        # earlier rows, attnOut
            parts.append((b, 4 * pairs * NQH * hd))
    else:
        V, H = case["vocab"], case["hidden"]
        parts = [(2 * V * H + 4 * H + 4 * V, 2 * V * H)]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    """Largest relative error (2-norm) that another correct implementation shows: f32 accumulation in another order
    moves GEMV rows and attention outputs by under 1e-6 of their norm; rows rounded to f16 on the way (the stored K/V row,
    the prefill's q and probabilities) can fall to the neighbouring value."""
    kind = case["kind"]
    if kind == "prefill":
        return {"rel": 2e-3, "max": 2e-2}
    if kind in ("head", "engine"):
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 2e-5, "max": 2e-3}


# ---- the same in 64 bits -----------------------------------------------------------------

def _inv64(window, hd):
    """The inverse frequencies as the model defines them: f32 values of 1 / pow(theta, 2 i / hd), divided by the
    proportional table on global layers (1 for the first 64 pairs, infinite after them)."""
    theta, div = _theta(window)
    i = torch.arange(hd // 2, dtype=torch.float64, device="cuda")
    e = (2 * i / hd).float().double()
    inv = (1.0 / torch.tensor(theta, dtype=torch.float64, device="cuda").pow(e).float()).double()
    if div:
        inv = torch.where(i < 64, inv, torch.zeros_like(inv))
    return inv.float()


def _norm64(x, weight=None):
    x = x.double()
    y = x / (x.square().mean(dim=-1, keepdim=True) + EPS).sqrt()
    return y if weight is None else y * weight.double()


def _rope64(x, pos, window):
    """x [..., hd] at positions pos [T] (x [T, heads, hd]): the angle is the f32 product, cos and sin in 64 bits."""
    hd = x.shape[-1]
    a = (pos.float()[:, None] * _inv64(window, hd)).double()[:, None, :]
    c, s = a.cos(), a.sin()
    x0, x1 = x[..., :hd // 2], x[..., hd // 2:]
    return torch.cat([x0 * c - x1 * s, x0 * s + x1 * c], dim=-1)


def _prep64(q, k, v, qw, kw, pos, window, hd):
    """Post-norm, post-RoPE q [T, NQH, hd], k and v [T, hd]."""
    q64 = _rope64(_norm64(q.view(-1, NQH, hd), qw), pos, window)
    k64 = _rope64(_norm64(k.view(-1, NKH, hd), kw), pos, window)
    return q64, k64[:, 0], _norm64(v.view(-1, hd))


def _attend64(q, k, v, lo):
    p = (q @ k[lo:].T).softmax(dim=-1)
    return p @ v[lo:]


def _decode64(it, hd, window, pos, kc, vc):
    """(attnOut, k row, v row) of one step entry whose raw q/k/v and cache rows are given."""
    at = torch.tensor([pos], device="cuda")
    q, k, v = _prep64(it["q"], it["k"], it["v"], it["q_weight"], it["k_weight"], at, window, hd)
    lo = max(0, pos + 1 - window) if window else 0
    K = torch.cat([kc[lo:pos].double(), k])
    V = torch.cat([vc[lo:pos].double(), v])
    return _attend64(q[0], K, V, 0).reshape(-1), k[0], v[0]


def _dequant64(fmt, w, rows, n):
    if fmt == "f16":
        return w[0].double()
    if fmt == "q8":
        return w[0].double() * w[1].double().repeat_interleave(32, dim=1)
    q, meta = w
    shifts = torch.arange(0, 32, 4, device=q.device)
    nib = ((q.long()[..., None] >> shifts) & 15).reshape(rows, n).double()
    m = meta.double()
    s, b = (m[..., :8].reshape(rows, n // 32), m[..., 8:].reshape(rows, n // 32))
    return nib * s.repeat_interleave(32, dim=1) + b.repeat_interleave(32, dim=1)


def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, prepare(case, seed))


def _exact_step(case, s):
    r = {n: t.double() for n, t in s["result"].items()}
    for i, (hd, w, p) in enumerate(s["layers"]):
        k, v, own, _, idx = s["caches"][hd]
        j = own.index(p)
        o, kr, vr = _decode64(s["items"][i], hd, w, case["pos"], k[j], v[j])
        r["out%d" % hd][idx.index(i)] = o
        if p == i:
            r["k%d" % hd][j, case["pos"]], r["v%d" % hd][j, case["pos"]] = kr, vr
    return r


_exact_pair = _exact_step


def _exact_batch(case, s):
    r = {n: t.double() for n, t in s["result"].items()}
    at = 0
    for i, n in enumerate(_lengths(case)):
        it = s["items"][i]
        o, kr, vr = _decode64(it, case["head_dim"], case["window"], n - 1, it["k_cache"], it["v_cache"])
        r["out"][i], r["k"][at + n - 1], r["v"][at + n - 1] = o, kr, vr
        at += n
    return r


def _exact_block(case, s):
    r, fmt = {}, case["format"]
    for i, L in enumerate(s["layers"]):
        hd, it = L["hd"], L["item"]
        raw = [_dequant64(fmt, w, rows, HIDDEN) @ L["x"].double() for w, _, rows in L["qkv"]]
        o, kr, vr = _decode64(dict(it, q=raw[0], k=raw[1], v=raw[2]), hd, L["window"], case["pos"], it["k_cache"],
                              it["v_cache"])
        k, v = it["k_cache"].double(), it["v_cache"].double()
        k[-1], v[-1] = kr, vr
        r["%d" % i] = {"y": _dequant64(fmt, L["o"], HIDDEN, NQH * hd) @ o, "attn": o, "k": k, "v": v}
    return r


def _exact_engine(case, s):
    hd, pos, w, fmt = s["hd"], s["pos"], s["window"], s["fmt"]
    raw = [_dequant64(fmt, s[t], rows, HIDDEN) @ s["x"].double()
           for t, rows in (("wq", NQH * hd), ("wk", NKH * hd), ("wv", NKH * hd))]
    at = torch.tensor([pos], device="cuda")
    q, k, v = _prep64(*raw, s["q_weight"], s["k_weight"], at, w, hd)
    K, V = s["k_cache"].double(), s["v_cache"].double()
    K[pos], V[pos] = k[0], v[0]
    z = q[0] @ K.T
    if w and pos + 1 > w:
        z[:, :pos + 1 - w] = -float("inf")
    p = z.softmax(dim=-1)
    o = (p @ V).reshape(-1)
    return {"q": q.reshape(-1), "k": k.reshape(-1), "v": v.reshape(-1), "k_cache": K, "v_cache": V,
            "scores": p.reshape(-1), "attn": o, "y": _dequant64(fmt, s["wo"], HIDDEN, NQH * hd) @ o}


def _exact_prefill(case, s):
    hd, T, s0, r = case["head_dim"], case["tokens"], case["start"], {}
    pos = s0 + torch.arange(T, device="cuda")
    for li, L in enumerate(s["layers"]):
        w = L["window"]
        q, k, v = _prep64(L["q"], L["k"], L["v"], L["q_weight"], L["k_weight"], pos, w, hd)
        K, V = L["k_cache"].double(), L["v_cache"].double()
        K[s0:], V[s0:] = k, v
        out = torch.empty(T, NQH, hd, dtype=torch.float64, device="cuda")
        keys = torch.arange(s0 + T, device="cuda")
        for a in range(0, T, 256):
            p = pos[a:a + 256]
            live = keys[None] <= p[:, None]
            if w:
                live &= keys[None] > p[:, None] - w
            z = (q[a:a + 256].reshape(-1, hd) @ K.T).view(-1, NQH, s0 + T)
            z = z.masked_fill(~live[:, None], -float("inf")).softmax(dim=-1)
            out[a:a + 256] = (z.reshape(-1, s0 + T) @ V).view(-1, NQH, hd)
        r["%d" % li] = {"attn": out.reshape(T, -1), "q": q.reshape(T, -1), "k": K, "v": V}
    return r


def _exact_head(case, s):
    z = torch.empty(case["vocab"], dtype=torch.float64, device="cuda")
    for a in range(0, case["vocab"], 1 << 15):
        z[a:a + (1 << 15)] = s["w"][a:a + (1 << 15)].double() @ s["x"].double()
    if case["cap"] > 0:
        z = (z / case["cap"]).tanh() * case["cap"]
    return {"logits": z, "top": z.argmax().to(torch.int32).reshape(1)}
