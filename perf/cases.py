"""Performance cases of the paged KV-cache path: what one serving process has it do, sized by use.

A case is a dict of plain values.  ``listed()`` names twelve of them and ``draw(rng)`` gives more of
the same ranges; ``prepare`` builds what a server holds before the call (pools, block tables,
activations of a few decoder layers, a captured graph where the engine replays one), ``run`` makes one
pass through the public entry points and returns everything it computes, ``work`` says what such a pass
cannot do without and ``exact`` recomputes it in 64-bit torch.

Kinds:
  step         a captured decode step, every elementwise piece around the projections included:
               rms_norm, rope_decode_attention, rms_norm with the residual, silu_mul, per layer
  decode       a captured decode step's attention calls (append + attention), per layer
  verify       speculative verify, eager: s_q draft rows per sequence, over private contexts or over
               one cached prefix the whole batch shares
  prefill      prompt chunks onto cached prefixes, eager
  elementwise  a prefill chunk's elementwise pieces, eager: rms_norm, rope_qk with the paged append,
               rms_norm with the residual, silu_mul
"""
from __future__ import annotations

import math

import numpy as np
import torch

import prism_amd

PAGE = 256
# decoder shapes of prism_amd.workloads, with the hidden and MLP widths of the same models
SHAPES = {
    "0.5B": dict(n_heads=14, n_kv=2, head_dim=64, layers=24, hidden=896, mlp=4864),
    "7B": dict(n_heads=28, n_kv=4, head_dim=128, layers=28, hidden=3584, mlp=18944),
    "14B": dict(n_heads=40, n_kv=8, head_dim=128, layers=48, hidden=5120, mlp=13824),
    # one GPU of a 4-way tensor-parallel 7B: its heads and its share of the MLP
    "7B-tp4": dict(n_heads=7, n_kv=1, head_dim=128, layers=28, hidden=3584, mlp=4736),
}
MAX_KEYS = 32768           # the longest context a sequence may reach
MAX_POOL_BYTES = 6 << 30   # of one state's K and V pools
MAX_FLOPS = 3.8e11         # of one pass


def listed() -> list[dict]:
    return [
        # a draft model's decode step for a few users: the smallest kernels, 4 launches per layer
        dict(name="step_05b_b4", kind="step", shape="0.5B", layers=24, batch=4, s_q=1, spread="uniform", ctx=1024,
             prefix=0, lengths=1),
        # a lightly loaded 7B server: 8 sequences at 2048 tokens
        dict(name="decode_7b_b8", kind="decode", shape="7B", layers=28, batch=8, s_q=1, spread="same", ctx=2048,
             prefix=0, lengths=0),
        # continuous batching, the headline: 32 ragged sequences
        dict(name="decode_7b_b32", kind="decode", shape="7B", layers=28, batch=32, s_q=1, spread="lognormal",
             ctx=1500, prefix=0, lengths=0),
        # a few long documents on the larger model
        dict(name="decode_14b_long", kind="decode", shape="14B", layers=12, batch=6, s_q=1, spread="lognormal",
             ctx=9000, prefix=0, lengths=3),
        # speculative verify of 64 branches of one cached prompt
        dict(name="verify_7b_shared", kind="verify", shape="7B", layers=4, batch=64, s_q=5, spread="uniform",
             ctx=1024, prefix=2048, lengths=0),
        # speculative verify of 8 unrelated conversations
        dict(name="verify_7b_b8", kind="verify", shape="7B", layers=4, batch=8, s_q=5, spread="lognormal", ctx=1500,
             prefix=0, lengths=5),
        # a short question to the draft model: the smallest eager calls, two launches each
        dict(name="prompt_05b_short", kind="prefill", shape="0.5B", layers=24, batch=1, s_q=45, spread="same", ctx=0,
             prefix=0, lengths=0),
        # a few prompts at once on the draft model (head_dim 64), some on a cached system prompt
        dict(name="prompts_05b", kind="prefill", shape="0.5B", layers=8, batch=4, s_q=1000, spread="uniform",
             ctx=1000, prefix=0, lengths=2),
        # the next turn of one long conversation: few new tokens, a long cached prefix
        dict(name="turn_7b", kind="prefill", shape="7B", layers=4, batch=1, s_q=150, spread="same", ctx=3500,
             prefix=0, lengths=0),
        # one whole prompt
        dict(name="prompt_7b", kind="prefill", shape="7B", layers=2, batch=1, s_q=4096, spread="same", ctx=0,
             prefix=0, lengths=0),
        # chunked prefill beside each other: 8 chunks of 512 onto ragged prefixes
        dict(name="chunks_14b", kind="prefill", shape="14B", layers=2, batch=8, s_q=512, spread="uniform", ctx=4096,
             prefix=0, lengths=0),
        # the elementwise pieces around those chunks
        dict(name="elementwise_14b", kind="elementwise", shape="14B", layers=2, batch=8, s_q=512, spread="uniform",
             ctx=4096, prefix=0, lengths=0),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    while True:
        kind = rng.choice(["step", "decode", "decode", "verify", "verify", "prefill", "prefill", "prefill",
                           "elementwise"])
        shape = rng.choice(["0.5B", "7B", "7B", "14B", "7B-tp4"])
        c = dict(kind=kind, shape=shape, prefix=0, lengths=rng.randrange(1 << 20))
        c["spread"] = rng.choice(["same", "uniform", "lognormal"])
        if kind in ("step", "decode"):
            c.update(layers=rng.choice([8, 12, 16]), batch=_log_int(rng, 1, 64), s_q=1, ctx=_log_int(rng, 16, 20000))
        elif kind == "verify":
            c.update(layers=4, batch=_log_int(rng, 2, 64), s_q=rng.randint(2, 6), ctx=_log_int(rng, 16, 6000))
            if rng.random() < 0.5:
                c.update(prefix=_log_int(rng, 300, 8000), spread="uniform", ctx=_log_int(rng, 16, 1200))
        elif kind == "prefill":
            c.update(layers=rng.choice([1, 2, 4]), batch=_log_int(rng, 1, 8), s_q=_log_int(rng, 20, 4096),
                     ctx=rng.choice([0, _log_int(rng, 16, 8000)]))
        else:
            c.update(layers=2, batch=_log_int(rng, 1, 8), s_q=_log_int(rng, 32, 1024), ctx=_log_int(rng, 16, 4000))
        if c["ctx"] == 0:
            c["spread"] = "same"
        s = SHAPES[shape]
        pool = _pool_pages(c) * PAGE * s["n_kv"] * s["head_dim"] * 4 * c["layers"]
        w = work(c)
        if pool <= MAX_POOL_BYTES and w["flops"] <= MAX_FLOPS and w["bytes"] <= 6e9:
            return c


# ---------------------------------------------------------------------------------- lengths and pages
def _contexts(case: dict) -> np.ndarray:
    """Cached keys of each sequence before the call (behind a shared prefix: the private suffixes)."""
    rng = np.random.default_rng(case["lengths"])
    n, ctx, room = case["batch"], case["ctx"], MAX_KEYS - case["s_q"] - case["prefix"]
    if case["spread"] == "same":
        c = np.full(n, ctx)
    elif case["spread"] == "uniform":
        c = rng.integers(0 if case["prefix"] or case["kind"] in ("prefill", "elementwise") else 1, ctx + 1, size=n)
    else:
        c = np.clip(np.round(rng.lognormal(math.log(ctx), 1.0, size=n)), 16, MAX_KEYS)
    return np.minimum(c, room).astype(np.int64)


def _shared_tokens(case: dict) -> int:
    """Tokens of the shared prompt: its last page is partly filled, as prompts end anywhere."""
    if not case["prefix"]:
        return 0
    return case["prefix"] - int(np.random.default_rng(case["lengths"] + 1).integers(1, PAGE))


def _pool_pages(case: dict) -> int:
    keys = _contexts(case) + case["s_q"] + _shared_tokens(case) % PAGE
    need = int(np.ceil(keys / PAGE).sum()) + case["batch"] + _shared_tokens(case) // PAGE + 2
    return int(need * 1.5) + 4


def _randn(shape, g, dev, scale=1.0) -> torch.Tensor:
    return torch.empty(shape, dtype=torch.bfloat16, device=dev).normal_(0.0, scale, generator=g)


def _paged(case: dict, g, seed: int):
    """A pool of N(0, 1) keys and values, the batch's pages scattered over it in a seeded order."""
    s, dev = SHAPES[case["shape"]], torch.device("cuda:0")
    kv = prism_amd.FlashAttnKVCache(case["layers"], s["n_kv"], s["head_dim"], _pool_pages(case), PAGE, dev,
                                    torch.bfloat16)
    kv.k_pool.normal_(0.0, 1.0, generator=g)
    kv.v_pool.normal_(0.0, 1.0, generator=g)
    kv.free_pages = [int(p) for p in np.random.default_rng(seed).permutation(kv.max_pages)]
    ids = list(range(case["batch"]))
    ctx, shared = _contexts(case), _shared_tokens(case)
    if shared:
        root = len(ids)
        kv.new_sequence(root)
        kv._ensure_capacity(root, shared)
        kv.seq_len[root] = shared
        for i in ids:
            kv.fork_sequence(root, i)
        kv.free_sequence(root)
    else:
        for i in ids:
            kv.new_sequence(i)
    kv.prepare_append(ids, [int(c) for c in ctx])
    for i, c in zip(ids, ctx):
        kv.seq_len[i] += int(c)
    kv.prepare_append(ids, case["s_q"])
    bt, sl = kv.build_block_table(ids)
    return kv, bt, sl


def _state(case: dict, seed: int) -> dict:
    s, dev = SHAPES[case["shape"]], torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    kv, bt, sl = _paged(case, g, seed)
    L, B, S, nh, nk, hd = case["layers"], case["batch"], case["s_q"], s["n_heads"], s["n_kv"], s["head_dim"]
    st = dict(case=case, kv=kv, bt=bt, sl=sl)
    # the fused projection's output; rotary leaves q and k in tensors of their own, v stays a view
    st["qkv"] = [_randn((B, S, (nh + 2 * nk) * hd), g, dev) for _ in range(L)]
    if case["kind"] in ("decode", "verify", "prefill"):
        st["q"] = [_randn((B, S, nh, hd), g, dev) for _ in range(L)]
        st["k"] = [_randn((B, S, nk, hd), g, dev) for _ in range(L)]
        st["v"] = [t[:, :, (nh + nk) * hd:].unflatten(2, (nk, hd)) for t in st["qkv"]]
        return st
    m = s["mlp"]
    st["cos"], st["sin"] = prism_amd.rope_tables(hd, MAX_KEYS + 1, 1e6, dev)
    st["x"] = [_randn((B, S, s["hidden"]), g, dev) for _ in range(L)]
    st["o"] = [_randn((B, S, s["hidden"]), g, dev) for _ in range(L)]
    st["gu"] = [_randn((B, S, 2 * m), g, dev, 2.0) for _ in range(L)]
    st["w"] = [[_randn((s["hidden"],), g, dev, 0.1).add_(1.0) for _ in range(2)] for _ in range(L)]
    return st


# ---------------------------------------------------------------------------------- one pass
def _attention(st: dict, l: int, out=None) -> torch.Tensor:
    kv = st["kv"]
    return prism_amd.flash_attn_with_kvcache(st["q"][l], kv.k_caches[l], kv.v_caches[l], k=st["k"][l], v=st["v"][l],
                                             cache_seqlens=st["sl"], block_table=st["bt"], causal=True, out=out)


def _step_layer(st: dict, l: int) -> None:
    s, kv, o = SHAPES[st["case"]["shape"]], st["kv"], st["outs"]
    m = s["mlp"]
    prism_amd.rms_norm(st["x"][l], st["w"][l][0], out=o["norm"][l])
    prism_amd.rope_decode_attention(st["qkv"][l], kv.k_caches[l], kv.v_caches[l], st["cos"], st["sin"],
                                    cache_seqlens=st["sl"], block_table=st["bt"], n_heads=s["n_heads"],
                                    n_kv=s["n_kv"], out=o["attn"][l])
    prism_amd.rms_norm(st["o"][l], st["w"][l][1], residual=st["x"][l], out=o["norm2"][l], h_out=o["hidden"][l])
    prism_amd.silu_mul(st["gu"][l][..., :m], st["gu"][l][..., m:], out=o["act"][l])


def _elementwise_layer(st: dict, l: int) -> dict:
    s, kv = SHAPES[st["case"]["shape"]], st["kv"]
    m = s["mlp"]
    norm = prism_amd.rms_norm(st["x"][l], st["w"][l][0])
    q, k = prism_amd.rope_qk(st["qkv"][l], st["sl"], st["cos"], st["sin"], s["n_heads"], s["n_kv"],
                             k_cache=kv.k_caches[l], v_cache=kv.v_caches[l], block_table=st["bt"],
                             cache_seqlens=st["sl"])
    norm2, hidden = prism_amd.rms_norm(st["o"][l], st["w"][l][1], residual=st["x"][l])
    act = prism_amd.silu_mul(st["gu"][l][..., :m], st["gu"][l][..., m:])
    return dict(norm=norm, q=q, k=k, norm2=norm2, hidden=hidden, act=act)


def prepare(case: dict, seed: int) -> dict:
    st = _state(case, seed)
    if case["kind"] not in ("step", "decode"):
        return st
    # the engine's decode step: warmed up on the current stream, captured once, then replayed
    s, dev = SHAPES[case["shape"]], torch.device("cuda:0")
    L, B, S = case["layers"], case["batch"], case["s_q"]

    def buf(*shape):
        return torch.empty((L, B, S) + shape, dtype=torch.bfloat16, device=dev)

    st["outs"] = dict(attn=buf(s["n_heads"], s["head_dim"]))
    if case["kind"] == "step":
        st["outs"].update(norm=buf(s["hidden"]), norm2=buf(s["hidden"]), hidden=buf(s["hidden"]), act=buf(s["mlp"]))

    def layer(l):
        if case["kind"] == "step":
            _step_layer(st, l)
        else:
            _attention(st, l, st["outs"]["attn"][l])

    layer(0)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for l in range(L):
            layer(l)
    st["graph"] = graph
    return st


def run(st: dict):
    kind, kv = st["case"]["kind"], st["kv"]
    cache = dict(k_pool=kv.k_pool, v_pool=kv.v_pool)
    if "graph" in st:
        st["graph"].replay()
        return dict(st["outs"], **cache)
    if kind == "elementwise":
        return dict(layers=[_elementwise_layer(st, l) for l in range(kv.num_layers)], **cache)
    return dict(attn=[_attention(st, l) for l in range(kv.num_layers)], **cache)


# ---------------------------------------------------------------------------------- what a pass needs
def work(case: dict) -> dict:
    s = SHAPES[case["shape"]]
    L, B, S, nh, nk, hd = case["layers"], case["batch"], case["s_q"], s["n_heads"], s["n_kv"], s["head_dim"]
    rows, kv_row = B * S, nk * hd * 2 * 2          # kv_row: one token's K and V
    shared = _shared_tokens(case)
    ctx = _contexts(case) + shared
    table = 4 * (int(np.ceil((ctx + S) / PAGE).sum()) + B)
    flops = nbytes = 0.0
    if case["kind"] != "elementwise":
        # cached keys once (a shared prefix once for the batch), new rows read and written, q and out
        cached = int(ctx.sum()) - shared // PAGE * PAGE * (B - 1) if shared else int(ctx.sum())
        nbytes += cached * kv_row + rows * kv_row * 2 + rows * nh * hd * 2 * 2 + table
        visible = float(((ctx + 1) * S + S * (S - 1) / 2).sum())
        flops += 4.0 * nh * hd * visible
    if case["kind"] == "elementwise":
        # qkv in; q, k and the two cache rows out
        nbytes += rows * ((nh + 2 * nk) * hd * 2 + nh * hd * 2 + nk * hd * 2 + kv_row + 2 * hd * 2) + table
    if case["kind"] in ("step", "elementwise"):
        # rms_norm: x in, norm out; with the residual: o and x in, norm and hidden out; silu_mul
        nbytes += rows * (s["hidden"] * 2 * 6 + s["mlp"] * 2 * 3) + 2 * s["hidden"] * 2
        flops += rows * (s["hidden"] * 9 + s["mlp"] * 5)
    return dict(bytes=nbytes * L, flops=flops * L)


def tolerance(case: dict) -> dict:
    # bf16 outputs of fp32 sums: about 2.5e-3 from 64 bits (P and the outputs rounded to bf16)
    return {"rel": 1e-2, "max": 0.1}


# ---------------------------------------------------------------------------------- 64-bit reference
def _rms64(x, w, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _rope64(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos + torch.cat([-x[..., half:], x[..., :half]], -1) * sin


def _attention64(st: dict, l: int, q, k, v) -> torch.Tensor:
    """Causal attention of one layer, sequence by sequence: q [B, S, nh, hd], new rows k and v."""
    kv, case = st["kv"], st["case"]
    B, S, nh, hd = q.shape
    nk = k.shape[2]
    g = nh // nk
    bt, sl = st["bt"].cpu(), st["sl"].cpu().tolist()
    out = torch.empty((B, S, nh, hd), dtype=torch.float64, device=q.device)
    for b, c in enumerate(sl):
        pages = bt[b, :-(-c // PAGE)].long().to(q.device)
        past_k = kv.k_caches[l][pages].reshape(-1, nk, hd)[:c].double()
        past_v = kv.v_caches[l][pages].reshape(-1, nk, hd)[:c].double()
        keys, vals = torch.cat([past_k, k[b].double()]), torch.cat([past_v, v[b].double()])
        seen = torch.arange(c + S, device=q.device)[None] <= torch.arange(c, c + S, device=q.device)[:, None]
        for h in range(nk):
            qh = q[b, :, h * g:(h + 1) * g].double().transpose(0, 1).reshape(g * S, hd)
            sc = (qh @ keys[:, h].contiguous().t().contiguous()) / math.sqrt(hd)
            sc.view(g, S, -1).masked_fill_(~seen, -math.inf)
            o = torch.softmax(sc, -1) @ vals[:, h].contiguous()
            out[b, :, h * g:(h + 1) * g] = o.view(g, S, hd).transpose(0, 1)
    return out


def exact(case: dict, seed: int):
    st = _state(case, seed)
    s, L = SHAPES[case["shape"]], case["layers"]
    none = dict(k_pool=None, v_pool=None)
    if "q" in st:
        a = [_attention64(st, l, st["q"][l], st["k"][l], st["v"][l]) for l in range(L)]
        return dict(none, attn=torch.stack(a) if case["kind"] == "decode" else a)
    nh, nk, hd, m = s["n_heads"], s["n_kv"], s["head_dim"], s["mlp"]
    pos = st["sl"].long()[:, None] + torch.arange(case["s_q"], device=st["sl"].device)[None]
    cos, sin = (st[n][pos].double()[:, :, None] for n in ("cos", "sin"))
    layers = []
    for l in range(L):
        qkv = st["qkv"][l]
        q = _rope64(qkv[..., :nh * hd].unflatten(2, (nh, hd)).double(), cos, sin)
        k = _rope64(qkv[..., nh * hd:(nh + nk) * hd].unflatten(2, (nk, hd)).double(), cos, sin)
        v = qkv[..., (nh + nk) * hd:].unflatten(2, (nk, hd)).double()
        x, h = st["x"][l].double(), st["x"][l].double() + st["o"][l].double()
        gate, up = st["gu"][l][..., :m].double(), st["gu"][l][..., m:].double()
        d = dict(norm=_rms64(x, st["w"][l][0]), norm2=_rms64(h, st["w"][l][1]), hidden=h,
                 act=gate / (1 + torch.exp(-gate)) * up)
        d.update(dict(attn=_attention64(st, l, q, k, v)) if case["kind"] == "step" else dict(q=q, k=k))
        layers.append(d)
    if case["kind"] == "step":
        return dict(none, **{n: torch.stack([d[n] for d in layers]) for n in layers[0]})
    return dict(none, layers=layers)
