"""prefill_tile_kernel at the sizes where its pipeline, its rows and its pages can go wrong: every
count of key stages around the ring depths (an odd count does its first stage apart, the rings
hold 4), row blocks with a remainder, rows that see no key, pages of exactly one stage,
both head dims, with stale NaN behind every sequence.  Against the fp64 oracle at the bf16 tolerance."""
import numpy as np
import pytest
import torch

import prism_amd
from oracle import paged_attention as pa
from pkv_testutil import assert_attn_close, make_paged_case

pytestmark = pytest.mark.gpu

# head_dim, n_heads, n_kv, page, s_q, prefixes
CASES = [
    # 1 .. 12 stages of 32 tokens (head_dim 128), one sequence each
    (128, 14, 2, 32, 19, [0, 14, 46, 77, 110, 141, 172, 206, 237, 269, 301, 333]),
    # 1 .. 8 stages of 64 tokens (head_dim 64)
    (64, 14, 2, 64, 19, [0, 46, 110, 173, 238, 301, 365, 429]),
    # 128-row blocks: one row short, full, one row over, at a group size that does not divide them
    (128, 5, 1, 256, 51, [3, 250]),
    (64, 4, 4, 256, 128, [0, 64, 1]),
    (64, 14, 2, 128, 37, [0, 63, 65, 1000]),
    # pages smaller than a stage keep the per-wave kernel
    (64, 14, 2, 32, 40, [0, 31, 100]),
    (128, 8, 2, 16, 40, [0, 17, 100]),
]


def _nan_behind(d, ctx, s_q, page):
    """Every slot past a sequence's keys in its last page holds NaN."""
    for b, c in enumerate(ctx):
        end = int(c) + s_q
        last = int(d["block_table"][b, (end - 1) // page])
        for cache in (d["k_cache"], d["v_cache"]):
            cache[last, (end - 1) % page + 1:] = float("nan")


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("case", CASES, ids=[f"hd{c[0]}-p{c[3]}-s{c[4]}-g{c[1] // c[2]}" for c in CASES])
def test_prefill_stage_and_row_edges(gpu, case, causal):
    hd, nh, nk, page, s_q, ctx = case
    cpu, d = make_paged_case(gpu, batch=len(ctx), ctx=ctx, page_size=page, n_kv=nk, n_heads=nh, head_dim=hd, s_q=s_q,
                             seed=hd + page + s_q)
    _nan_behind(d, ctx, s_q, page)
    out = torch.full((len(ctx), s_q, nh, hd), float("nan"), dtype=torch.bfloat16, device=gpu)
    prism_amd.prefill_attention(d["q"], d["k_cache"], d["v_cache"], d["k"], d["v"], cache_seqlens=d["cache_seqlens"],
                                block_table=d["block_table"], causal=causal, out=out)
    ref, _, _ = pa.flash_attn_with_kvcache_ref(cpu["q"], cpu["k_cache"], cpu["v_cache"], cpu["k"], cpu["v"],
                                               cache_seqlens=cpu["cache_seqlens"], block_table=cpu["block_table"],
                                               causal=causal)
    torch.cuda.synchronize()
    # rows that see a handful of keys: the output's own bf16 rounding passes 1e-2 where |o| > 2
    few = np.array([[causal and c + j + 1 <= 8 for j in range(s_q)] for c in ctx])
    got = out.float().cpu().numpy()
    assert np.isfinite(got).all()
    err = np.abs(got - ref)
    ulp = np.maximum(1e-2, np.abs(ref) * 2.0 ** -7)
    assert (err[few] <= ulp[few]).all() and err[~few].max(initial=0.0) <= 1e-2 and err.mean() <= 1e-3
    assert prism_amd.read_status(gpu) == 0


@pytest.mark.parametrize("hd,nh,nk", [(128, 14, 2), (64, 14, 2)])
def test_prefill_rows_that_see_no_key(gpu, hd, nh, nk):
    """Causal, no append, fewer cached keys than queries: the first rows see none and are zero."""
    ctx, s_q = [5, 30, 100], 40
    cpu, d = make_paged_case(gpu, batch=3, ctx=ctx, page_size=256, n_kv=nk, n_heads=nh, head_dim=hd, s_q=s_q, seed=3)
    out = prism_amd.prefill_attention(d["q"], d["k_cache"], d["v_cache"], cache_seqlens=d["cache_seqlens"],
                                      block_table=d["block_table"], causal=True)
    ref, _, _ = pa.flash_attn_with_kvcache_ref(cpu["q"], cpu["k_cache"], cpu["v_cache"],
                                               cache_seqlens=cpu["cache_seqlens"], block_table=cpu["block_table"],
                                               causal=True)
    torch.cuda.synchronize()
    assert (out[0, :s_q - 5] == 0).all() and (out[1, :s_q - 30] == 0).all()
    assert_attn_close(out[2:], ref[2:], "rows with keys")
    assert np.isfinite(out.float().cpu().numpy()).all()


def test_prefill_flags_a_bad_page(gpu):
    cpu, d = make_paged_case(gpu, batch=2, ctx=[300, 10], page_size=64, n_kv=2, n_heads=14, head_dim=64, s_q=20, seed=9)
    d["block_table"][0, 2] = 100000
    prism_amd.prefill_attention(d["q"], d["k_cache"], d["v_cache"], d["k"], d["v"], cache_seqlens=d["cache_seqlens"],
                                block_table=d["block_table"], causal=True)
    assert prism_amd.read_status(gpu) & 1


# head_dim, n_heads, n_kv, page, s_q, prefixes: few enough row blocks that the keys split, over ranges
# of one, a few and the most stages, uneven lengths (some sequences one range, some none)
SPLIT_CASES = [
    (128, 28, 4, 256, 33, [3000]),
    (128, 8, 8, 64, 129, [0, 700, 5]),
    (64, 14, 2, 256, 70, [5000, 0]),
    (64, 2, 2, 64, 257, [1, 1500, 255]),
    (128, 7, 1, 256, 20, [16000]),
]


@pytest.mark.parametrize("append", [True, False])
@pytest.mark.parametrize("case", SPLIT_CASES, ids=[f"hd{c[0]}-kv{c[2]}-s{c[4]}" for c in SPLIT_CASES])
def test_prefill_split_keys_matches_unsplit_and_oracle(gpu, case, append):
    hd, nh, nk, page, s_q, ctx = case
    cpu, d = make_paged_case(gpu, batch=len(ctx), ctx=ctx, page_size=page, n_kv=nk, n_heads=nh, head_dim=hd, s_q=s_q,
                             seed=hd + nk + s_q)
    kw = dict(cache_seqlens=d["cache_seqlens"], block_table=d["block_table"], causal=True)
    k, v = (d["k"], d["v"]) if append else (None, None)
    assert prism_amd._lib.load().pkv_prefill_workspace_bytes(len(ctx), s_q, nh, nk, hd, page,
                                                             d["block_table"].shape[1]) > 0
    out = torch.full((len(ctx), s_q, nh, hd), float("nan"), dtype=torch.bfloat16, device=gpu)
    one = torch.full_like(out, float("nan"))
    prism_amd.prefill_attention(d["q"], d["k_cache"], d["v_cache"], k, v, out=out, **kw)
    prism_amd.flash_attn_with_kvcache(d["q"], d["k_cache"], d["v_cache"], k, v, out=one, noalloc=True, **kw)
    ref, _, _ = pa.flash_attn_with_kvcache_ref(cpu["q"], cpu["k_cache"], cpu["v_cache"], cpu["k"] if append else None,
                                               cpu["v"] if append else None, cache_seqlens=cpu["cache_seqlens"],
                                               block_table=cpu["block_table"], causal=True)
    torch.cuda.synchronize()
    a, b = out.float().cpu().numpy(), one.float().cpu().numpy()
    assert np.isfinite(a).all() and np.isfinite(b).all()
    # the same products in another order of fp32 sums (and another running max per range, so P rounds
    # differently): two bf16 units of the row, or of 1e-2
    assert (np.abs(a - b) <= np.maximum(1e-2, np.abs(b) * 2.0 ** -6)).all()
    few = np.array([[c + j + (1 if append else 1 - s_q) <= 8 for j in range(s_q)] for c in ctx])
    err = np.abs(a - ref)
    assert err[~few].max(initial=0.0) <= 1e-2 and err.mean() <= 1e-3
    assert prism_amd.read_status(gpu) == 0


def test_prefill_captured_runs_unsplit(gpu):
    """A captured call takes no workspace, also where eager calls have sized one (its replays may run
    beside them on other streams): its replays give the unsplit result."""
    cpu, d = make_paged_case(gpu, batch=1, ctx=[900], page_size=256, n_kv=4, n_heads=28, head_dim=128, s_q=40, seed=1)
    kw = dict(cache_seqlens=d["cache_seqlens"], block_table=d["block_table"], causal=True)
    args = d["q"], d["k_cache"], d["v_cache"], d["k"], d["v"]
    want = prism_amd.flash_attn_with_kvcache(*args, noalloc=True, **kw)
    split = prism_amd.flash_attn_with_kvcache(*args, **kw)
    assert not torch.equal(split, want)  # other fp32 sum orders: the eager call does split
    out, out2 = torch.empty_like(want), torch.empty_like(want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        prism_amd.flash_attn_with_kvcache(*args, out=out, **kw)
        prism_amd.prefill_attention(*args, out=out2, **kw)
    for _ in range(3):
        out.zero_()
        out2.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(out2, want)
        assert torch.equal(prism_amd.flash_attn_with_kvcache(*args, **kw), split)


@pytest.mark.parametrize("hd,page,ctx", [(128, 32, [4200, 4500]), (64, 64, [8300, 9000])])
def test_prefill_block_table_window_refills(gpu, hd, page, ctx):
    """Over 130 pages in one workgroup's walk (unsplit): its 64-column window of the table is loaded twice more
    inside the loop."""
    cpu, d = make_paged_case(gpu, batch=2, ctx=ctx, page_size=page, n_kv=1, n_heads=7, head_dim=hd, s_q=20, seed=hd)
    out = prism_amd.flash_attn_with_kvcache(d["q"], d["k_cache"], d["v_cache"], d["k"], d["v"], noalloc=True,
                                            cache_seqlens=d["cache_seqlens"], block_table=d["block_table"],
                                            causal=True)
    ref, _, _ = pa.flash_attn_with_kvcache_ref(cpu["q"], cpu["k_cache"], cpu["v_cache"], cpu["k"], cpu["v"],
                                               cache_seqlens=cpu["cache_seqlens"], block_table=cpu["block_table"],
                                               causal=True)
    assert_attn_close(out, ref, f"hd {hd}")
    assert prism_amd.read_status(gpu) == 0
