"""Speculative verify on prefill_tile_kernel's two-wave form: 17 to 64 query rows per KV head, with the
new rows appended by the ranges that cover them (a chunk that straddles two stages or two ranges, empty
caches, new rows on a page boundary), ragged batches whose ranges differ in number, the largest batch of
the rule and the one past it, and the head counts and dims that the balanced kernel keeps.  Caches
bit-exact, outputs against the fp64 oracle, and against the balanced kernel the merge flag selects."""
import numpy as np
import pytest
import torch

import prism_amd
from oracle import paged_attention as pa
from pkv_testutil import assert_attn_close, make_paged_case

pytestmark = pytest.mark.gpu

# head_dim, n_heads, n_kv, page, s_q, contexts
CASES = [
    (128, 28, 4, 256, 5, [0, 27, 30, 253, 254, 4000]),
    (128, 28, 4, 32, 3, [29, 30, 31, 500, 0]),
    (128, 40, 8, 64, 4, [62, 1000, 7]),
    (128, 32, 4, 256, 8, [1]),
    (128, 28, 4, 256, 5, [9000, 3, 700]),
    (128, 7, 1, 256, 5, [9000, 3, 700]),  # the balanced kernel, and the next two
    (64, 14, 2, 64, 5, [60, 61, 0, 3000, 700]),
    (64, 16, 4, 256, 16, [255, 100, 2000]),
    (128, 28, 4, 256, 5, [(i * 37) % 400 for i in range(64)]),
    (128, 28, 4, 256, 5, [(i * 37) % 300 for i in range(65)]),  # past the rule: the balanced kernel
]


@pytest.mark.parametrize("append", [True, False])
@pytest.mark.parametrize("case", CASES, ids=[f"hd{c[0]}-kv{c[2]}-p{c[3]}-s{c[4]}-b{len(c[5])}" for c in CASES])
def test_verify_matches_oracle_and_balanced_kernel(gpu, case, append):
    hd, nh, nk, page, s_q, ctx = case
    cpu, d = make_paged_case(gpu, batch=len(ctx), ctx=ctx, page_size=page, n_kv=nk, n_heads=nh, head_dim=hd, s_q=s_q,
                             seed=hd + nk + page + s_q)
    for b, c in enumerate(ctx):   # stale slots behind the sequence hold NaN
        end = c + s_q
        for name in ("k_cache", "v_cache"):
            for t in (cpu, d):
                t[name][int(cpu["block_table"][b, (end - 1) // page]), (end - 1) % page + 1:] = float("nan")
    kw = dict(cache_seqlens=d["cache_seqlens"], block_table=d["block_table"], causal=True, shared_prefix_tokens=0)
    k, v = (d["k"], d["v"]) if append else (None, None)
    if not append:
        d["cache_seqlens"] += s_q
    other = prism_amd.flash_attn_with_kvcache(d["q"], d["k_cache"].clone(), d["v_cache"].clone(), k, v, two_pass=True,
                                              **kw)
    out = torch.full((len(ctx), s_q, nh, hd), float("nan"), dtype=torch.bfloat16, device=gpu)
    prism_amd.flash_attn_with_kvcache(d["q"], d["k_cache"], d["v_cache"], k, v, out=out, **kw)
    torch.cuda.synchronize()
    ref, kb, vb = pa.flash_attn_with_kvcache_ref(
        cpu["q"], cpu["k_cache"], cpu["v_cache"], cpu["k"] if append else None, cpu["v"] if append else None,
        cache_seqlens=d["cache_seqlens"].cpu(), block_table=cpu["block_table"], causal=True)
    assert np.array_equal(pa.bf16_bits(d["k_cache"]), kb) and np.array_equal(pa.bf16_bits(d["v_cache"]), vb)
    got = out.float().cpu().numpy()
    assert np.isfinite(got).all()
    err, near = np.abs(got - ref), np.abs(got - other.float().cpu().numpy())
    few = np.array([[c + j + 1 <= 8 for j in range(s_q)] for c in ctx])
    # a bf16 output is within half a unit of its value, P's own rounding within another: rows of a few
    # keys reach one unit of the value where that passes 1e-2
    assert err[~few].max(initial=0.0) <= 1e-2 and err.mean() <= 1e-3
    assert (err[few] <= np.maximum(1e-2, np.abs(ref[few]) * 2.0 ** -7)).all()
    assert (near <= np.maximum(1.6e-2, np.abs(ref) * 2.0 ** -6)).all()
    assert prism_amd.read_status(gpu) == 0


@pytest.mark.parametrize("hd,nh,nk", [(64, 14, 2), (64, 16, 4), (128, 7, 1), (128, 14, 2)])
def test_verify_keeps_the_more_exact_kernel(gpu, hd, nh, nk):
    """head_dim 64 and one or two KV heads: the call is the balanced kernel's launch, bit-identical to the
    one a merge flag selects."""
    cpu, d = make_paged_case(gpu, batch=6, ctx=[0, 27, 30, 253, 254, 600], page_size=256, n_kv=nk, n_heads=nh,
                             head_dim=hd, s_q=5, seed=5)
    kw = dict(cache_seqlens=d["cache_seqlens"], block_table=d["block_table"], causal=True, shared_prefix_tokens=0)
    a = prism_amd.flash_attn_with_kvcache(d["q"], d["k_cache"], d["v_cache"], d["k"], d["v"], **kw)
    b = prism_amd.flash_attn_with_kvcache(d["q"], d["k_cache"], d["v_cache"], d["k"], d["v"], two_pass=True, **kw)
    assert torch.equal(a, b)


def test_verify_noalloc_is_bit_identical(gpu):
    cpu, d = make_paged_case(gpu, batch=6, ctx=[0, 27, 30, 253, 254, 4000], page_size=256, n_kv=4, n_heads=28,
                             head_dim=128, s_q=5, seed=5)
    kw = dict(cache_seqlens=d["cache_seqlens"], block_table=d["block_table"], causal=True, shared_prefix_tokens=0)
    a = prism_amd.flash_attn_with_kvcache(d["q"], d["k_cache"], d["v_cache"], d["k"], d["v"], **kw)
    b = prism_amd.flash_attn_with_kvcache(d["q"], d["k_cache"], d["v_cache"], d["k"], d["v"], noalloc=True, **kw)
    assert torch.equal(a, b)


@pytest.mark.parametrize("nh,nk,s_q,ctx", [(28, 4, 5, [600, 90, 1400, 33]), (40, 8, 6, [500, 150]),
                                           (28, 4, 6, [16, 300, 45, 8, 120, 700])])
def test_verify_error_is_the_output_rounding(gpu, nh, nk, s_q, ctx):
    """Rounding N(0, s) values to bf16 leaves a relative error of 1.66e-3 (2-norm); P rounded to bf16 once
    brings it to 1.9e-3 and more, held as a pair it adds nothing that shows."""
    cpu, d = make_paged_case(gpu, batch=len(ctx), ctx=ctx, page_size=256, n_kv=nk, n_heads=nh, head_dim=128, s_q=s_q,
                             seed=nh + s_q)
    out = prism_amd.flash_attn_with_kvcache(d["q"], d["k_cache"], d["v_cache"], d["k"], d["v"], causal=True,
                                            cache_seqlens=d["cache_seqlens"], block_table=d["block_table"])
    ref, _, _ = pa.flash_attn_with_kvcache_ref(cpu["q"], cpu["k_cache"], cpu["v_cache"], cpu["k"], cpu["v"],
                                               cache_seqlens=cpu["cache_seqlens"], block_table=cpu["block_table"],
                                               causal=True)
    got = out.double().cpu().numpy()
    assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < 1.8e-3


def test_verify_infinite_value_stays_infinite(gpu):
    """One infinite V element that every row sees: that output element is the infinity, the others finite
    (neither half of P may meet it as a zero, or with the other sign)."""
    cpu, d = make_paged_case(gpu, batch=2, ctx=[300, 40], page_size=256, n_kv=4, n_heads=28, head_dim=128, s_q=5,
                             seed=2)
    for b, value in ((0, float("inf")), (1, -float("inf"))):
        d["v_cache"][int(cpu["block_table"][b, 0]), 7, 1, 3] = value
    out = prism_amd.flash_attn_with_kvcache(d["q"], d["k_cache"], d["v_cache"], d["k"], d["v"], causal=True,
                                            cache_seqlens=d["cache_seqlens"], block_table=d["block_table"])
    assert (out[0, :, 7:14, 3] == float("inf")).all() and (out[1, :, 7:14, 3] == -float("inf")).all()
    out[:, :, 7:14, 3] = 0
    assert out.isfinite().all()


@pytest.mark.parametrize("base,stride", [(8, 0), (0, 8), (8, 8)], ids=["base", "page-stride", "both"])
def test_verify_appends_off_a_cache_line_keep_the_balanced_kernel(gpu, base, stride):
    """Caches 16 bytes off a 128-byte line, or pages that are: a row appended in the launch could share a line
    with one that another workgroup has read, so an appending call stays on the balanced kernel.  Without an
    append it does not matter."""
    P, nk = 64, 4
    cpu, d = make_paged_case(gpu, batch=4, ctx=[0, 63, 130, 700], page_size=P, n_kv=nk, n_heads=28, head_dim=128,
                             s_q=5, seed=4)

    def view(t):
        ps = t[0].numel() + stride
        buf = torch.zeros(base + t.shape[0] * ps, dtype=t.dtype, device=gpu)
        v = buf.as_strided(t.shape, (ps, nk * 128, 128, 1), base)
        return v.copy_(t)

    kc, vc = view(d["k_cache"]), view(d["v_cache"])
    kw = dict(cache_seqlens=d["cache_seqlens"], block_table=d["block_table"], causal=True, shared_prefix_tokens=0)
    other = prism_amd.flash_attn_with_kvcache(d["q"], d["k_cache"].clone(), d["v_cache"].clone(), d["k"], d["v"],
                                              two_pass=True, **kw)
    out = prism_amd.flash_attn_with_kvcache(d["q"], kc, vc, d["k"], d["v"], **kw)
    ref, kb, vb = pa.flash_attn_with_kvcache_ref(cpu["q"], cpu["k_cache"], cpu["v_cache"], cpu["k"], cpu["v"],
                                                 cache_seqlens=cpu["cache_seqlens"], block_table=cpu["block_table"],
                                                 causal=True)
    assert np.array_equal(pa.bf16_bits(kc), kb) and np.array_equal(pa.bf16_bits(vc), vb)
    assert torch.equal(out, other)
    assert_attn_close(out, ref, "off a cache line")
    kw["cache_seqlens"] = d["cache_seqlens"] + 5
    again = prism_amd.flash_attn_with_kvcache(d["q"], kc, vc, **kw)
    assert_attn_close(again, ref, "off a cache line, no append")
    assert prism_amd.read_status(gpu) == 0


@pytest.mark.parametrize("nh,ctx,tiles", [(28, [10200, 5], True), (28, [10300, 5], False), (28, [100] * 16, False),
                                          (28, [100] * 17, True)])
def test_verify_rule_by_table_width(gpu, nh, ctx, tiles):
    """Both sides of the rule's lines: on the tile kernel the P of a call is a pair, on the balanced kernel
    the call is bit-identical to the one a merge flag selects.  Either is within the tolerance."""
    cpu, d = make_paged_case(gpu, batch=len(ctx), ctx=ctx, page_size=256, n_kv=4, n_heads=nh, head_dim=128, s_q=5,
                             seed=len(ctx))
    kw = dict(cache_seqlens=d["cache_seqlens"], block_table=d["block_table"], causal=True, shared_prefix_tokens=0)
    a = prism_amd.flash_attn_with_kvcache(d["q"], d["k_cache"], d["v_cache"], d["k"], d["v"], **kw)
    b = prism_amd.flash_attn_with_kvcache(d["q"], d["k_cache"], d["v_cache"], d["k"], d["v"], two_pass=True, **kw)
    ref, _, _ = pa.flash_attn_with_kvcache_ref(cpu["q"], cpu["k_cache"], cpu["v_cache"], cpu["k"], cpu["v"],
                                               cache_seqlens=cpu["cache_seqlens"], block_table=cpu["block_table"],
                                               causal=True)
    assert_attn_close(b, ref, "balanced")
    assert_attn_close(a, ref, "the rule's choice")
    assert torch.equal(a, b) is not tiles
