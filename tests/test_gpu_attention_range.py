"""The generic attention path's matrix-core form (gen_tile_kernel) over the
range of inputs that its fp32 form takes, against float64."""
import numpy as np
import pytest
import torch

from conftest import case_banner
from speculative_decode_engine_amd import KVCache
from speculative_decode_engine_amd import workloads as W

pytestmark = pytest.mark.gpu


def build(rng, K, V, nkv, dph, bs):
    """A cache of one layer that holds the fp32 rows K, V behind a fragmented
    table; returns it and the rows as fp16 stored them."""
    n = -(-K.shape[0] // bs) + 1
    cache = KVCache(1, nkv * dph, n, bs, n + 7)
    cache.set_block_table(0, W.make_tables(rng, 1, n, n + 7)[0])
    with np.errstate(over="ignore"):
        K16, V16 = K.astype(np.float16), V.astype(np.float16)
    cache.write_fp16(0, torch.from_numpy(K16.view(np.int16)).cuda(),
                     torch.from_numpy(V16.view(np.int16)).cuda(), 0)
    return cache, K16.astype(np.float32), V16.astype(np.float32)


def rows(rng, n, width, scale=1.0):
    return (rng.standard_normal((n, width)) * scale).astype(np.float32)


@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("qexp,kexp", [(20, -20), (-12, 10)])
@pytest.mark.parametrize("nh,nkv,dph,bs", [(4, 2, 8, 16), (4, 2, 64, 12), (3, 1, 96, 16),
                                           (8, 2, 256, 16)])
def test_queries_of_any_magnitude(gpu, oracle, nh, nkv, dph, bs, qexp, kexp, rope):
    """Rows of a group that differ by a power of two of 40, at head sizes with
    two and with three fp16 parts of q, the smallest and the largest.  A scaled
    row carries q to 2^-22 of its largest element, a logit's sum is fp32 and
    the logits here are N(0, 1) or smaller, so weights are within some 2^-20
    and outputs within 1e-5 of their scale."""
    case_banner("query range", nh, nkv, dph, bs, qexp, kexp, rope)
    rng = np.random.default_rng(dph + qexp + 2 * rope + 12)
    ctx, M = 300, 5
    K, V = rows(rng, ctx + M, nkv * dph, 2.0 ** kexp), rows(rng, ctx + M, nkv * dph)
    q = rows(rng, M, nh * dph, 2.0 ** qexp)
    q[1] *= 2.0 ** -20
    q[3] *= 2.0 ** -40
    q[:, :dph // 2] *= 2.0 ** -6  # (a head whose elements differ)
    cache, K, V = build(rng, K, V, nkv, dph, bs)
    qt = torch.from_numpy(q).cuda()
    if rope:
        k, v = rows(rng, M, nkv * dph, 2.0 ** kexp), rows(rng, M, nkv * dph)
        out = cache.rope_append_attention(0, qt, torch.from_numpy(k).cuda(),
                                          torch.from_numpy(v).cuda(), nh, nkv, dph, ctx)
        K, V = (t.cpu().numpy() for t in cache.read(0, 0, ctx + M))
        q = oracle.rope_rotate_half_f64(q, nh, dph, np.arange(ctx, ctx + M))
    else:
        out = cache.attention(0, qt, nh, nkv, dph, ctx)
    ref = oracle.attention_f64_np(q, K, V, nh, nkv, dph, ctx)
    err = np.abs(out.cpu().numpy() - ref).max(axis=1) / np.abs(ref).max(axis=1)
    assert (err <= 1e-5).all(), err
    cache.free()


@pytest.mark.parametrize("gap", [8.0, 14.0])
@pytest.mark.parametrize("nh,nkv,dph,bs,ctx,M", [
    (32, 32, 40, 16, 1200, 256),  # one partition: a wave's 300 keys beside the sink
    (16, 8, 256, 16, 4000, 5),
    (4, 2, 96, 16, 120, 1),       # a wave's 32 keys
])
def test_keys_beside_a_dominant_one(gpu, oracle, nh, nkv, dph, bs, ctx, M, gap):
    """One key `gap` nats above the others whose V is small, as an attention
    sink's: the other keys' weights of some e^-gap make a visible part of the
    output.

    A weight of 2^-20 of the largest is carried to 2^-22 and the rest of the
    arithmetic is fp32: a logit near 25 (log2) is within some 2^-20, which its
    key's weight takes on, and half the output (gap 8) or some percent of it
    (gap 14) comes from the other keys' independent errors: 2e-6 in all."""
    case_banner("dominant key", nh, nkv, dph, ctx, M, gap)
    rng = np.random.default_rng(dph + int(gap))
    u = np.sign(rng.standard_normal(dph)).astype(np.float32)
    K, V = rows(rng, ctx + M, nkv * dph), rows(rng, ctx + M, nkv * dph)
    K[0] = np.tile(u * np.float32(gap / np.sqrt(dph)), nkv)
    V[0] *= 0.02
    q = rows(rng, M, nh * dph) + np.tile(u, nh)
    cache, K, V = build(rng, K, V, nkv, dph, bs)
    out = cache.attention(0, torch.from_numpy(q).cuda(), nh, nkv, dph, ctx).cpu().numpy()
    for m in range(0, M, max(1, M // 6)):
        ref = oracle.attention_f64_np(q[m:m + 1], K[:ctx + m + 1], V[:ctx + m + 1], nh, nkv, dph,
                                      ctx + m)
        err = np.linalg.norm(out[m] - ref[0]) / np.linalg.norm(ref[0])
        assert err <= 2e-6, (m, err)
    cache.free()


def special(x):
    """0 where finite, 1 / -1 where +-Inf, 2 where NaN."""
    return np.where(np.isnan(x), 2, np.where(np.isinf(x), np.sign(x), 0))


@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("what", ["V", "K", "q"])
@pytest.mark.parametrize("nh,nkv,dph,bs,ctx,M", [
    (4, 2, 32, 16, 300, 3),      # three partitions
    (4, 2, 96, 16, 100, 1),      # one partition
    (10, 2, 256, 12, 700, 5),    # 25 rows: two groups of rows
    (4, 4, 40, 16, 900, 21),
])
def test_nonfinite_values_that_rows_see(gpu, oracle, nh, nkv, dph, bs, ctx, M, what, rope):
    """Inf in V reaches its features with its sign, a logit of -Inf weighs
    nothing and one of +Inf or NaN makes its row NaN, as fp32 arithmetic has
    it; every other output keeps its precision."""
    case_banner("visible non-finite", nh, nkv, dph, bs, ctx, M, what, rope)
    rng = np.random.default_rng(dph + ctx)
    K, V = rows(rng, ctx + M, nkv * dph), rows(rng, ctx + M, nkv * dph)
    q = rows(rng, M, nh * dph)
    if what == "V":
        V[7, ::3], V[90, 1::3] = np.inf, -np.inf
        V[40, dph - 1] = np.nan
        V[ctx - 1, 5] = np.inf  # (in the last partition)
    elif what == "K":
        K[70, 3] = np.inf
        q.reshape(M, nh, dph)[:, ::2, 3] = -1.0
    else:
        q[0, 5], q[M - 1, dph + 2] = np.inf, np.nan
    cache, K, V = build(rng, K, V, nkv, dph, bs)
    qt = torch.from_numpy(q).cuda()
    if rope:
        k, v = rows(rng, M, nkv * dph), rows(rng, M, nkv * dph)
        out = cache.rope_append_attention(0, qt, torch.from_numpy(k).cuda(),
                                          torch.from_numpy(v).cuda(), nh, nkv, dph, ctx)
        K, V = (t.cpu().numpy() for t in cache.read(0, 0, ctx + M))
        with np.errstate(invalid="ignore"):
            q = oracle.rope_rotate_half_f64(q, nh, dph, np.arange(ctx, ctx + M))
    else:
        out = cache.attention(0, qt, nh, nkv, dph, ctx)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = oracle.attention_f64_np(q, K, V, nh, nkv, dph, ctx)
    got = out.cpu().numpy()
    # (RoPE gives the feature that meets K's Inf either sign)
    assert (special(ref) == 0).any() and (what == "K" or (special(ref) != 0).any())
    assert np.array_equal(special(got), special(ref)), np.argwhere(special(got) != special(ref))[:8]
    live = special(ref) == 0
    assert np.abs(got[live] - ref[live]).max() <= 1e-5 * np.abs(ref[live]).max()
    cache.free()
