"""GPU parity of wide causal windows (prompts and prompt chunks: the kernel
of csrc/attention_window.hip) through sde_paged_attention, against the fp64
oracle.

A workgroup of that kernel holds 128 rows -- (query, head in group) pairs of
a KV head -- 32 per wave and two waves per 64-token tile, and cuts the context
into partitions where the row groups alone leave CUs idle; it takes windows of
96 rows or more whose rows x keys are many.  The shapes sit at its edges: the
fewest rows it takes and one row group more or less, rows that do not fill a
wave or a group, query groups that straddle waves (G = 7), windows that begin
and end inside a tile, no context and long context (partitions), the largest
number of row groups a call may have, block sizes that are and are not powers
of two.

Tolerance: the products carry ~22 bits of q and of the softmax weights and
sums are fp32, so a row's error is some 1e-6 of the output's scale; the
bound is 1e-5 of it (and the contract's 2e-3 + 1e-2 |ref|, far above)."""
import numpy as np
import pytest
import torch

from conftest import case_banner
from speculative_decode_engine_amd import workloads as W
from test_gpu_attention import assert_close, build_layer

pytestmark = pytest.mark.gpu

CASES = [
    # nh, nkv, dph, bs, ctx, M
    (8, 2, 128, 16, 60100, 24),   # 96 rows: the smallest window of the kernel
    (8, 1, 128, 16, 90116, 16),   # 128 rows: one full row group, long context
    (8, 1, 128, 16, 90095, 16),   # the same just short of its rows x keys: the 16-row kernel
    (8, 2, 128, 16, 46000, 33),   # 132 rows: a second group of four rows
    (8, 8, 64, 16, 11100, 129),   # G = 1: one row past a group
    (28, 4, 128, 32, 11200, 37),  # G = 7: 259 rows, queries straddle waves
    (32, 4, 64, 16, 1500, 256),   # a prompt chunk
    (16, 4, 128, 8, 11099, 65),   # window starts inside a tile, block size 8
    (4, 4, 64, 24, 7000, 400),    # block size not a power of two
    (32, 8, 128, 16, 0, 1001),    # no context: causal all the way
    (32, 8, 128, 16, 0, 2048),    # the most row groups a call may have
    (32, 8, 64, 8, 17000, 2048),  # more blocks than the kernel's table in LDS holds
]


def check(got, ref, what):
    assert_close(got, ref, what)
    scale = np.abs(ref).max()
    err = np.abs(got.astype(np.float64) - ref).max()
    assert err <= 1e-5 * scale, f"{what}: max abs err {err:.3e}, output scale {scale:.3e}"


@pytest.mark.parametrize("nh,nkv,dph,bs,ctx,M", CASES)
def test_wide_window_matches_float64(gpu, oracle, nh, nkv, dph, bs, ctx, M):
    case_banner("wide window", nh, nkv, dph, bs, ctx, M)
    nblk = -(-(ctx + M) // bs)
    cache, K, V, rng = build_layer(nh, nkv, dph, bs, ctx, M, nblk + 7, dph + ctx + M)
    q = W.queries(rng, M, nh, dph)
    qt = torch.from_numpy(q).cuda()
    out = cache.attention(0, qt, nh, nkv, dph, ctx, out=torch.full((M, nh * dph), float("nan"),
                                                                   device="cuda"))
    again = cache.attention_noalloc(0, qt, nh, nkv, dph, ctx, out=torch.full_like(out, -1.0))
    ws = torch.empty(cache.workspace_size(nh, nkv, dph, M, ctx + M) // 4 + 1, device="cuda")
    third = cache.attention(0, qt, nh, nkv, dph, ctx, workspace=ws)
    torch.cuda.synchronize()
    assert torch.equal(out, again) and torch.equal(out, third)
    rows = sorted({0, 1, M // 2, M - 2, M - 1} | set(range(0, M, max(1, M // 24))))
    ref = np.concatenate([oracle.attention_f64_np(q[m:m + 1], K[:ctx + m + 1], V[:ctx + m + 1],
                                                  nh, nkv, dph, ctx + m) for m in rows])
    check(out.cpu().numpy()[rows], ref, f"{nh}/{nkv} dph {dph} ctx {ctx} M {M}")
    cache.free()


@pytest.mark.parametrize("nh,nkv,dph,ctx,M,gap", [
    (32, 8, 128, 0, 2003, 14.0),
    (32, 8, 128, 0, 2003, 8.0),
    (32, 4, 64, 1500, 256, 14.0),   # partitions
])
def test_keys_beside_a_dominant_one(gpu, oracle, nh, nkv, dph, ctx, M, gap):
    """One key `gap` nats above the others whose V is small, as an attention
    sink's: the other keys' weights of some e^-gap make a visible part of the
    output.

    A weight of 2^-20 of the largest is carried to 2^-12 of itself at the
    least (a quantum of 2^-32) and the rest of the arithmetic is fp32; half the
    output (gap 8) or some percent of it (gap 14) comes from the other keys,
    whose errors are independent: 2e-6 in all."""
    case_banner("wide window, dominant key", nh, nkv, dph, ctx, M, gap)
    cache, K, V, rng = build_layer(nh, nkv, dph, 16, ctx, M, -(-(ctx + M) // 16) + 7, dph + M)
    u = np.sign(rng.standard_normal(dph)).astype(np.float32)
    K[0] = np.tile(u * np.float32(gap / np.sqrt(dph)), nkv).astype(np.float16)
    V[0] = (V[0] * 0.02).astype(np.float16)
    cache.append(0, torch.from_numpy(K[:1].copy()).cuda(), torch.from_numpy(V[:1].copy()).cuda(), 0)
    q = W.queries(rng, M, nh, dph) + np.tile(u, nh)
    out = cache.attention(0, torch.from_numpy(q).cuda(), nh, nkv, dph, ctx).cpu().numpy()
    for m in sorted({M // 2, M - 1} | set(range(M // 3, M, max(1, M // 8)))):
        ref = oracle.attention_f64_np(q[m:m + 1], K[:ctx + m + 1], V[:ctx + m + 1], nh, nkv, dph,
                                      ctx + m)
        err = np.linalg.norm(out[m] - ref[0]) / np.linalg.norm(ref[0])
        assert err <= 2e-6, (m, err)
    cache.free()


@pytest.mark.parametrize("dph", [64, 128])
def test_wide_window_hidden_nonfinite_rows(gpu, oracle, dph):
    """Inf / NaN in V (and NaN in K) at window positions and in stale slots
    past the window reach only the queries that see them."""
    case_banner("wide window, hidden non-finite", dph)
    nh, nkv, bs, ctx, M = 8, 2, 16, 19430, 75
    cache, K, V, rng = build_layer(nh, nkv, dph, bs, ctx, M, 1230, dph)
    bad = ctx + 20  # window row 20; seen from query 20 on
    k, v = K[bad].copy(), V[bad].copy()
    v[::3], v[1::3], k[5] = np.inf, np.nan, np.nan
    cache.append(0, torch.from_numpy(k[None]).cuda(), torch.from_numpy(v[None]).cuda(), bad)
    table = cache.block_table(0)
    last = ctx + M
    view = cache.pool_blocks_view()
    view[int(table[last // bs]), :, last % bs:] = 0x7E00  # NaN
    q = W.queries(rng, M, nh, dph)
    out = cache.attention(0, torch.from_numpy(q).cuda(), nh, nkv, dph, ctx).cpu().numpy()
    n = bad - ctx
    ref = oracle.attention_f64_np(q[:n], K[:bad], V[:bad], nh, nkv, dph, ctx)
    check(out[:n], ref, "queries that do not see it")
    # a NaN logit poisons the row's sum: the whole row is not finite or, by
    # the l > 1e-20 && finite rule, scaled by zero
    assert not np.isfinite(out[n:]).all(axis=1).any()
    cache.free()


def test_wide_window_combine_keeps_inf(gpu):
    """Inf in V that every row sees, in the last partition of the rows before
    position 4032 (576 tokens each): a part of a pair makes NaN of it where the
    lo part is negative, as in every fp16 pair product here, but the combine of
    seven partitions must not."""
    case_banner("wide window, Inf in the last partition")
    nh, nkv, dph, bs, ctx, M = 32, 8, 128, 16, 4000, 128
    cache, K, V, rng = build_layer(nh, nkv, dph, bs, ctx, M, 270, 3)
    v = V[3900:3901].copy()
    v[0, 7] = np.inf
    cache.append(0, torch.from_numpy(K[3900:3901].copy()).cuda(), torch.from_numpy(v).cuda(), 3900)
    q = torch.from_numpy(W.queries(rng, M, nh, dph)).cuda()
    out = cache.attention(0, q, nh, nkv, dph, ctx).view(M, nh, dph)
    assert not torch.isfinite(out[:, :4, 7]).any()
    assert torch.isfinite(out[:, :, 8:]).all() and torch.isfinite(out[:, 4:]).all()
    assert (out[:32, :4, 7] == float("inf")).any() and (out[32:, :4, 7] == float("inf")).any()
    cache.free()


def test_wide_window_replays_in_a_graph(gpu):
    """Captured with a workspace, and captured with none on a cache that owns
    none yet (one partition then): replays match the eager call."""
    case_banner("wide window graph")
    nh, nkv, dph, bs, ctx, M = 32, 4, 64, 16, 1500, 256
    cache, K, V, rng = build_layer(nh, nkv, dph, bs, ctx, M, 120, 5)
    q = torch.from_numpy(W.queries(rng, M, nh, dph)).cuda()
    outs = [torch.zeros(M, nh * dph, device="cuda") for _ in range(2)]
    ws = torch.empty(cache.workspace_size(nh, nkv, dph, M, ctx + M) // 4 + 1, device="cuda")
    g = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(g, stream=s):
        cache.attention(0, q, nh, nkv, dph, ctx, out=outs[0])
        cache.attention(0, q, nh, nkv, dph, ctx, out=outs[1], workspace=ws)
    for i in range(3):
        eager = cache.attention(0, q, nh, nkv, dph, ctx)
        for o in outs:
            o.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(outs[1], eager)
        assert torch.allclose(outs[0], eager, rtol=0, atol=1e-5)
        q.mul_(-0.5)
    cache.free()
