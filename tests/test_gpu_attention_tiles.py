"""GPU parity of the matrix-core form of the generic attention path (head
sizes that are multiples of 8 up to 256, any block size: gen_tile_kernel)
against the fp64 oracle.

A workgroup there takes 16 rows -- (query, head in group) pairs of a KV head
-- and its four waves 32-token tiles in turn; a tile is loaded as a flat run
of 16-byte units, so the head size in units (odd, even, a multiple of 4, 8,
16) decides the lanes' tokens, the LDS swizzle and the tail load, and the
head size within its padding to 32 what must be dropped.  The shapes go over
those, over row groups that are not full, one row past a group, contexts that
end inside a tile or fill partitions exactly, none at all, and block sizes
that no tile aligns with.

Tolerance: products carry ~22 bits of q and the weights, sums are fp32: some
1e-6 of the output's scale; the bound is 1e-5 of it."""
import numpy as np
import pytest
import torch

from conftest import case_banner
from speculative_decode_engine_amd import workloads as W
from test_gpu_attention import assert_close, build_layer

pytestmark = pytest.mark.gpu


def check(got, ref, what):
    assert_close(got, ref, what)
    scale = np.abs(ref).max()
    err = np.abs(got.astype(np.float64) - ref).max()
    assert err <= 1e-5 * scale, f"{what}: max abs err {err:.3e}, output scale {scale:.3e}"


SIZES = [(4, 2, dph, bs, ctx, 3)
         for dph, bs, ctx in [(8, 16, 130), (16, 8, 255), (24, 5, 300), (32, 16, 1000),
                              (40, 16, 511), (48, 1, 77), (56, 32, 640), (72, 16, 1023),
                              (80, 7, 900), (88, 16, 129), (96, 24, 2045), (104, 16, 64),
                              (112, 16, 1500), (120, 48, 95), (136, 16, 700), (160, 9, 515),
                              (168, 16, 31), (184, 16, 1280), (192, 64, 257), (200, 16, 900),
                              (232, 3, 700), (248, 16, 385), (256, 16, 3000), (64, 12, 1000),
                              (128, 20, 1000)]]
ROWS = [
    (16, 1, 96, 16, 500, 1),     # 16 rows: one full group
    (17, 1, 96, 16, 500, 1),     # one row past it
    (5, 5, 80, 16, 5000, 1),     # one row per KV head, many partitions
    (6, 2, 256, 16, 0, 50),      # 150 rows, no context: groups that see little of the window
    (32, 32, 96, 16, 4095, 1),   # a context that fills its last tile
    (7, 1, 112, 16, 16300, 9),   # 63 rows, long context
    (8, 8, 32, 16, 127, 1),      # one partition exactly
    (8, 8, 32, 16, 128, 1),      # and one key more
    (2, 2, 224, 16, 0, 1),       # the window's own key alone
]


@pytest.mark.parametrize("nh,nkv,dph,bs,ctx,M", SIZES + ROWS)
def test_tile_form_matches_float64(gpu, oracle, nh, nkv, dph, bs, ctx, M):
    case_banner("tile form", nh, nkv, dph, bs, ctx, M)
    cache, K, V, rng = build_layer(nh, nkv, dph, bs, ctx, M, -(-(ctx + M) // bs) + 9, dph + ctx)
    q = W.queries(rng, M, nh, dph)
    qt = torch.from_numpy(q).cuda()
    nan = torch.full((M, nh * dph), float("nan"), device="cuda")
    out = cache.attention(0, qt, nh, nkv, dph, ctx, out=nan.clone())
    again = cache.attention_noalloc(0, qt, nh, nkv, dph, ctx, out=nan.clone())
    ws = torch.empty(max(4, cache.workspace_size(nh, nkv, dph, M, ctx + M)) // 4, device="cuda")
    third = cache.attention(0, qt, nh, nkv, dph, ctx, out=nan.clone(), workspace=ws)
    torch.cuda.synchronize()
    assert torch.equal(out, again) and torch.equal(out, third)
    ref = oracle.attention_f64_np(q, K, V, nh, nkv, dph, ctx)
    check(out.cpu().numpy(), ref, f"dph {dph} bs {bs} ctx {ctx}")
    cache.free()


@pytest.mark.parametrize("dph,bs", [(24, 16), (80, 16), (96, 16), (200, 16), (256, 7)])
def test_tile_form_hidden_nonfinite_rows(gpu, oracle, dph, bs):
    """Inf / NaN in V and NaN in K at a window position, and stale NaN past
    the window, reach only the queries that see them; fp16 padding features
    never reach an output."""
    case_banner("tile form, hidden non-finite", dph, bs)
    nh, nkv, ctx, M = 4, 2, 200, 9
    cache, K, V, rng = build_layer(nh, nkv, dph, bs, ctx, M, 60, dph)
    bad = ctx + 4
    k, v = K[bad].copy(), V[bad].copy()
    v[::3], v[1::3], k[5] = np.inf, np.nan, np.nan
    cache.append(0, torch.from_numpy(k[None]).cuda(), torch.from_numpy(v[None]).cuda(), bad)
    last = ctx + M
    if last % bs:
        table = cache.block_table(0)
        cache.pool_blocks_view()[int(table[last // bs]), :, last % bs:] = 0x7E00  # NaN
    q = W.queries(rng, M, nh, dph)
    out = cache.attention(0, torch.from_numpy(q).cuda(), nh, nkv, dph, ctx).cpu().numpy()
    ref = oracle.attention_f64_np(q[:4], K[:bad], V[:bad], nh, nkv, dph, ctx)
    check(out[:4], ref, "queries that do not see it")
    # (KV head 0's rows hold the NaN key: not finite from query 4 on)
    assert not np.isfinite(out[4:, :dph]).any()
    cache.free()


def _rotated(q, heads, dph, ctx, theta):
    """Rotate-half RoPE in 64 bits at the path's own fp32 angles."""
    half = dph // 2
    inv = np.exp(-np.log(theta) * 2.0 * np.arange(half) / dph).astype(np.float32)
    pos = np.arange(ctx, ctx + q.shape[0], dtype=np.float32)
    ang = (pos[:, None] * inv[None, :]).astype(np.float64)[:, None, :]
    x = q.astype(np.float64).reshape(q.shape[0], heads, dph)
    a, b = x[..., :half], x[..., half:]
    y = np.concatenate([a * np.cos(ang) - b * np.sin(ang), a * np.sin(ang) + b * np.cos(ang)], -1)
    return y.reshape(q.shape).astype(np.float32)


@pytest.mark.parametrize("nh,nkv,dph,bs,ctx,M", [
    (1, 1, 8, 16, 0, 1),       # four pairs in all
    (3, 1, 24, 16, 130, 1),    # halves that are no multiple of 8
    (16, 1, 32, 16, 500, 1),   # a full group of 16 rows
    (17, 1, 40, 16, 500, 1),   # one row past it
    (7, 1, 96, 16, 300, 5),    # groups that begin inside a query's heads
    (4, 4, 120, 12, 700, 9),
    (12, 4, 64, 12, 700, 3),   # head size 64 with a block size of this form
    (16, 8, 256, 16, 3000, 5),
    (32, 2, 256, 16, 257, 2),  # 32 rows, all pairs of a thread in use
    (24, 2, 200, 16, 900, 9),  # 108 rows, the last group not full
])
def test_tile_form_rope_equals_rotated_queries(gpu, nh, nkv, dph, bs, ctx, M):
    """The call with RoPE against the same call on queries rotated beforehand."""
    case_banner("tile form, rope", nh, nkv, dph, bs, ctx, M)
    cache, K, V, rng = build_layer(nh, nkv, dph, bs, ctx, M, -(-(ctx + M) // bs) + 9, dph + ctx)
    q = W.queries(rng, M, nh, dph)
    k = rng.standard_normal((M, nkv * dph)).astype(np.float32)
    v = rng.standard_normal((M, nkv * dph)).astype(np.float32)
    got = cache.rope_append_attention(0, *(torch.from_numpy(t).cuda() for t in (q, k, v)), nh,
                                      nkv, dph, ctx, theta=10000.0)
    # (the window's keys are in the cache now, rotated)
    want = cache.attention(0, torch.from_numpy(_rotated(q, nh, dph, ctx, 10000.0)).cuda(), nh,
                           nkv, dph, ctx)
    keys, _ = cache.read(0, 0, ctx + M)
    # An element's rotation is within 2^-21 of its pair's norm (sine, cosine,
    # two products and a sum in fp32), so a logit within 2^-21 |q| |k| /
    # sqrt(dph) and a softmax mean within twice that of the largest |v|; both
    # calls' own sums add 2^-19.
    qn = float(np.linalg.norm(q.reshape(-1, dph), axis=1).max())
    kn = float(keys.reshape(-1, dph).norm(dim=1).max())
    vmax = max(float(np.abs(V).max()) if ctx else 0.0, float(np.abs(v).max()))
    bound = (2.0 ** -20 * qn * kn / np.sqrt(dph) + 2.0 ** -19) * vmax
    assert float((got - want).abs().max()) <= bound
    cache.free()
