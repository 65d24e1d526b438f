"""The attention workspace that a cache owns: what it costs in device memory,
and calls captured into a HIP graph without a workspace of their own."""
import gc

import pytest
import torch

from conftest import case_banner
from speculative_decode_engine_amd import KVCache
from speculative_decode_engine_amd._native import SDEError

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def free_bytes():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def small_cache(nkv, dph, keys, bs=16):
    return KVCache(1, nkv * dph, -(-keys // bs), bs)


def test_a_cache_takes_its_workspace_when_a_call_needs_it(gpu):
    """A cache per sequence: 32 of them take their pools and tables, and a
    decode call each its own split's partials (here 0.5 MiB), not the most
    that a plan can take."""
    case_banner("workspace of many caches")
    nh, nkv, dph, keys = 32, 8, 128, 2048
    q = torch.randn(1, nh * dph, device="cuda")
    out = torch.empty_like(q)
    small_cache(nkv, dph, keys).attention(0, q, nh, nkv, dph, keys - 1, out=out)
    gc.collect()
    before = free_bytes()
    caches = [KVCache(1, nkv * dph, keys // 16, 16, pool="library") for _ in range(32)]
    pools = 32 * 2 * keys * nkv * dph * 2
    assert before - free_bytes() <= pools + 32 * 2 * MIB  # (allocations come in 2 MiB)
    for c in caches:
        c.attention(0, q, nh, nkv, dph, keys - 1, out=out)
    assert before - free_bytes() <= pools + 32 * 4 * MIB
    for c in caches:
        c.free()


def test_workspace_growth_ends_at_the_largest_plan(gpu):
    """A chunk whose split takes 12.7 MiB, then one that takes 16.3: the
    second call's growth stops at the 18 MiB that any plan takes."""
    case_banner("workspace growth")
    nh, nkv, dph = 32, 8, 128
    cache = small_cache(nkv, dph, 4400)
    outs = []
    for m in (400, 128):
        q = torch.randn(m, nh * dph, device="cuda")
        out = torch.empty_like(q)
        before = free_bytes()
        cache.attention(0, q, nh, nkv, dph, 4000, out=out)
        outs.append(before - free_bytes())
    assert outs[0] > 0 and outs[1] <= 20 * MIB
    before = free_bytes()
    for m in (400, 128):
        cache.attention(0, torch.randn(m, nh * dph, device="cuda"), nh, nkv, dph, 4000)
    torch.cuda.empty_cache()
    assert before - free_bytes() <= 0
    cache.free()


def capture(cache, fn):
    g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(g, stream=s):
        fn()
    return g


SHAPES = [
    # nh, nkv, dph, ctx, m: the matrix-core form's plan takes less than the
    # fp32 form's in the first three, more in the fourth; the 16-row kernels;
    # a wide window that they would run in one partition, and one in several
    (32, 32, 96, 4199, 1),
    (16, 8, 256, 12000, 1),
    (16, 2, 256, 12000, 9),
    (8, 8, 64, 2000, 3),
    (32, 8, 128, 3000, 5),
    (32, 4, 64, 1500, 256),
    (8, 2, 128, 60100, 24),
]


@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("nh,nkv,dph,ctx,m", SHAPES)
def test_a_call_captures_after_its_eager_run(gpu, nh, nkv, dph, ctx, m, rope):
    """On the cache's own workspace, which the eager call made: the captured
    call runs the same plan, so that replays, with other eager work between
    them, give the same bits."""
    case_banner("capture after eager", nh, nkv, dph, ctx, m, rope)
    if rope and m > 32:
        pytest.skip("the call with RoPE takes 32 queries")
    bs = 12 if dph == 64 and nh == 8 else 16
    cache = small_cache(nkv, dph, ctx + m, bs)
    cache.pool.copy_(torch.randn(cache.pool.numel(), device="cuda").half().view(torch.int16))
    q = torch.randn(m, nh * dph, device="cuda")
    k, v = torch.randn(2, m, nkv * dph, device="cuda").unbind(0)
    out = torch.zeros_like(q)

    def call(q, out):
        if rope:
            return cache.rope_append_attention(0, q, k, v, nh, nkv, dph, ctx, out=out)
        return cache.attention(0, q, nh, nkv, dph, ctx, out=out)

    call(q, out)
    g = capture(cache, lambda: call(q, out))
    for _ in range(3):
        eager = call(q, torch.empty_like(out)).clone()
        call(-q, torch.empty_like(out))
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        q.mul_(0.75)
    cache.free()


@pytest.mark.parametrize("nh,nkv,dph,ctx", [(32, 8, 128, 3000), (16, 8, 256, 3000),
                                            (32, 32, 96, 4199)])
def test_a_split_call_that_is_the_first_is_refused_under_capture(gpu, nh, nkv, dph, ctx):
    case_banner("capture first", nh, nkv, dph, ctx)
    cache = small_cache(nkv, dph, ctx + 1)
    q = torch.randn(1, nh * dph, device="cuda")
    out = torch.zeros_like(q)
    other = torch.zeros_like(q)

    def call():
        other.copy_(q)
        with pytest.raises(SDEError, match="workspace"):
            cache.attention(0, q, nh, nkv, dph, ctx, out=out)

    capture(cache, call)
    cache.free()
