"""The attention workspace that a cache owns: what it costs in device memory,
and calls captured into a HIP graph without a workspace of their own."""
import gc

import pytest
import torch

from conftest import case_banner
from speculative_decode_engine_amd import KVCache

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
