"""The Python entry points' argument checks over the forms a tensor can take:
the one-pass test of the usual case accepts exactly what the full checks
return unchanged, every other form is accepted with the same result or
refused with the same exception, and calls go to the stream they name (or
the current one)."""
import pytest
import torch

from conftest import case_banner
from speculative_decode_engine_amd import KVCache, matvec, matvec_packed, PackedWeight
from speculative_decode_engine_amd.kv_cache import _dev_f32, _is_f32

pytestmark = pytest.mark.gpu


def forms():
    x = torch.randn(3, 128, device="cuda")
    sub = torch.nn.Parameter(x.clone(), requires_grad=False)
    return {"plain": x, "parameter": sub, "grad": x.clone().requires_grad_(),
            "double": x.double(), "half": x.half(), "cpu": x.cpu(), "strided": x.t().t()[:, ::1],
            "transposed": torch.randn(128, 3, device="cuda").t(),
            "gaps": torch.randn(3, 256, device="cuda")[:, ::2], "short": x[:2],
            "flat": x.reshape(-1), "three": x.view(3, 2, 64), "array": x.cpu().numpy()}


def test_one_pass_check_agrees_with_the_full_one(gpu):
    case_banner("call forms: predicate")
    for name, t in forms().items():
        try:
            same = _dev_f32(t, "t", (3, 128)) is t
        except (TypeError, ValueError):
            same = False
        assert not _is_f32(t, (3, 128)) or same, name
        if name in ("plain", "grad", "strided"):
            assert _is_f32(t, (3, 128)), name


def test_attention_and_append_forms(gpu):
    case_banner("call forms: attention")
    cache = KVCache(1, 128, 8, 16)
    k = torch.randn(20, 128, device="cuda")
    cache.append(0, k, k, 0)
    q = forms()
    ref = cache.attention(0, q["plain"], 2, 2, 64, 10)
    for name in ("parameter", "grad", "strided"):
        t = q[name].detach() if name == "grad" else q[name]
        assert torch.equal(cache.attention(0, t, 2, 2, 64, 10),
                           cache.attention(0, t.clone(), 2, 2, 64, 10)), name
    one = cache.attention(0, q["plain"][0], 2, 2, 64, 10)  # a single row, 1-D
    assert torch.equal(one, ref[:1])
    for name, err in [("double", TypeError), ("half", TypeError), ("cpu", TypeError),
                      ("transposed", ValueError), ("gaps", ValueError)]:
        with pytest.raises(err):
            cache.attention(0, q[name], 2, 2, 64, 10)
        with pytest.raises(err):
            cache.append(0, q[name], q["plain"], 10)
    with pytest.raises(ValueError):
        cache.attention(0, q["plain"], 2, 2, 64, 10, out=q["short"].clone())
    with pytest.raises(TypeError):
        cache.attention(0, q["plain"], 2, 2, 64, 10, out=q["half"].clone())
    side = torch.cuda.Stream()
    out = torch.zeros_like(ref)
    side.wait_stream(torch.cuda.current_stream())
    cache.attention(0, q["plain"], 2, 2, 64, 10, out=out, stream=side)
    side.synchronize()
    assert torch.equal(out, ref)
    with torch.cuda.stream(side):
        assert torch.equal(cache.attention(0, q["plain"], 2, 2, 64, 10), ref)
    torch.cuda.synchronize()
    cache.free()
    with pytest.raises(RuntimeError):
        cache.attention(0, q["plain"], 2, 2, 64, 10)


def test_matvec_forms(gpu):
    case_banner("call forms: matvec")
    W = torch.randn(128, 64, device="cuda").half()
    P = PackedWeight(W)
    x = forms()
    for fn, w in ((matvec, W), (matvec_packed, P)):
        ref = fn(x["plain"], w)
        assert torch.equal(fn(x["parameter"], w), fn(x["parameter"].detach().clone(), w))
        assert fn(x["plain"][1], w).shape == (64,)
        out = torch.zeros(3 * 64, device="cuda")  # (any contiguous fp32 of the size)
        assert torch.equal(fn(x["plain"], w, out=out).view(3, 64), ref)
        for name in ("double", "cpu", "transposed", "gaps"):
            with pytest.raises(TypeError):
                fn(x[name], w)
        for bad in (torch.zeros(2, 64, device="cuda"), ref.double(), ref.cpu(),
                    torch.zeros(64, 3, device="cuda").t()):
            with pytest.raises(TypeError):
                fn(x["plain"], w, out=bad)
        with pytest.raises(ValueError):
            fn(x["plain"], w, accumulate=True)
