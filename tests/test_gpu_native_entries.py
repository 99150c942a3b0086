"""The functions of qgemm_amd through the extension module and through ctypes: the same library entries, so the same bits
and the same errors."""
import pytest
import torch

import qgemm_amd as Q
from qgemm_amd import ops
from tests.util import say

pytestmark = pytest.mark.gpu


@pytest.fixture(params=["native", "ctypes"])
def way(request, monkeypatch):
    module = ops._native()
    assert module, "the extension module is not built"
    if request.param == "ctypes":
        monkeypatch.setattr(ops, "_native_module", False)
    return request.param


def _both(f, monkeypatch):
    with_native = f()
    monkeypatch.setattr(ops, "_native_module", False)
    return with_native, f()


@pytest.mark.parametrize("source", [torch.float32, torch.bfloat16, torch.float16])
def test_the_same_bits(source, monkeypatch):
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    x, w = (torch.randn(r, 300, generator=g, device="cuda").to(source) for r in (70, 200))

    def all_of_them():
        out = []
        say("entries", source, bool(ops._native()))
        for dt in (torch.int8, torch.float8_e4m3fn):
            for mode in (Q.QUANT_PER_MATRIX, Q.QUANT_BLOCK_1x128, Q.QUANT_BLOCK_128x128):
                for rc in (False, True):
                    out += Q.quantize(x[:, 4:], dt, mode, rc)
            (q, s), (v, t) = Q.quantize(x, dt, Q.QUANT_BLOCK_1x128), Q.quantize(w, dt, Q.QUANT_BLOCK_128x128)
            out.append(Q.scaled_gemm(q, v, s, t, torch.empty(70, 256, dtype=torch.bfloat16, device="cuda")[:, :200], 70, 200, 300,
                                     Q.SCALE_BLOCK128).clone())
        out.append(Q.matrix_transpose(x, torch.empty(300, 70, dtype=source, device="cuda")))
        if source != torch.float32:
            out.append(Q.gemm(x, w, torch.empty(70, 200, device="cuda")))
            out.append(Q.gemm(x, w.t().contiguous(), torch.empty(70, 200, device="cuda"), "kn"))
            out.append(Q.gemm(x, w, torch.empty(70, 200, device="cuda"), "nk", M=3, N=70, K=128, ldA=300)[:3, :70].clone())
        return out

    native, plain = _both(all_of_them, monkeypatch)
    assert len(native) == len(plain)
    for a, b in zip(native, plain):
        assert a.shape == b.shape and a.dtype == b.dtype
        view = {1: torch.uint8, 2: torch.int16, 4: torch.int32}[a.element_size()]
        assert torch.equal(a.contiguous().view(view), b.contiguous().view(view))


def test_the_same_errors(way):
    a = torch.zeros(32, 128, dtype=torch.bfloat16, device="cuda")
    c = torch.zeros(32, 32, device="cuda")
    with pytest.raises(ValueError):
        Q.gemm(a.cpu(), a, c)
    with pytest.raises(TypeError):
        Q.gemm(a.double(), a, c)
    with pytest.raises(TypeError):
        Q.gemm(a, a, c.to(torch.uint8))
    with pytest.raises(KeyError):
        Q.gemm(a, a, c, "nn")
    with pytest.raises(Q.QgemmError) as e:
        Q.gemm(a, a, c, "nk", ldC=1)
    assert e.value.status == 1
    with pytest.raises(Q.QgemmError) as e:
        Q.scaled_gemm(a, a, None, None, c, 32, 32, 128, Q.SCALE_PER_MATRIX)
    assert e.value.status == 2
    with pytest.raises(Q.QgemmError) as e:
        Q.quantize(a, torch.int32)
    assert e.value.status == 2
    with pytest.raises(AssertionError):
        Q.quantize(a[0])
    with pytest.raises(Q.QgemmError) as e:
        Q.matrix_transpose(a.double(), a.double())
    assert e.value.status == 2
