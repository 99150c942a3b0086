"""Captured products whose operands the MFMA kernels cannot copy as they stand: replays are ordered by nobody, so they keep
nothing in the workspace that all calls share.  The same for the entry on the static scratch."""
import ctypes as C

import numpy as np
import pytest
import torch

import qgemm_amd as Q
from oracle import cpu_ref as R
from qgemm_amd import lib as L
from tests.util import dev, host, say, scalar

pytestmark = pytest.mark.gpu


class _Bytes:
    def __init__(self, base, size):
        self.__cuda_array_interface__ = dict(data=(base, False), shape=(size,), typestr="|u1", version=2)


def _workspace():
    """The library's block as a tensor."""
    base, size = C.c_void_p(), C.c_size_t()
    L.check(L.load_library().qgemm_reserve_workspace(32 << 20))
    L.check(L.load_library().qgemm_workspace_info(C.byref(base), C.byref(size)))
    return torch.as_tensor(_Bytes(base.value, size.value), device="cuda")


def _capture(f):
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        f()
    return g


def _products(seed):
    """(call, output, expected): int8 with one scale, bf16 with B stored K x N, int8 with block scales; small integers and
    powers of two, exact in every order of summation."""
    rng = np.random.default_rng(seed)
    M, N, K = 130, 700, 1001
    KB = (K + 127) // 128
    a, b = rng.integers(-4, 5, (M, K)), rng.integers(-4, 5, (N, K))
    ref = R.gemm_i8_i32(a.astype(np.int8), b.astype(np.int8))
    one = scalar(1.0)
    a8, b8 = dev(a.astype(np.int8)), dev(b.astype(np.int8))
    c8 = torch.zeros(M, N, dtype=torch.int32, device="cuda")
    yield lambda: Q.int8_mm(a8, b8, one, one, c8), c8, ref
    ah, bh = dev(a.astype(np.float32)).bfloat16(), dev(np.ascontiguousarray(b.T).astype(np.float32)).bfloat16()
    ch = torch.zeros(M, N, device="cuda")
    yield lambda: Q.gemm(ah, bh, ch, "kn"), ch, ref.astype(np.float32)
    as_ = (2.0 ** rng.integers(-1, 2, (M, KB))).astype(np.float32)
    bs = (2.0 ** rng.integers(-1, 2, ((N + 127) // 128, KB))).astype(np.float32)
    sa, sb, cs = dev(as_), dev(bs), torch.zeros(M, N, device="cuda")
    yield lambda: Q.scaled_gemm(a8, b8, sa, sb, cs, M, N, K, Q.SCALE_BLOCK128), cs, R.gemm_i8_block(a.astype(np.int8), b.astype(np.int8), as_, bs)


def test_captured_products_leave_the_workspace_alone():
    ws = _workspace()
    for call, c, want in _products(1):
        say("captured any-shape product beside the workspace")
        g = _capture(call)
        ws.fill_(0x5A)
        for _ in range(3):
            c.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert np.array_equal(host(c), want)
        assert bool((ws == 0x5A).all())


def test_replays_on_two_streams():
    _workspace()
    pairs = list(zip(_products(2), _products(3)))
    for first, second in pairs:
        graphs = [(_capture(call), c, want, torch.cuda.Stream()) for call, c, want in (first, second)]
        say("any-shape replays on two streams")
        for _ in range(4):
            for _, c, _, _ in graphs:
                c.zero_()
            torch.cuda.synchronize()
            for _ in range(20):
                for g, _, _, s in graphs:
                    with torch.cuda.stream(s):
                        g.replay()
            torch.cuda.synchronize()
            for _, c, want, _ in graphs:
                assert np.array_equal(host(c), want)


@pytest.mark.parametrize("N", [300, 33000])        # (packed, the second B alone would exceed the scratch)
def test_the_static_entry(N):
    M, K = 40, 1019
    rng = np.random.default_rng(N)
    a, b = (rng.integers(-127, 128, (r, K)).astype(np.int8) for r in (M, N))
    ad, bd, sa, sb = dev(a), dev(b), scalar(0.5), scalar(3.0)
    lib, stream = L.load_library(), C.c_void_p(torch.cuda.current_stream().cuda_stream)
    out = []
    for fn in (lib.qgemm_scaled_gemm, lib.qgemm_scaled_gemm_static):
        say("any-shape product, static entry", (M, N, K))
        c = torch.zeros(M, N, device="cuda")
        assert fn(Q.DT_I8, Q.DT_F32, Q.SCALE_PER_MATRIX, Q.LAYOUT_K_CONTIGUOUS, ad.data_ptr(), bd.data_ptr(), sa.data_ptr(),
                  sb.data_ptr(), c.data_ptr(), N, M, N, K, 0, stream) == 0
        out.append(host(c))
    assert np.array_equal(out[0], R.scale_i32_to_f32(R.gemm_i8_i32(a, b), np.float32(0.5), np.float32(3.0)))
    assert np.array_equal(out[0], out[1])
