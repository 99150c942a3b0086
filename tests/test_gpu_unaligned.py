"""Rows of any address, distance and length on the MFMA kernels as they stand (option any_shape = 3: wherever possible): every row
of every family by name, the rest of K behind the last 16-byte chunk, what lies around the operands.  Small integers and powers of two:
every product and sum is exact, so the results are the oracle's."""
import ctypes as C

import numpy as np
import pytest
import torch

import qgemm_amd as Q
from oracle import cpu_ref as R
from qgemm_amd import lib as L
from tests.util import dev, host, say, scalar

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn


@pytest.fixture(autouse=True)
def _unaligned():
    Q.set_option("any_shape", 3)
    yield
    Q.set_option("any_shape", 1)
    Q.set_option("kmajor", 1)
    Q.set_option("force_split", 0)
    Q.force_config(None)


def _ints(rng, shape):
    return rng.integers(-4, 5, size=shape).astype(np.float32)


def _tensor(x, dtype, pad=0, off=0, around=float("nan")):
    """x on the device with `pad` elements between rows and `off` in front of the first, all of them `around` where the type has it."""
    r, c = x.shape
    if dtype == torch.int8:
        around = -128
    flat = torch.full((off + r * (c + pad) + 8,), around, dtype=torch.float32, device="cuda").to(dtype)
    t = flat[off:off + r * (c + pad)].view(r, c + pad)[:, :c]
    t.copy_(torch.from_numpy(x).to("cuda").to(dtype))
    return t


def _ran(row=None):
    c = Q.last_config()
    return c.startswith("unaligned+") and (row is None or row in c)


FAMILIES = [("nk", torch.bfloat16), ("nk", torch.float16), ("nk", torch.int8), ("nk", FP8), ("kn", torch.bfloat16), ("kn", torch.float16)]


def _rows(dtype, scale_mode, k_major):
    """Rows of the family that runs (fp8 rows run widened: names that family has not got are not taken as they stand)."""
    return Q.variant_names({torch.bfloat16: Q.DT_BF16, torch.float16: Q.DT_F16, torch.int8: Q.DT_I8, FP8: Q.DT_F8E4M3}[dtype], scale_mode, k_major)


@pytest.mark.parametrize("layout,dtype", FAMILIES)
@pytest.mark.parametrize("shape", [(130, 264, 1001), (257, 136, 129), (70, 392, 47)])
def test_every_row_by_name(shape, layout, dtype):
    M, N, K = shape
    rng = np.random.default_rng(M + K)
    a, b = _ints(rng, (M, K)), _ints(rng, (N, K))
    ref = torch.from_numpy(R.gemm_f32acc(a, b))
    at, bt = _tensor(a, dtype), _tensor(b if layout == "nk" else np.ascontiguousarray(b.T), dtype, 0 if layout == "nk" else 8, 0 if layout == "nk" else 8)
    ran = 0
    for row in _rows(dtype, 0, 0 if layout == "nk" else 2):
        for split in (1, 3):
            say("unaligned", shape, layout, dtype, row, split)
            Q.force_config(row)
            Q.set_option("force_split", split)
            c = torch.full((M, N), 7.0, dtype=torch.float32, device="cuda")
            Q.gemm(at, bt, c, layout)
            assert _ran(row) or dtype == FP8, Q.last_config()
            ran += _ran(row)
            assert torch.equal(c.cpu(), ref), (row, split)
    assert ran >= 8


@pytest.mark.parametrize("dtype", [torch.int8, FP8])
@pytest.mark.parametrize("K", [1001, 1025, 143, 271, 4104])
def test_block_scales_on_every_row(K, dtype):
    """K ends inside a block of scales, and one element or more into a block of its own."""
    M, N = 133, 260
    rng = np.random.default_rng(K)
    a, b, KB = _ints(rng, (M, K)), _ints(rng, (N, K)), (K + 127) // 128
    as_ = (2.0 ** rng.integers(-1, 2, size=(M, KB))).astype(np.float32)
    bs = (2.0 ** rng.integers(-1, 2, size=((N + 127) // 128, KB))).astype(np.float32)
    ref = torch.from_numpy(R.gemm_fp8_block(a, b, as_, bs))
    at, bt = _tensor(a, dtype), _tensor(b, dtype)
    ran = 0
    for row in [None] + _rows(dtype, Q.SCALE_BLOCK128, 0):
        for split in (1, 2):
            say("unaligned, block scales", K, dtype, row, split)
            Q.force_config(row)
            Q.set_option("force_split", split)
            c = torch.zeros((M, N), dtype=torch.bfloat16, device="cuda")
            Q.scaled_gemm(at, bt, dev(as_), dev(bs), c, M, N, K, Q.SCALE_BLOCK128)
            assert torch.equal(c.cpu(), ref.to(torch.bfloat16)), (row, split, Q.last_config())
            # (a row's twin for the arrangement of the scales may stand in for it; fp8 rows run on a family with fewer names)
            assert _ran(row and row.replace("_ks", "")) or (row and dtype == FP8), (row, Q.last_config())
            ran += _ran(row and row.replace("_ks", ""))
    assert ran >= 16, ran


@pytest.mark.parametrize("layout,dtype", FAMILIES)
@pytest.mark.parametrize("K", [256, 131, 72])
def test_strides_and_pointers(K, layout, dtype):
    """Gaps between the rows, full of NaNs, and pointers at any element; B stored K x N keeps its rows whole."""
    M, N = 150, 200
    rng = np.random.default_rng(K)
    a, b = _ints(rng, (M, K)), _ints(rng, (N, K))
    ref = torch.from_numpy(R.gemm_f32acc(a, b))
    bt = b if layout == "nk" else np.ascontiguousarray(b.T)
    ways = [((3, 0), (0, 0)), ((0, 5), (1, 0)), ((7, 1), (3, 5)), ((0, 0), (0, 1)), ((4, 8), (2, 6))] if layout == "nk" else [((3, 0), (0, 0)), ((0, 8), (1, 8)), ((7, 0), (3, 0))]
    for pads, offs in ways:
        say("unaligned, strides", K, layout, dtype, pads, offs)
        wide = torch.full((M, N + 3), 7.0, dtype=torch.float32, device="cuda")
        c = wide[:, :N]
        Q.gemm(_tensor(a, dtype, pads[0], offs[0]), _tensor(bt, dtype, pads[1], offs[1]), c, layout)
        assert _ran() or (layout == "kn" and K % 8 == 0), Q.last_config()
        assert torch.equal(c.cpu(), ref)
        assert bool((wide[:, N:] == 7).all())


def test_infinities_stay_in_their_rows():
    """An infinity or NaN inside a row reaches that row of C alone, also from the chunk K ends in."""
    M, N, K = 70, 130, 1003
    rng = np.random.default_rng(5)
    a, b = _ints(rng, (M, K)), np.abs(_ints(rng, (N, K))) + 1
    for k in (0, K - 1, K - 12, K - 14):
        x = a.copy()
        x[13, k], x[40, k] = np.inf, np.nan
        for row in (None, "128x128_w2x2_k2", "256x256_w2x4_solo8", "256x256_w2x2_solo", "skinny_64x64_k8"):
            say("unaligned, infinities", k, row)
            Q.force_config(row)
            c = torch.zeros((M, N), dtype=torch.float32, device="cuda")
            Q.gemm(_tensor(x, torch.bfloat16), _tensor(b, torch.bfloat16), c, "nk")
            assert _ran(row), Q.last_config()
            ref = R.gemm_f32acc(a, b)
            ref[13], ref[40] = np.inf, np.nan
            assert np.array_equal(host(c), ref, equal_nan=True)


def test_int8_accumulators():
    M, N, K = 300, 259, 777
    rng = np.random.default_rng(7)
    a, b = rng.integers(-128, 128, size=(M, K)).astype(np.int8), rng.integers(-128, 128, size=(N, K)).astype(np.int8)
    acc = R.gemm_i8_i32(a, b)
    for row in (None, "256x256_w2x2_solo", "192x256_w2x4_solo8", "64x128_w1x4_k2"):
        Q.force_config(row)
        for dtype, want in ((torch.int32, acc), (torch.float32, R.scale_i32_to_f32(acc, np.float32(0.5), np.float32(3.0)))):
            c = torch.zeros((M, N), dtype=dtype, device="cuda")
            Q.int8_mm(dev(a), dev(b), scalar(0.5), scalar(3.0), c)
            assert _ran(row), Q.last_config()
            assert np.array_equal(host(c), want)


def _chosen():
    """(call, output, expected): products that the estimates leave as they stand, by their own choice."""
    rng = np.random.default_rng(11)
    a, b = _ints(rng, (203, 1381)), _ints(rng, (4320, 1381))
    at, bt = _tensor(a, torch.float16), _tensor(np.ascontiguousarray(b.T), torch.float16)
    c = torch.empty((203, 4320), dtype=torch.float16, device="cuda")
    yield lambda: Q.gemm(at, bt, c, "kn"), c, torch.from_numpy(a @ b.T).half()
    a, b = rng.integers(-127, 128, (1532, 1004)).astype(np.int8), rng.integers(-127, 128, (1024, 1004)).astype(np.int8)
    ai, bi, one = dev(a), dev(b), scalar(1)
    ci = torch.empty((1532, 1024), dtype=torch.int32, device="cuda")
    yield lambda: Q.int8_mm(ai, bi, one, one, ci), ci, torch.from_numpy(R.gemm_i8_i32(a, b))
    M, N, K = 164, 1152, 2407
    a, b, KB = _ints(rng, (M, K)), _ints(rng, (N, K)), (K + 127) // 128
    as_, bs = (2.0 ** rng.integers(-1, 2, (M, KB))).astype(np.float32), (2.0 ** rng.integers(-1, 2, (N // 128, KB))).astype(np.float32)
    af, bf, sa, sb = _tensor(a, FP8), _tensor(b, FP8), dev(as_), dev(bs)
    cf = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    yield lambda: Q.scaled_gemm(af, bf, sa, sb, cf, M, N, K, Q.SCALE_BLOCK128), cf, torch.from_numpy(R.gemm_fp8_block(a, b, as_, bs)).to(torch.bfloat16)


def test_chosen_eager_and_captured():
    Q.set_option("any_shape", 1)
    for call, c, want in _chosen():
        c.zero_()
        call()
        say("unaligned, chosen", Q.last_config())
        assert _ran(), Q.last_config()
        assert torch.equal(c.cpu(), want)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            call()
        assert _ran(), Q.last_config()
        for _ in range(3):
            c.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(c.cpu(), want)


def test_chosen_on_the_static_scratch():
    Q.set_option("any_shape", 1)
    M, N, K = 1532, 1024, 1004
    rng = np.random.default_rng(13)
    a, b = rng.integers(-127, 128, (M, K)).astype(np.int8), rng.integers(-127, 128, (N, K)).astype(np.int8)
    ad, bd, one, c = dev(a), dev(b), scalar(1), torch.zeros((M, N), dtype=torch.int32, device="cuda")
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    L.check(L.load_library().qgemm_scaled_gemm_static(Q.DT_I8, Q.DT_I32, Q.SCALE_PER_MATRIX, Q.LAYOUT_K_CONTIGUOUS, ad.data_ptr(), bd.data_ptr(),
                                                      one.data_ptr(), one.data_ptr(), c.data_ptr(), N, M, N, K, 0, stream))
    assert _ran(), Q.last_config()
    assert np.array_equal(host(c), R.gemm_i8_i32(a, b))


@pytest.mark.parametrize("dtype", [torch.int8, FP8])
@pytest.mark.parametrize("K", [1001, 1025, 143, 4104])
def test_block_scales_against_64_bits(K, dtype):
    """Values of every size: an element is a sum of KB + 1 folded parts, the last block's in two, rounded once each beside the roundings
    of factor and product, and a few where K groups and slices meet; fp8 parts are fp32 sums of up to 128 products themselves."""
    M, N, KB = 133, 260, (K + 127) // 128
    rng = np.random.default_rng(K + 1)
    if dtype == torch.int8:
        at, bt = (dev(rng.integers(-127, 128, (rows, K)).astype(np.int8)) for rows in (M, N))
    else:
        at, bt = (dev(rng.normal(size=(rows, K)).astype(np.float32) * 60).clamp(-440, 440).to(FP8) for rows in (M, N))
    as_, bs = rng.uniform(1e-3, 1e-1, (M, KB)).astype(np.float32), rng.uniform(1e-3, 1e-1, ((N + 127) // 128, KB)).astype(np.float32)
    a = at.float().cpu().double() * torch.from_numpy(as_).double().repeat_interleave(128, 1)[:, :K]
    b = bt.float().cpu().double() * torch.from_numpy(bs).double().repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)[:, :K]
    ref, size = a @ b.T, a.abs() @ b.abs().T
    bound = (KB + 1 + 2 + 8 + (128 if dtype == FP8 else 0)) * 2.0 ** -24 * size
    for row in [None] + _rows(dtype, Q.SCALE_BLOCK128, 0):
        for split in (1, 2):
            say("unaligned, block scales, 64 bits", K, dtype, row, split)
            Q.force_config(row)
            Q.set_option("force_split", split)
            c = torch.zeros((M, N), dtype=torch.float32, device="cuda")
            Q.scaled_gemm(at, bt, dev(as_), dev(bs), c, M, N, K, Q.SCALE_BLOCK128)
            if dtype == FP8 and not _ran():
                continue
            assert _ran(row and row.replace("_ks", "")), (row, Q.last_config())
            assert bool(((c.cpu().double() - ref).abs() <= bound).all()), (row, split, Q.last_config())
