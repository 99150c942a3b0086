"""Rows of any address, distance and length on the MFMA kernels as they stand (option any_shape = 3: wherever possible): every row
of every family by name, the rest of K behind the last 16-byte chunk, what lies around the operands.  Small integers and powers of two:
every product and sum is exact, so the results are the oracle's."""
import numpy as np
import pytest
import torch

import qgemm_amd as Q
from oracle import cpu_ref as R
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
    for row in [None] + _rows(dtype, Q.SCALE_BLOCK128, 0):
        for split in (1, 2):
            say("unaligned, block scales", K, dtype, row, split)
            Q.force_config(row)
            Q.set_option("force_split", split)
            c = torch.zeros((M, N), dtype=torch.bfloat16, device="cuda")
            Q.scaled_gemm(at, bt, dev(as_), dev(bs), c, M, N, K, Q.SCALE_BLOCK128)
            assert torch.equal(c.cpu(), ref.to(torch.bfloat16)), (row, split, Q.last_config())


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
