"""Operands the MFMA kernels cannot copy as they stand (K bytes not a multiple of 16, unaligned rows or pointers): packed for
those kernels (any_shape = 2) and on the any-shape kernel (any_shape = 0).  Inputs are small integers, every product and sum
of which is exact in every type the kernels sum in, so both forms give the oracle's numbers exactly."""
import numpy as np
import pytest
import torch

import qgemm_amd as Q
from oracle import cpu_ref as R
from tests.util import dev, host, say, scalar

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _reset_options():
    yield
    Q.set_option("any_shape", 1)
    Q.set_option("force_split", 0)


def _ran(any_shape):
    """Did the way that was asked for run?  (Both give the same numbers here.)"""
    return Q.last_config().startswith("pack+") if any_shape == 2 else Q.last_config() == "strided_any_shape"


def _ints(rng, shape):
    return rng.integers(-4, 5, size=shape).astype(np.float32)


def _tensor(x, dtype, pad_cols=0, off=0):
    """x on the device as dtype; pad_cols: extra columns between rows; off: elements between a 16-byte boundary and the first."""
    r, c = x.shape
    flat = torch.zeros(off + r * (c + pad_cols), dtype=torch.float32, device="cuda")
    t = flat.to(dtype)[off:].view(r, c + pad_cols)[:, :c]
    t.copy_(torch.from_numpy(x).to("cuda").to(dtype))
    return t


# edges of the packing: one 16-byte piece and less, one element around 128-byte steps and 64 / 128 / 256 tiles
SHAPES = [(1, 1, 65), (3, 5, 127), (16, 33, 129), (65, 255, 71), (64, 257, 193), (129, 127, 1001), (300, 130, 513), (33, 513, 2049)]


@pytest.mark.parametrize("any_shape", [0, 2])
@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.int8, torch.float8_e4m3fn])
@pytest.mark.parametrize("shape", SHAPES)
def test_product(shape, dtype, layout, any_shape):
    M, N, K = shape
    say("any shape", shape, dtype, layout, any_shape)
    rng = np.random.default_rng(M + N + K)
    a, b = _ints(rng, (M, K)), _ints(rng, (N, K))
    ref = R.gemm_f32acc(a, b)
    out = torch.bfloat16 if dtype == torch.float8_e4m3fn else torch.float32
    Q.set_option("any_shape", any_shape)
    c = torch.full((M, N), 7.0, dtype=out, device="cuda")
    Q.gemm(_tensor(a, dtype), _tensor(b if layout == "nk" else np.ascontiguousarray(b.T), dtype), c, layout)
    assert _ran(any_shape), Q.last_config()
    assert torch.equal(c.cpu(), torch.from_numpy(ref).to(out))


@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.int8])
@pytest.mark.parametrize("K", [256, 131])
def test_leading_dimensions_and_pointers(K, dtype, layout):
    M, N = 70, 90
    rng = np.random.default_rng(K)
    a, b = _ints(rng, (M, K)), _ints(rng, (N, K))
    ref = torch.from_numpy(R.gemm_f32acc(a, b))
    bt = b if layout == "nk" else np.ascontiguousarray(b.T)
    Q.set_option("any_shape", 2)
    for pads, offs in (((3, 0), (0, 0)), ((0, 5), (1, 0)), ((7, 1), (3, 5)), ((0, 0), (0, 1))):
        say("any shape, strides", dtype, layout, pads, offs)
        wide = torch.full((M, N + 3), 7.0, dtype=torch.float32, device="cuda")
        c = wide[:, :N]
        Q.gemm(_tensor(a, dtype, pads[0], offs[0]), _tensor(bt, dtype, pads[1], offs[1]), c, layout)
        if layout == "nk" or K % 16 or pads != (0, 0):        # (else B goes through the transpose kernel alone)
            assert _ran(2), Q.last_config()
        assert torch.equal(c.cpu(), ref)
        assert bool((wide[:, N:] == 7).all())            # (what lies between the rows of C)


@pytest.mark.parametrize("dtype", [torch.int8, torch.float8_e4m3fn])
@pytest.mark.parametrize("shape", [(5, 129, 130), (70, 140, 1023), (200, 300, 391)])
def test_block_scales(shape, dtype):
    M, N, K = shape
    say("any shape, block scales", shape, dtype)
    rng = np.random.default_rng(K)
    a, b, KB = _ints(rng, (M, K)), _ints(rng, (N, K)), (K + 127) // 128
    as_ = (2.0 ** rng.integers(-1, 2, size=(M, KB))).astype(np.float32)
    bs = (2.0 ** rng.integers(-1, 2, size=((N + 127) // 128, KB))).astype(np.float32)
    ref = torch.from_numpy(R.gemm_fp8_block(a, b, as_, bs))
    for any_shape in (0, 2):
        for split in (0, 2):
            Q.set_option("any_shape", any_shape)
            Q.set_option("force_split", split)
            c = torch.zeros((M, N), dtype=torch.bfloat16, device="cuda")
            Q.scaled_gemm(_tensor(a, dtype), _tensor(b, dtype), dev(as_), dev(bs), c, M, N, K, Q.SCALE_BLOCK128)
            assert _ran(any_shape), Q.last_config()
            assert torch.equal(c.cpu(), ref.to(torch.bfloat16)), (any_shape, split)


def test_int8_accumulators_and_one_scale():
    M, N, K = 130, 259, 777
    rng = np.random.default_rng(7)
    a, b = rng.integers(-127, 128, size=(M, K)).astype(np.int8), rng.integers(-127, 128, size=(N, K)).astype(np.int8)
    acc = R.gemm_i8_i32(a, b)
    Q.set_option("any_shape", 2)
    for dtype, want in ((torch.int32, acc), (torch.float32, R.scale_i32_to_f32(acc, np.float32(0.5), np.float32(3.0)))):
        c = torch.zeros((M, N), dtype=dtype, device="cuda")
        Q.int8_mm(dev(a), dev(b), scalar(0.5), scalar(3.0), c)
        assert _ran(2), Q.last_config()
        assert np.array_equal(host(c), want)


def test_capture_without_room_uses_no_workspace():
    """While a stream is captured nothing is packed: the any-shape kernel, which needs no workspace, runs."""
    Q.load_library().qgemm_shutdown()       # (gives the workspace back: it is empty when the capture begins)
    a, b = (torch.randint(-3, 4, (r, 9001), device="cuda").to(torch.int8) for r in (64, 96))
    c, want = (torch.zeros(64, 96, dtype=torch.int32, device="cuda") for _ in range(2))
    one = scalar(1.0)
    Q.set_option("any_shape", 0)
    Q.int8_mm(a, b, one, one, want)
    Q.set_option("any_shape", 2)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        Q.int8_mm(a, b, one, one, c)
    assert _ran(0), Q.last_config()
    for _ in range(3):
        c.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, want)


@pytest.mark.parametrize("shape", [(1, 1), (7, 9), (63, 257), (129, 130), (200, 1001), (255, 16), (16, 255), (1999, 301)])
@pytest.mark.parametrize("dtype", [torch.uint8, torch.bfloat16, torch.int32])
def test_transpose(shape, dtype):
    x = torch.randint(0, 200, shape, device="cuda").to(dtype)
    for off in (0, 1):
        say("transpose", shape, dtype, off)
        src = torch.zeros(x.numel() + off, dtype=dtype, device="cuda")[off:].view(shape)
        src.copy_(x)
        guard = torch.full((x.numel() + 2 * off + 16,), 99, dtype=dtype, device="cuda")
        dst = guard[off:off + x.numel()].view(shape[1], shape[0])
        Q.matrix_transpose(src, dst)
        assert torch.equal(dst, x.t())
        assert bool((guard[:off] == 99).all()) and bool((guard[off + x.numel():] == 99).all())


@pytest.mark.parametrize("out", [torch.bfloat16, torch.float16, torch.float32, torch.int32])
@pytest.mark.parametrize("row", ["256x256_w2x2_solo", "256x256_w2x4_solo8", "256x128_w2x2_cw", "128x128_w2x2_k2", "64x128_w1x4_k2", "128x128_w2x2_dma"])
def test_rows_of_c_that_end_inside_a_piece(row, out):
    """The last 16-byte piece of a row of C holds 1 .. 7 elements (1 .. 3 of four bytes): the same numbers, and nothing written
    beside them.  Small integers: exact in every output type."""
    M, K = 77, 128
    Q.force_config(row)
    try:
        for N in list(range(257, 265)) + [1, 5, 7]:
            say("ends of rows", row, out, N)
            rng = np.random.default_rng(N)
            a, b = rng.integers(-2, 3, size=(M, K)).astype(np.int8), rng.integers(-1, 2, size=(N, K)).astype(np.int8)
            c = torch.full((M, N + 9), 7, dtype=out, device="cuda")
            Q.scaled_gemm(dev(a), dev(b), scalar(1), scalar(1), c[:, :N], M, N, K, Q.SCALE_PER_MATRIX)
            assert Q.last_config().startswith(row), Q.last_config()
            assert np.array_equal(c[:, :N].float().cpu().numpy(), R.gemm_i8_i32(a, b).astype(np.float32)), N
            assert bool((c[:, N:] == 7).all()), N
    finally:
        Q.force_config(None)


@pytest.mark.parametrize("dtype", [torch.float8_e4m3fn, torch.int8, torch.bfloat16])
@pytest.mark.parametrize("shape, packed", [((16, 2048, 1036), False), ((2048, 2048, 4001), True)])
def test_the_way_that_is_estimated_faster(shape, packed, dtype):
    M, N, K = shape
    say("any shape, by the estimate", shape, dtype)
    rng = np.random.default_rng(K)
    a, b = _ints(rng, (M, K)), _ints(rng, (N, K))
    c = torch.zeros((M, N), dtype=torch.float32, device="cuda")
    Q.gemm(_tensor(a, dtype), _tensor(b, dtype), c)
    assert _ran(2 if packed else 0), Q.last_config()
    assert torch.equal(c.cpu(), torch.from_numpy(a) @ torch.from_numpy(b).t())
