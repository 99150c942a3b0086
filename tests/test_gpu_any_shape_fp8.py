"""fp8 operands on the any-shape path are summed in fp32: packed for the MFMA kernels (any_shape = 2) and on the any-shape
kernel (0)."""
import numpy as np
import pytest
import torch

import qgemm_amd as Q
from oracle import cpu_ref as R
from tests.util import dev, fp8_tensor, say, scalar

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[0, 2], ids=["any_shape_kernel", "packed"], autouse=True)
def _way(request):
    Q.set_option("any_shape", request.param)
    yield request.param
    Q.set_option("any_shape", 1)
    Q.set_option("force_split", 0)
    Q.force_config(None)


def _cancelling(M, N, K):
    """In every block of 128 elements of K one pair of products +448^2, -448^2 and small products, multiples of 1/32: the sum
    of the small ones, exactly.  fp32 holds every partial sum (18 bits above the point, 5 below; 2^-6 is its last bit beside
    448^2), in any order inside a block; a sum with fewer bits loses them."""
    rng = np.random.default_rng(M * N + K)
    a = rng.integers(-1, 2, (M, K)).astype(np.float32) / 8
    b = rng.integers(-1, 2, (N, K)).astype(np.float32) / 4
    for k0 in range(0, K - 1, 128):
        i, j = rng.choice(min(128, K - k0), 2, replace=False) + k0
        a[:, [i, j]] = 448
        b[:, i], b[:, j] = 448, -448
    small = np.abs(a) < 448
    ref = (a * small).astype(np.float64) @ (b * (np.abs(b) < 448)).astype(np.float64).T
    return fp8_tensor(R.encode_fp8(a)), fp8_tensor(R.encode_fp8(b)), torch.from_numpy(ref.astype(np.float32))


@pytest.mark.parametrize("out", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(5, 70, 129), (16, 200, 1001), (64, 700, 4097), (130, 300, 2001), (700, 520, 1025), (1100, 1030, 777)])
def test_no_bits_are_lost(shape, out, _way):
    M, N, K = shape
    say("fp8 any shape, cancelling products", shape, out)
    a, b, ref = _cancelling(M, N, K)
    ones = torch.ones(M, (K + 127) // 128, device="cuda"), torch.ones((N + 127) // 128, (K + 127) // 128, device="cuda")
    for mode, sa, sb in ((Q.SCALE_PER_MATRIX, scalar(1), scalar(1)), (Q.SCALE_BLOCK128, *ones)):
        for split in (1, 0):
            c = torch.full((M, N), 7.0, dtype=out, device="cuda")
            Q.scaled_gemm(a, b, sa, sb, c, M, N, K, mode, split_k=split)
            assert Q.last_config().startswith("pack+") == (_way == 2), Q.last_config()
            assert torch.equal(c.cpu(), ref.to(out)), (mode, split, Q.last_config())


def _rows():
    names = set()
    for mode in (Q.SCALE_PER_MATRIX, Q.SCALE_BLOCK128):
        names |= set(Q.variant_names(Q.DT_F8E4M3, mode, 0))
    return sorted(names)


@pytest.mark.parametrize("mode", [Q.SCALE_PER_MATRIX, Q.SCALE_BLOCK128])
def test_every_row(mode):
    """Every row by name (a row the widened family does not have leaves the call to the any-shape kernel)."""
    M, N, K = 270, 300, 1169
    a, b, ref = _cancelling(M, N, K)
    sa, sb = (scalar(1), scalar(1)) if mode == Q.SCALE_PER_MATRIX else \
        (torch.ones(M, (K + 127) // 128, device="cuda"), torch.ones((N + 127) // 128, (K + 127) // 128, device="cuda"))
    for row in _rows():
        say("fp8 any shape, row", row, mode)
        Q.force_config(row)
        for split in (1, 3):
            c = torch.zeros(M, N, device="cuda")
            Q.scaled_gemm(a, b, sa, sb, c, M, N, K, mode, split_k=split)
            assert torch.equal(c.cpu(), ref), (row, split)


@pytest.mark.parametrize("layout", ["nk", "kn"])
def test_every_code(layout):
    """One code a row times 1: the code's value, subnormals and NaNs among them."""
    codes = np.arange(256, dtype=np.uint8)
    M, N, K = 256, 90, 77
    say("fp8 any shape, every code", layout)
    a, b = np.zeros((M, K), np.uint8), np.zeros((N, K), np.uint8)
    a[codes, codes % K] = codes
    b[:] = R.encode_fp8(np.ones((N, K), np.float32)).view(np.uint8)
    bt = b if layout == "nk" else np.ascontiguousarray(b.T)
    c = torch.zeros(M, N, device="cuda")
    Q.gemm(fp8_tensor(a), fp8_tensor(bt), c, layout)
    want = np.repeat(R.decode_fp8(codes)[:, None], N, 1)
    assert np.array_equal(c.cpu().numpy(), want, equal_nan=True)
