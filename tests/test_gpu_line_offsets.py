"""Operands whose rows start anywhere in a 128-byte cache line, on the rows with two K groups: there a copy fetches whole
lines and the chunks of a K step that lie in a row's second line arrive with the next stage (gemm_mfma.cuh).  Offsets of
the two operands apart from each other (none, the same, every multiple of 16 bytes by row), from one K step to past twice
the ring, whole and partial last steps, a start rotated over K, K slices; block scales below and from 32
steps on, where that form begins.  What lies beside the rows would show in any
sum; small integers sum exactly, so the results have to equal the CPU oracle bit for bit."""
import numpy as np
import pytest
import torch

import qgemm_amd as Q
from oracle import cpu_ref as R
from tests.util import dev, host, say

pytestmark = pytest.mark.gpu
ROWS = ["128x128_w2x2_k2", "64x128_w1x4_k2"]
# start of the first row and gap between rows, bytes past a 128-byte line, for A and for B
OFFSETS = [((0, 0), (16, 0)), ((112, 0), (0, 0)), ((0, 16), (0, 16)), ((48, 80), (96, 112)), ((64, 64), (0, 32))]


@pytest.fixture(autouse=True)
def _reset_options():
    yield
    Q.force_config(None)
    for k, v in (("force_split", 0), ("k_rot", -1)):
        Q.set_option(k, v)


def _placed(x, start, gap, fill):
    """x in a buffer of `fill`, its first row `start` bytes past a line, its rows `gap` bytes past a multiple of 128 apart."""
    rows, cols = x.shape
    es = x.element_size()
    pitch = (-(-cols * es // 128) * 128 + gap) // es if (cols * es) % 128 or gap else cols
    buf = torch.full((rows * pitch + 128,), fill, dtype=x.dtype, device="cuda")
    assert buf.data_ptr() % 128 == 0
    view = buf[start // es:start // es + rows * pitch].view(rows, pitch)[:, :cols]
    view.copy_(x)
    return view, pitch


@pytest.mark.parametrize("row", ROWS)
@pytest.mark.parametrize("fam", ["i8", "bf16"])
@pytest.mark.parametrize("offsets", OFFSETS, ids=str)
def test_rows_anywhere_in_a_line(row, fam, offsets):
    M, N = 139, 200                                          # ragged in both directions, several tiles
    rng = np.random.default_rng(5)
    lib = Q.load_library()
    for kbytes in (64, 128, 144, 256, 368, 640, 752, 1024, 1152, 1776):
        K = kbytes // (2 if fam == "bf16" else 1)
        for split, k_rot in ((1, 0), (1, 3)) + (((2, 0),) if kbytes >= 640 else ()):
            say("line offsets", row, fam, (M, N, K), offsets, "split", split, "k_rot", k_rot)
            a, b = rng.integers(-3, 4, size=(M, K)), rng.integers(-3, 4, size=(N, K))
            dt = torch.bfloat16 if fam == "bf16" else torch.int8
            av, lda = _placed(dev(a).to(dt), *offsets[0], fill=77)
            bv, ldb = _placed(dev(b).to(dt), *offsets[1], fill=77)
            c = torch.full((M, N), -7, dtype=torch.float32 if fam == "bf16" else torch.int32, device="cuda")
            Q.force_config(row)
            Q.set_option("force_split", split)
            Q.set_option("k_rot", k_rot)
            args = (Q.DT_BF16, Q.DT_F32) if fam == "bf16" else (Q.DT_I8, Q.DT_I32)
            assert lib.qgemm_gemm(*args, 1, av.data_ptr(), lda, bv.data_ptr(), ldb, c.data_ptr(), N, M, N, K, None) == 0
            assert Q.last_config().startswith(row), Q.last_config()
            ref = R.gemm_i8_i32(a.astype(np.int8), b.astype(np.int8))
            assert np.array_equal(host(c), ref), (kbytes, split, k_rot)


@pytest.mark.parametrize("row", ROWS)
@pytest.mark.parametrize("as_groups", [0, 1])
def test_block_scales(row, as_groups):
    M, N = 139, 200
    rng = np.random.default_rng(6)
    for start_a, start_b in ((16, 0), (0, 112), (48, 80)):
        for K in (128, 1168, 3968, 4096, 4112, 4224, 4896):
            KB = -(-K // 128)
            say("line offsets, block scales", row, (M, N, K), start_a, start_b)
            a, b = (rng.integers(-3, 4, size=s).astype(np.float32) for s in ((M, K), (N, K)))
            as_ = (2.0 ** rng.integers(-3, 4, size=(M, KB))).astype(np.float32)
            bs = (2.0 ** rng.integers(-3, 4, size=(-(-N // 128), KB))).astype(np.float32)
            place = lambda q, start: torch.cat([torch.full((start,), 0x78, dtype=torch.uint8, device="cuda"),  # noqa: E731
                                                dev(q).flatten()])[start:].view(q.shape).view(torch.float8_e4m3fn)
            c = torch.full((M, N), -7.0, dtype=torch.float32, device="cuda")
            Q.force_config(row)
            Q.set_option("force_split", 1)
            Q.set_option("as_groups", as_groups)
            try:
                Q.scaled_gemm(place(R.encode_fp8(a), start_a), place(R.encode_fp8(b), start_b), dev(as_), dev(bs), c, M, N, K,
                              Q.SCALE_BLOCK128)
                assert Q.last_config().startswith(row), Q.last_config()
                assert np.array_equal(host(c), R.gemm_fp8_block(a, b, as_, bs)), (K, start_a, start_b)
            finally:
                Q.set_option("as_groups", 1)
