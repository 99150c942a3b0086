"""a_scale with the K blocks contiguous on the rows that fetch four blocks of a row per copy, with any number of blocks in a
row and in a slice.  Integer operands and power-of-two scales: every sum is exact, so the oracle's numbers are the bar."""
import numpy as np
import pytest
import torch

import qgemm_amd as Q
from oracle import cpu_ref as R
from tests.util import dev, fp8_tensor, say

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _reset_options():
    yield
    Q.force_config(None)
    Q.set_option("force_split", 0)
    Q.set_option("k_rot", -1)
    Q.set_option("as_groups", 1)


def _problem(M, N, K, seed):
    rng = np.random.default_rng(seed)
    a, b, KB = rng.integers(-3, 4, (M, K)).astype(np.float32), rng.integers(-3, 4, (N, K)).astype(np.float32), (K + 127) // 128
    as_ = (2.0 ** rng.integers(-2, 3, size=(M, KB))).astype(np.float32)
    bs = (2.0 ** rng.integers(-2, 3, size=((N + 127) // 128, KB))).astype(np.float32)
    return a, b, as_, bs


def _run(a, b, as_, bs, dtype, off=0):
    (M, K), N = a.shape, b.shape[0]
    conv = (lambda x: fp8_tensor(R.encode_fp8(x))) if dtype == torch.float8_e4m3fn else (lambda x: dev(x.astype(np.int8)))
    s = torch.zeros(as_.size + off, device="cuda")[off:].view(as_.shape)
    s.copy_(dev(as_))
    c = torch.zeros((M, N), dtype=torch.float32, device="cuda")
    Q.scaled_gemm(conv(a), conv(b), s, dev(bs), c, M, N, K, Q.SCALE_BLOCK128)
    return c.cpu().numpy()


@pytest.mark.parametrize("dtype", [torch.float8_e4m3fn, torch.int8])
@pytest.mark.parametrize("row", ["128x128_w2x2_k2", "64x128_w1x4_k2"])
@pytest.mark.parametrize("K", [128 * 5, 128 * 9 + 16, 128 * 14, 128 * 19 + 96])
def test_rows_with_two_k_groups(K, row, dtype):
    for M, N in ((150, 300), (300, 130)):                # (up to 256 rows the K loops start rotated where they may)
        p = _problem(M, N, K, seed=K + M)
        ref = R.gemm_fp8_block(*p)
        for split in (0, 1, 2, 3):
            for off in (0, 1):
                say("scale groups", row, (M, N, K), dtype, split, off)
                Q.force_config(row)
                Q.set_option("force_split", split)
                assert np.array_equal(_run(*p, dtype, off), ref)
        Q.set_option("k_rot", 3)                         # a rotation by other than whole groups: one block per copy
        assert np.array_equal(_run(*p, dtype), ref)
        Q.set_option("k_rot", -1)


@pytest.mark.parametrize("M, N, K", [(2048, 4096, 128 * 13), (2000, 4000, 128 * 14 + 32), (2048, 4096, 128 * 17), (2000, 4096, 128 * 11 + 16)])
def test_copying_waves(M, N, K):
    p = _problem(M, N, K, seed=K)
    say("scale groups, copying waves", (M, N, K))
    got = _run(*p, torch.float8_e4m3fn)
    assert Q.last_config() == "256x128_w2x2_cw_ks"
    rows = np.r_[0:70, M - 70:M]                         # (the oracle on the first and last rows)
    assert np.array_equal(got[rows], R.gemm_fp8_block(p[0][rows], p[1], p[2][rows], p[3]))


@pytest.mark.parametrize("dtype", [torch.float8_e4m3fn, torch.int8])
@pytest.mark.parametrize("K", [128 * 5, 128 * 9 + 16, 128 * 14, 128 * 19 + 96])
def test_copying_waves_pinned(K, dtype):
    """A row pinned by name reads the scales as the planner's choice does, also where K slices begin between groups of four
    blocks; as_groups = 0 takes the other row of the pair, on a transposed copy of a_scale."""
    M, N = 300, 200
    p = _problem(M, N, K, seed=K)
    ref = R.gemm_fp8_block(*p)
    for groups, name in ((1, "256x128_w2x2_cw_ks"), (0, "256x128_w2x2_cw")):
        for split in (1, 2, 3):
            for off in (0, 1):
                say("scale groups, copying waves, pinned", (M, N, K), dtype, groups, split, off)
                Q.force_config("256x128_w2x2_cw")
                Q.set_option("as_groups", groups)
                Q.set_option("force_split", split)
                assert np.array_equal(_run(*p, dtype, off), ref)
                assert Q.last_config() == name + (f"_splitk{split}" if split > 1 else "")
