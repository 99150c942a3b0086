"""The 64-row tile of the reference's storage (both operands K-major, block scales): k rows of 64 bytes two to an LDS row.  Around half a
tile of rows, partial column tiles and K steps, and K splits; small integers and powers of two, exact."""
import numpy as np
import pytest
import torch

import qgemm_amd as Q
from oracle import cpu_ref as R
from tests.util import dev, fp8_tensor, host, say

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _row():
    Q.set_option("kmajor", 2)
    Q.force_config("64x128_w1x4_k2")
    yield
    Q.force_config(None)
    Q.set_option("kmajor", 1)
    Q.set_option("force_split", 0)


@pytest.mark.parametrize("M", [32, 64, 96, 224])
@pytest.mark.parametrize("N,K", [(32, 32), (128, 128), (160, 416), (288, 1056)])
def test_rows_columns_and_steps(M, N, K):
    rng = np.random.default_rng(M + N + K)
    KB, NB = (K + 127) // 128, (N + 127) // 128
    a, b = rng.integers(-4, 5, (M, K)).astype(np.float32), rng.integers(-4, 5, (N, K)).astype(np.float32)
    as_, bs = (2.0 ** rng.integers(-1, 2, (M, KB))).astype(np.float32), (2.0 ** rng.integers(-1, 2, (NB, KB))).astype(np.float32)
    ref = R.gemm_fp8_block(a, b, as_, bs)
    at, bt = (fp8_tensor(np.ascontiguousarray(R.encode_fp8(x).T)).t() for x in (a, b))
    sat, sbt = (dev(np.ascontiguousarray(x.T)).t() for x in (as_, bs))
    for split in (1, 3):
        say("64 rows, K-major", M, N, K, split)
        Q.set_option("force_split", split)
        c = torch.full((M, N), 7.0, dtype=torch.float32, device="cuda")
        Q.fp8_mm(at, bt, sat, sbt, c)
        assert Q.last_config().startswith("64x128_w1x4_k2_tn"), Q.last_config()
        assert np.array_equal(host(c), ref), (M, N, K, split)
