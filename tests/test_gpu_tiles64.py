"""The 64 x 64 tile with two K groups (the reference's storage; 16-bit types with B stored K x N; rows of 9 .. 15 K steps): edges of
tiles, partial last K steps, more and fewer steps than stages, K splits and rows of any length; small integers and powers of two, exact.
An fp32 output that shows how its sums are made keeps the rows it had."""
import numpy as np
import pytest
import torch

import qgemm_amd as Q
from oracle import cpu_ref as R
from tests.util import dev, fp8_tensor, host, say

pytestmark = pytest.mark.gpu
ROW = "64x64_w2x2_k2"


@pytest.fixture
def row():
    Q.set_option("kmajor", 2)
    Q.force_config(ROW)
    yield
    Q.force_config(None)
    Q.set_option("kmajor", 1)
    Q.set_option("any_shape", 1)
    Q.set_option("force_split", 0)


@pytest.mark.parametrize("M", [32, 64, 160])
@pytest.mark.parametrize("N,K", [(32, 32), (64, 128), (96, 416), (224, 1056), (160, 2048)])
def test_reference_storage(M, N, K, row):
    rng = np.random.default_rng(M + N + K)
    KB, NB = (K + 127) // 128, (N + 127) // 128
    a, b = rng.integers(-4, 5, (M, K)).astype(np.float32), rng.integers(-4, 5, (N, K)).astype(np.float32)
    as_, bs = (2.0 ** rng.integers(-1, 2, (M, KB))).astype(np.float32), (2.0 ** rng.integers(-1, 2, (NB, KB))).astype(np.float32)
    ref = R.gemm_fp8_block(a, b, as_, bs)
    at, bt = (fp8_tensor(np.ascontiguousarray(R.encode_fp8(x).T)).t() for x in (a, b))
    sat, sbt = (dev(np.ascontiguousarray(x.T)).t() for x in (as_, bs))
    for split in (1, 3):
        say("64 x 64, both K-major", M, N, K, split)
        Q.set_option("force_split", split)
        c = torch.full((M, N), 7.0, dtype=torch.float32, device="cuda")
        Q.fp8_mm(at, bt, sat, sbt, c)
        assert Q.last_config().startswith(ROW + "_tn"), Q.last_config()
        assert np.array_equal(host(c), ref), (M, N, K, split)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (64, 64, 64), (65, 72, 200), (129, 136, 704), (200, 248, 2048), (65, 80, 203), (130, 56, 1053)])
def test_b_stored_k_by_n(dtype, M, N, K, row):
    rng = np.random.default_rng(M + N + K)
    a, b = rng.integers(-4, 5, (M, K)).astype(np.float32), rng.integers(-4, 5, (K, N)).astype(np.float32)
    ref = a @ b                                       # whole numbers below 2^24
    Q.set_option("any_shape", 3)
    whole = K % 8 == 0
    out = torch.float32 if whole else dtype           # (rows of any length come here only where the output hides the order of sums)
    want = torch.from_numpy(ref).to(out)
    for split in (1, 2) if whole else (1,):
        say("64 x 64, B stored K x N", dtype, M, N, K, split)
        Q.set_option("force_split", split)
        c = torch.full((M, N), 7.0, dtype=out, device="cuda")
        Q.gemm(dev(a).to(dtype), dev(b).to(dtype), c, "kn")
        assert ROW + "_nn" in Q.last_config(), Q.last_config()
        assert torch.equal(c.cpu(), want), (M, N, K, split)


@pytest.mark.parametrize("M,N,K", [(512, 688, 600), (64, 2816, 560), (256, 2176, 1080)])
def test_fp32_outputs_keep_their_rows(M, N, K):
    a, b = torch.ones(M, K, dtype=torch.bfloat16, device="cuda"), torch.ones(K, N, dtype=torch.bfloat16, device="cuda")
    for out, taken in ((torch.bfloat16, True), (torch.float32, False)):
        say("64 x 64 chosen", M, N, K, out)
        c = torch.empty(M, N, dtype=out, device="cuda")
        Q.gemm(a, b, c, "kn")
        assert Q.last_config().startswith(ROW) == taken, (out, Q.last_config())
        assert torch.equal(c, torch.full_like(c, K))


@pytest.mark.parametrize("dtype,mode", [("fp8", 1), ("fp8", 2), ("int8", 1), ("int8", 2)])
@pytest.mark.parametrize("M,N,K", [(401, 64, 1152), (448, 72, 1040), (1030, 960, 1920)])
def test_rows_of_k(dtype, mode, M, N, K):
    rng = np.random.default_rng(M + N + K)
    KB, NB = (K + 127) // 128, (N + 127) // 128
    a, b = rng.integers(-4, 5, (M, K)).astype(np.float32), rng.integers(-4, 5, (N, K)).astype(np.float32)
    as_, bs = [(2.0 ** rng.integers(-1, 2, s if mode == 2 else (1,))).astype(np.float32) for s in ((M, KB), (NB, KB))]
    wide = (lambda s, rows: np.repeat(s, 128, 1)[:, :K] if rows else np.repeat(np.repeat(s, 128, 0)[:N], 128, 1)[:, :K]) if mode == 2 else (lambda s, rows: s)
    want = torch.from_numpy((a * wide(as_, True)) @ (b * wide(bs, False)).T).to(torch.bfloat16)      # (exact before it is rounded)
    at, bt = (fp8_tensor(R.encode_fp8(x)) if dtype == "fp8" else dev(x.astype(np.int8)) for x in (a, b))
    say("64 x 64, rows of K", dtype, mode, M, N, K)
    c = torch.full((M, N), 7.0, dtype=torch.bfloat16, device="cuda")
    Q.scaled_gemm(at, bt, dev(as_), dev(bs), c, M, N, K, mode)
    assert Q.last_config() == ROW, Q.last_config()
    assert torch.equal(c.cpu(), want)
