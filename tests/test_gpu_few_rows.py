"""The any-shape kernel for few rows: operands at any address and distance, 1 .. 128 rows, K from a few elements past one piece to
several turns of the eight waves with every kind of end, columns that end inside a strip; captured and eager.  Small integers (and
power-of-two scales) sum exactly, so the results equal the oracle's bit for bit."""
import numpy as np
import pytest
import torch

import qgemm_amd as Q
from oracle import cpu_ref as R
from tests.util import dev, host, say

pytestmark = pytest.mark.gpu
TYPES = {"i8": torch.int8, "i8_block": torch.int8, "f8": torch.float8_e4m3fn, "f8_block": torch.float8_e4m3fn, "bf16": torch.bfloat16, "f16": torch.float16}


@pytest.fixture(autouse=True)
def _reset_options():
    Q.set_option("any_shape", 0)
    Q.set_option("few_rows", 2)
    yield
    Q.set_option("any_shape", 1)
    Q.set_option("few_rows", 1)


def _ran_for_few_rows(M):
    return Q.last_config() == "strided_any_shape" and Q.last_any_kernel() == ("few_rows_16x32" if M <= 16 else "few_rows_32x32")


def _operand(x, dt, shift):
    """x in a buffer that starts `shift` elements in, rows without a gap."""
    flat = torch.zeros(x.size + shift, dtype=dt, device="cuda")
    flat[shift:] = dev(x.reshape(-1)).to(dt)
    return flat[shift:].view(x.shape)


@pytest.mark.parametrize("fam", sorted(TYPES))
@pytest.mark.parametrize("M,N", [(1, 1), (3, 33), (16, 100), (17, 31), (33, 65), (64, 200), (128, 40)])
def test_every_end_of_k(fam, M, N):
    rng = np.random.default_rng(M * 1000 + N)
    dt, block = TYPES[fam], fam.endswith("block")
    for K in (17, 31, 127, 129, 250, 641, 1025, 1153, 2051, 3333):
        shift = K % 4
        say("few rows", fam, (M, N, K), "shift", shift)
        a = rng.integers(-3, 4, size=(M, K)).astype(np.float32)
        b = rng.integers(-3, 4, size=(N, K)).astype(np.float32)
        qa, qb = _operand(a, dt, shift), _operand(b, dt, shift)
        ref = R.gemm_f32acc(a, b)
        c = torch.full((M, N), -7, dtype=torch.bfloat16 if fam in ("bf16", "f16") or block else (torch.int32 if fam == "i8" else torch.float32), device="cuda")
        if block:
            kb = (K + 127) // 128
            as_ = (2.0 ** rng.integers(-3, 4, size=(M, kb))).astype(np.float32)
            bs = (2.0 ** rng.integers(-3, 4, size=((N + 127) // 128, kb))).astype(np.float32)
            if fam == "i8_block":
                ref = R.gemm_i8_block(a.astype(np.int8), b.astype(np.int8), as_, bs)
            else:
                ref = R.gemm_fp8_block(a, b, as_, bs)
            run = lambda: Q.scaled_gemm(qa, qb, dev_as, dev_bs, c, M, N, K, Q.SCALE_BLOCK128)
            dev_as, dev_bs = dev(as_), dev(bs)
        elif fam in ("bf16", "f16"):
            run = lambda: Q.gemm(qa, qb, c, "nk", ldA=K, ldB=K, ldC=N)
        else:
            one = dev(np.ones(1, np.float32))
            run = lambda: Q.scaled_gemm(qa, qb, one, one, c, M, N, K, Q.SCALE_PER_MATRIX)
        run()
        assert _ran_for_few_rows(M), (Q.last_config(), Q.last_any_kernel())
        want = torch.from_numpy(np.ascontiguousarray(ref, dtype=np.float32)).to(c.dtype if c.dtype != torch.int32 else torch.float32)
        got = c.cpu()
        assert torch.equal(got.to(want.dtype), want), (fam, M, N, K)


@pytest.mark.parametrize("dt", [torch.int8, torch.float8_e4m3fn])
@pytest.mark.parametrize("M,N,K", [(1, 33, 3000), (16, 100, 3001), (17, 200, 3199), (64, 31, 3333), (128, 140, 4097)])
def test_block_scales_to_fp32(dt, M, N, K):
    """From 3000 elements of K on (below, the tiles' sums are closer to 64 bits).  Products of small integers and powers of two within
    2^24 units: every order of the sums gives the same fp32."""
    say("few rows, block scales to fp32", dt, (M, N, K))
    rng, kb = np.random.default_rng(K), (K + 127) // 128
    a, b = rng.integers(-3, 4, size=(M, K)), rng.integers(-3, 4, size=(N, K))
    as_, bs = ((2.0 ** rng.integers(-3, 4, size=(r, kb))).astype(np.float32) for r in (M, (N + 127) // 128))
    c = torch.full((M, N), -7.0, device="cuda")
    run = lambda: Q.scaled_gemm(_operand(a.astype(np.float32), dt, 3), _operand(b.astype(np.float32), dt, 1), dev(as_), dev(bs), c, M, N, K,  # noqa: E731
                                Q.SCALE_BLOCK128)
    run()
    assert _ran_for_few_rows(M), Q.last_any_kernel()
    scaled = lambda x, s: x * np.repeat(s.astype(np.float64), 128, 1)[:, :K]  # noqa: E731
    want = torch.from_numpy((scaled(a, as_) @ scaled(b, np.repeat(bs, 128, 0)[:N]).T).astype(np.float32))
    assert torch.equal(c.cpu(), want)
    Q.set_option("few_rows", 0)
    c.fill_(-7)
    run()
    assert Q.last_any_kernel().startswith("tiles") and torch.equal(c.cpu(), want)


def test_where_it_does_not_run():
    """Sums that the output would show to be less exact, more rows than 128, and B stored K x N, keep the tiles."""
    def ran(M, N, K, dt, out, layout="nk"):
        a, b = torch.ones(M, K, device="cuda").to(dt), torch.ones(*((N, K) if layout == "nk" else (K, N)), device="cuda").to(dt)
        Q.gemm(a, b, torch.empty(M, N, dtype=out, device="cuda"), layout)
        return Q.last_any_kernel()

    bf16, fp32 = torch.bfloat16, torch.float32
    assert ran(8, 40, 1001, bf16, bf16) == "few_rows_16x32" and ran(128, 40, 1001, bf16, bf16) == "few_rows_32x32"
    assert ran(8, 40, 1001, bf16, fp32) == "tiles_64x64"
    assert ran(129, 40, 1001, bf16, bf16) == "tiles_64x64"
    assert ran(8, 41, 1001, bf16, bf16, "kn") == "tiles_64x64"
    assert ran(8, 40, 7, bf16, bf16) == "short"


def test_special_values_stay_in_their_rows():
    """What lies behind a row's last element is the next row: a NaN or an infinity there must not reach the sums of this one."""
    M, N, K = 5, 40, 1001
    rng = np.random.default_rng(1)
    a = rng.integers(-3, 4, size=(M, K)).astype(np.float32)
    b = rng.integers(-3, 4, size=(N, K)).astype(np.float32)
    a[3, :8] = np.nan
    b[20, :8] = np.inf
    qa, qb = _operand(a, torch.bfloat16, 1), _operand(b, torch.bfloat16, 1)
    c = torch.zeros((M, N), dtype=torch.bfloat16, device="cuda")
    g = torch.cuda.CUDAGraph()
    Q.gemm(qa, qb, c, "nk")
    assert _ran_for_few_rows(M)
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        Q.gemm(qa, qb, c, "nk")
    keep_m, keep_n = [0, 1, 2, 4], [i for i in range(N) if i != 20]
    want = torch.from_numpy(R.gemm_f32acc(a[keep_m], b[keep_n])).bfloat16()
    for _ in range(3):
        c.zero_()
        g.replay()
        torch.cuda.synchronize()
        got = c.cpu()
        assert torch.equal(got[keep_m][:, keep_n], want)
        assert torch.isnan(got[3]).all() and not torch.isfinite(got[0, 20])


def test_more_columns_than_a_launch_has_threads_for():
    """2^28 columns would be 2^32 threads of the kernel for few rows: the tiles take them."""
    N, K, lead = 1 << 28, 129, 1 << 16
    say("few rows", (1, N, K), "69 GB of B")
    rng = np.random.default_rng(4)
    a = rng.integers(-3, 4, size=(1, K)).astype(np.float32)
    b = rng.integers(-3, 4, size=(lead, K)).astype(np.float32)
    torch.cuda.empty_cache()
    qb = torch.empty((N, K), dtype=torch.bfloat16, device="cuda")
    qb.view(N // lead, lead, K).copy_(dev(b).bfloat16())             # the same rows over and over
    c = torch.full((1, N), -7.0, dtype=torch.bfloat16, device="cuda")
    Q.gemm(dev(a).bfloat16(), qb, c, "nk")
    assert Q.last_any_kernel() == "tiles_128x128"
    want = torch.from_numpy(R.gemm_f32acc(a, b)).bfloat16().cuda()
    assert torch.equal(c.view(N // lead, lead), want.expand(N // lead, lead))
    del qb, c
    torch.cuda.empty_cache()
