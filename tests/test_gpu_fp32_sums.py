"""fp32 outputs of few rows against 64-bit sums: the estimate that picks a row up to 400 rows must not trade the eight short chains
of the skinny-M kernel for one long one, which an fp32 output shows (16-bit ones do not)."""
import math

import pytest
import torch

import qgemm_amd as Q
from tests.util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(8, 8788, 544), (1, 8336, 1040), (2, 12720, 576), (56, 1867, 1648), (109, 816, 1824)])
def test_sums_in_eight_parts_or_more(shape, dtype):
    """n additions into a sum that grows like their square root, each rounded to half of 2^-23 and uniform, leave
    2^-24 / sqrt(3) * sqrt(n / 2) of the result.  A matrix instruction of 32 products rounds twice.  Eight parts: K / 32 / 8 instructions
    each, K / 128 additions in all parts together, then the parts themselves meet in seven additions.  A quarter is left for fp16, whose
    products carry three bits more.  (One chain of K / 16 additions leaves 1.2 to 2.1 times the bound.)"""
    M, N, K = shape
    say("fp32 sums", shape, dtype)
    g = torch.Generator(device="cuda")
    g.manual_seed(M)
    a, b = (torch.randn(r, K, generator=g, device="cuda").to(dtype) for r in (M, N))
    c = torch.zeros(M, N, device="cuda")
    Q.gemm(a, b, c, "nk")
    ref = a.double().cpu() @ b.double().cpu().t()
    err = float((c.double().cpu() - ref).norm() / ref.norm())
    print(Q.last_config(), err)
    assert err < 1.25 * 2.0 ** -24 / math.sqrt(3) * math.sqrt(K / 128 / 2 + 7 / 2), (Q.last_config(), err)


@pytest.mark.parametrize("shape", [(51, 616, 7907), (47, 344, 6287), (40, 480, 7001)])
@pytest.mark.parametrize("block", [False, True])
def test_ragged_fp8_sums_as_it_does_packed(shape, block):
    """Packed rows with a K split sum in more parts than the kernel for few rows, which an fp32 output shows: the faster kernel is for
    outputs that hide it."""
    M, N, K = shape
    say("ragged fp8 to fp32", shape, "block scales" if block else "one scale")
    g = torch.Generator(device="cuda")
    g.manual_seed(N)
    a, b = ((60 * torch.randn(r, K, generator=g, device="cuda")).to(torch.float8_e4m3fn) for r in (M, N))
    kb = (K + 127) // 128 if block else 1
    sa, sb = torch.rand(M if block else 1, kb, generator=g, device="cuda"), torch.rand((N + 127) // 128 if block else 1, kb, generator=g, device="cuda")

    def run(dtype, any_shape):
        Q.set_option("any_shape", any_shape)
        try:
            c = torch.zeros(M, N, device="cuda", dtype=dtype)
            Q.scaled_gemm(a, b, sa, sb, c, M, N, K, Q.SCALE_BLOCK128 if block else Q.SCALE_PER_MATRIX)
            return c, Q.last_config()
        finally:
            Q.set_option("any_shape", 1)

    packed, row = run(torch.float32, 2)
    assert row.startswith("pack+") and "_splitk" in row, row
    c, name = run(torch.float32, 1)
    assert name == row and torch.equal(c, packed)
    assert run(torch.bfloat16, 1)[1] == "strided_any_shape"
