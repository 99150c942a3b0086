"""The any-shape kernel (option any_shape = 0) where its loads, tiles and steps end: K up to and around a 16-byte piece, a step
and two steps, operands shorter than one piece, rows shorter than one, both tile sizes, rows of C with neighbours; and the choice between
the tiles and the kernel for few rows as it stands.  Small
integers (and block scales that are powers of two) sum exactly, so the results equal the CPU oracle's."""
import numpy as np
import pytest
import torch

import qgemm_amd as Q
from oracle import cpu_ref as R
from tests.util import dev, say

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True, params=[0, 1], ids=["tiles", "as_chosen"])
def _any_shape_kernel(request):
    Q.set_option("any_shape", 0)
    Q.set_option("few_rows", request.param)
    yield request.param
    Q.set_option("any_shape", 1)
    Q.set_option("few_rows", 1)


def _at_the_end(x, dtype):
    """x as the last elements of a buffer whose length is no multiple of anything."""
    t = torch.zeros(5 + x.size, dtype=dtype, device="cuda")[5:].view(x.shape)
    t.copy_(dev(x.astype(np.float32)).to(dtype))
    return t


def _operands(M, N, K):
    rng = np.random.default_rng(M + N + K)
    return rng.integers(-4, 5, (M, K)), rng.integers(-4, 5, (N, K))


# operands of one to 15 elements, rows of fewer than 16 bytes, K one off a piece, a step, two steps; 128 x 128 tiles
SHAPES = [(1, 1, 1), (3, 5, 2), (2, 700, 7), (1, 15, 15), (40, 3, 16), (17, 9, 17), (65, 63, 31), (64, 130, 63), (5, 66, 65),
          (70, 131, 127), (33, 2, 129), (129, 257, 255), (2, 3, 1009), (2100, 2050, 143)]


@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.int8, torch.float8_e4m3fn])
@pytest.mark.parametrize("shape", SHAPES)
def test_products(shape, dtype, layout, _any_shape_kernel):
    M, N, K = shape
    if _any_shape_kernel and M > 128:
        pytest.skip("tiles in either case")
    say("any-shape kernel", shape, dtype, layout)
    a, b = _operands(M, N, K)
    ref = torch.from_numpy(a.astype(np.float32)) @ torch.from_numpy(b.astype(np.float32)).t()
    c = torch.full((M, N + 3), 7.0, device="cuda")
    Q.gemm(_at_the_end(a, dtype), _at_the_end(b if layout == "nk" else np.ascontiguousarray(b.T), dtype), c[:, :N], layout)
    assert Q.last_config() == "strided_any_shape"
    assert _any_shape_kernel or Q.last_any_kernel().startswith("tiles" if K >= 16 else ("tiles", "short"))
    assert torch.equal(c[:, :N].cpu(), ref)
    assert bool((c[:, N:] == 7).all())


@pytest.mark.parametrize("dtype", [torch.int8, torch.float8_e4m3fn])
@pytest.mark.parametrize("shape", [(1, 1, 3), (3, 300, 15), (70, 140, 63), (33, 257, 129), (65, 129, 193), (40, 70, 257), (2100, 2050, 191)])
def test_block_scales(shape, dtype, _any_shape_kernel):
    M, N, K = shape
    if _any_shape_kernel and M > 128:
        pytest.skip("tiles in either case")
    say("any-shape kernel, block scales", shape, dtype)
    a, b = _operands(M, N, K)
    KB, rng = (K + 127) // 128, np.random.default_rng(K)
    as_ = (2.0 ** rng.integers(-1, 2, (M, KB))).astype(np.float32)
    bs = (2.0 ** rng.integers(-1, 2, ((N + 127) // 128, KB))).astype(np.float32)
    scaled = lambda x, s: torch.from_numpy(x * np.repeat(s, 128, 1)[:, :K]).float()  # noqa: E731
    ref = scaled(a, as_) @ scaled(b, np.repeat(bs, 128, 0)[:N]).t()
    c = torch.zeros(M, N, device="cuda")
    Q.scaled_gemm(_at_the_end(a, dtype), _at_the_end(b, dtype), dev(as_), dev(bs), c, M, N, K, Q.SCALE_BLOCK128)
    assert torch.equal(c.cpu(), ref)
    if dtype == torch.int8 and M < 100:
        assert torch.equal(c.cpu(), torch.from_numpy(R.gemm_i8_block(a.astype(np.int8), b.astype(np.int8), as_, bs)))


@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_sums_of_16_bit_operands(dtype, layout):
    """fp32 output: steps of 64 products are added to two fp32 sums in turn.  The 33 / 2 additions into a sum that grows like their
    square root, each rounded to half of 2^-23 and uniform, leave 2^-24 / sqrt(3) * sqrt(33 / 4) = 9.9e-8 of the result; a chain of
    matrix instructions over the same K leaves 2.7e-7."""
    M, N, K = 64, 300, 2060
    say("any-shape kernel, 16-bit operands to fp32", dtype, layout)
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    a, b = (torch.randn(r, K, generator=g, device="cuda").to(dtype) for r in (M, N))
    c = torch.zeros(M, N, device="cuda")
    Q.gemm(a, b if layout == "nk" else b.t().contiguous(), c, layout)
    assert Q.last_config() == "strided_any_shape"
    ref = a.double().cpu() @ b.double().cpu().t()
    assert float((c.double().cpu() - ref).norm() / ref.norm()) < 1.4e-7
