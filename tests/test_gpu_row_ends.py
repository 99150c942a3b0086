"""Transposes and packing where rows end inside a piece: every remainder of 16 bytes, operands of fewer rows or elements than a
piece, addresses off its alignment.  Transposes move bytes; products of small integers are exact."""
import numpy as np
import pytest
import torch

import qgemm_amd as Q
from oracle import cpu_ref as R
from tests.util import dev, host, say

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _reset_options():
    yield
    Q.set_option("any_shape", 1)


@pytest.mark.parametrize("dt", [torch.int8, torch.bfloat16, torch.float32])
def test_transpose_at_every_remainder(dt):
    rng = np.random.default_rng(3)
    for M in (1, 3, 8, 17, 130):
        for N in (1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 31, 127, 129, 257):
            for off in (0, 1, 3):
                say("transpose", dt, M, N, off)
                flat = dev(rng.integers(-100, 100, size=M * N + 4).astype(np.float32)).to(dt)
                x = flat[off:off + M * N].view(M, N)
                out = torch.full((N, M), 77, dtype=dt, device="cuda")
                Q.matrix_transpose(x, out)
                assert torch.equal(out, x.t().contiguous()), (M, N, off)


@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("fam", ["i8", "bf16"])
def test_packed_products_at_every_remainder(fam, layout):
    rng = np.random.default_rng(5)
    Q.set_option("any_shape", 2)
    for M, N in ((1, 1), (3, 5), (70, 9), (33, 131)):
        for K in (1, 2, 3, 5, 7, 9, 15, 17, 31, 65, 127, 129, 255):
            say("packed", fam, layout, (M, N, K))
            a = rng.integers(-3, 4, size=(M, K)).astype(np.float32)
            b = rng.integers(-3, 4, size=(N, K)).astype(np.float32)
            c = torch.full((M, N), -7, dtype=torch.int32 if fam == "i8" else torch.float32, device="cuda")
            t = torch.int8 if fam == "i8" else torch.bfloat16
            qb = dev(b if layout == "nk" else np.ascontiguousarray(b.T)).to(t)
            Q.gemm(dev(a).to(t), qb, c, layout, ldA=K, ldB=K if layout == "nk" else N, ldC=N)
            assert np.array_equal(host(c), R.gemm_f32acc(a, b).astype(c.cpu().numpy().dtype)), (M, N, K)
