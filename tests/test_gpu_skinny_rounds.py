"""Block scales on the tall rows of the skinny-M kernel by K steps: one round of the eight waves and less, two, the last count whose first
round asks for its scales behind A and the first that asks in front, more; whole and partial last steps; scales with the rows or the K
blocks contiguous.  Small integers and power-of-two scales sum exactly, so the result is that of 64 bits."""
import numpy as np
import pytest
import torch

import qgemm_amd as Q
from tests.util import dev, say

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _heuristic_again():
    yield
    Q.force_config(None)


@pytest.mark.parametrize("steps", [1, 8, 9, 16, 17, 32, 33, 36, 37, 48, 49, 65])
@pytest.mark.parametrize("dt", [torch.int8, torch.float8_e4m3fn])
@pytest.mark.parametrize("row,M,N", [("skinny_64x32_k8", 33, 48), ("skinny_64x32_k8", 130, 160), ("skinny_128x32_k8", 128, 32), ("skinny_64x64_k8", 65, 144)])
def test_block_scales_by_k_steps(row, M, N, dt, steps):
    for K in (128 * steps, 128 * steps - 48):
        say(row, dt, (M, N, K))
        rng, kb = np.random.default_rng(K + M), (K + 127) // 128
        a, b = rng.integers(-3, 4, (M, K)), rng.integers(-3, 4, (N, K))
        as_, bs = ((2.0 ** rng.integers(-2, 3, (r, kb))).astype(np.float32) for r in (M, (N + 127) // 128))
        scaled = lambda x, s: x * np.repeat(s.astype(np.float64), 128, 1)[:, :K]  # noqa: E731
        want = torch.from_numpy((scaled(a, as_) @ scaled(b, np.repeat(bs, 128, 0)[:N]).T).astype(np.float32))
        qa, qb = (dev(x.astype(np.float32)).to(dt) for x in (a, b))
        c = torch.full((M, N), -7.0, device="cuda")
        Q.force_config(row)
        Q.scaled_gemm(qa, qb, dev(as_), dev(bs), c, M, N, K, Q.SCALE_BLOCK128)
        assert Q.last_config().startswith(row), Q.last_config()
        assert torch.equal(c.cpu(), want), (row, M, N, K)
