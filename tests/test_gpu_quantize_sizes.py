"""Quantisers at the sizes where another kernel takes over and where pieces of 16 bytes end inside a row: bytes and scales
against the CPU oracle, bit for bit."""
import numpy as np
import pytest
import torch

import qgemm_amd as Q
from oracle import cpu_ref as R
from tests.util import host, say

pytestmark = pytest.mark.gpu


def _u8(t):
    torch.cuda.synchronize()
    return t.view(torch.uint8).cpu().numpy()


def _input(rows, cols, dt, seed):
    x = torch.from_numpy(R.fill_normal((rows, cols), seed)).to(dt)
    return x.cuda(), x.float().numpy()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,cols", [(639, 2048), (640, 2048), (641, 2041), (1279, 1024), (5121, 255), (1, 129)])
def test_row_blocks_either_side_of_the_many_groups_rule(rows, cols, dt):
    say("quantize 1 x 128", rows, cols, dt)
    x, xf = _input(rows, cols, dt, 31)
    q, s = R.quantize_fp8_block(xf, 1, 128)
    g, gs = Q.quantize(x, torch.float8_e4m3fn, Q.QUANT_BLOCK_1x128)
    assert np.array_equal(host(gs), s) and np.array_equal(_u8(g), q)
