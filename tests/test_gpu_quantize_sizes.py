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


def _strided(x, gap):
    base = torch.zeros((x.shape[0], x.shape[1] + gap), dtype=x.dtype, device="cuda")
    base[:, gap:] = x
    return base[:, gap:]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,cols", [(1, 1), (5, 3), (3, 7), (129, 5), (2, 8), (16, 2045), (64, 2048), (64, 2049), (33, 1985), (260, 1027), (70, 4100), (16384, 1), (16385, 1), (32, 300), (33, 300), (8192, 8), (8193, 8), (8193, 9), (40, 2176)])
def test_every_mode_at_row_ends_and_either_side_of_the_small_matrix(rows, cols, dt):
    """64 x 2048 16-bit elements are the last small matrix, and 16384 rows of a piece or less in a capture (8192 outside one) where there is a gap between them, 32 rows the last low block; rows that end 1 .. 7 elements into a piece, shorter than one, with and
    without a gap between them; the largest element last."""
    say("quantize sizes", rows, cols, dt)
    x, xf = _input(rows, cols, dt, 33)
    x[-1, -1] = 9.0
    xf = x.float().cpu().numpy()
    for t in (x, _strided(x, 1), _strided(x, 3)):
        for qt, ref, block in ((torch.int8, R.quantize_int8, R.quantize_int8_block), (torch.float8_e4m3fn, R.quantize_fp8, R.quantize_fp8_block)):
            q, s = ref(xf)
            g, gs = Q.quantize(t, qt, Q.QUANT_PER_MATRIX)
            assert host(gs)[0] == s and np.array_equal(_u8(g), q.view(np.uint8)), (rows, cols, qt)
            for mode, br in ((Q.QUANT_BLOCK_1x128, 1), (Q.QUANT_BLOCK_128x128, 128)):
                q, s = block(xf, br, 128)
                g, gs = Q.quantize(t, qt, mode)
                assert np.array_equal(host(gs), s) and np.array_equal(_u8(g), q.view(np.uint8)), (rows, cols, qt, mode)


def test_rows_with_gaps_in_a_capture():
    """Between 128 and 256 KiB: two passes and the workspace outside a capture, one launch without it inside."""
    x, xf = _input(10000, 8, torch.bfloat16, 37)
    t = _strided(x, 3)
    ref_q, ref_s = R.quantize_int8(xf)
    for eager in (True, False):
        say("quantize with gaps", "eager" if eager else "captured")
        if eager:
            g, gs = Q.quantize(t, torch.int8, Q.QUANT_PER_MATRIX)
        else:
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                g, gs = Q.quantize(t, torch.int8, Q.QUANT_PER_MATRIX)
        for _ in range(1 if eager else 3):
            if not eager:
                g.zero_()
                gs.zero_()
                graph.replay()
            assert host(gs)[0] == ref_s and np.array_equal(_u8(g), ref_q.view(np.uint8))


@pytest.mark.parametrize("rows,cols", [(9, 517), (300, 1031), (3, 20), (40, 1024), (1, 5)])
@pytest.mark.parametrize("special", [float("nan"), float("inf"), -float("inf")])
def test_special_values_wherever_they_stand(rows, cols, special):
    """One NaN or infinity, in the last piece of a row and in the middle of one: the maximum is that of the numbers (infinity
    counts as one), every other element keeps its bytes, for the single launch as for the two passes."""
    x, _ = _input(rows, cols, torch.bfloat16, 35)
    for at in ((rows - 1, cols - 1), (rows // 2, min(128, cols - 1)), (0, 3)):
        say("quantize special", rows, cols, special, at)
        y = x.clone()
        y[at] = special
        yf = y.float().cpu().numpy()
        q, s = R.quantize_fp8(yf)
        g, gs = Q.quantize(y, torch.float8_e4m3fn, Q.QUANT_PER_MATRIX)
        assert np.array_equal(host(gs).view(np.uint32), np.array([s]).view(np.uint32)) and np.array_equal(_u8(g), q), at
        q, s = R.quantize_fp8_block(yf, 128, 128)
        g, gs = Q.quantize(y, torch.float8_e4m3fn, Q.QUANT_BLOCK_128x128)
        assert np.array_equal(host(gs).view(np.uint32), s.view(np.uint32)) and np.array_equal(_u8(g), q), at


def test_more_row_blocks_than_a_launch_has_threads_for():
    """2^27 blocks of fp32 are 2^32 threads: a second slice of rows takes what the first cannot."""
    rows, cols, lead = 1 << 27, 16, 1 << 20
    say("quantize 1 x 128", rows, cols, "float32")
    x = torch.empty((rows, cols), dtype=torch.float32, device="cuda")
    head = torch.from_numpy(R.fill_normal((lead, cols), 9)).cuda()
    x.view(rows // lead, lead, cols).copy_(head)                    # the same rows over and over
    q, s = Q.quantize(x, torch.float8_e4m3fn, Q.QUANT_BLOCK_1x128)
    del x
    want_q, want_s = Q.quantize(head, torch.float8_e4m3fn, Q.QUANT_BLOCK_1x128)
    assert torch.equal(s.view(rows // lead, lead, 1), want_s.expand(rows // lead, lead, 1))
    assert torch.equal(q.view(torch.uint8).view(rows // lead, lead, cols), want_q.view(torch.uint8).expand(rows // lead, lead, cols))
    del q, s
    torch.cuda.empty_cache()
