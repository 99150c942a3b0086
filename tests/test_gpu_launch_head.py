"""What the kernels derive from a launch's leading arguments: the K slice (the last one shorter than the others), the rotated
start inside it, the tile (groups of row tiles, the last one shorter).  Small integers and power-of-two scales sum exactly, so
a slice, a start or a tile that is off by one cannot hide."""
import numpy as np
import pytest
import torch

import qgemm_amd as Q
from oracle import cpu_ref as R
from tests.util import dev, fp8_tensor, host, say

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _reset_options():
    yield
    for k, v in (("force_config", -1), ("force_split", 0), ("k_rot", -1), ("group_m", 0)):
        Q.set_option(k, v)


@pytest.mark.parametrize("row", ["skinny_16x32_k8", "skinny_32x16_k8", "skinny_64x64_k8", "skinny_128x32_k8", "64x128_w1x4_k2",
                                 "64x128_w1x4_dma", "128x128_w2x2_dma"])
def test_uneven_slices_rotated_starts_and_short_groups(row):
    M, N = (200, 700) if "64x" in row or "128x" in row else (40, 700)
    Q.force_config(row)
    for ksteps, split, k_rot, group in ((1, 1, 3, 0), (7, 1, 3, 2), (9, 2, 3, 1), (17, 4, 5, 3), (19, 8, 0, 0), (33, 3, 40, 5)):
        K = 128 * ksteps - 16 * (ksteps % 3)
        say("launch head", row, (M, N, K), "split", split, "k_rot", k_rot, "group", group)
        Q.set_option("force_split", split)
        Q.set_option("k_rot", k_rot)
        Q.set_option("group_m", group)
        rng = np.random.default_rng(ksteps)
        a = rng.integers(-3, 4, size=(M, K)).astype(np.float32)
        b = rng.integers(-3, 4, size=(N, K)).astype(np.float32)
        as_ = (2.0 ** rng.integers(-3, 4, size=(M, ksteps))).astype(np.float32)
        bs = (2.0 ** rng.integers(-3, 4, size=((N + 127) // 128, ksteps))).astype(np.float32)
        qa, qb = fp8_tensor(R.encode_fp8(a)), fp8_tensor(R.encode_fp8(b))
        c = torch.full((M, N), -7.0, dtype=torch.float32, device="cuda")
        Q.scaled_gemm(qa, qb, dev(as_), dev(bs), c, M, N, K, Q.SCALE_BLOCK128)
        assert Q.last_config().startswith(row), Q.last_config()
        assert np.array_equal(host(c), R.gemm_fp8_block(a, b, as_, bs)), (row, ksteps, split, k_rot, group)
        c.fill_(-7.0)
        Q.scaled_gemm(qa, qb, dev(np.array([0.5], np.float32)), dev(np.array([4.0], np.float32)), c, M, N, K, Q.SCALE_PER_MATRIX)
        assert np.array_equal(host(c), 2.0 * R.gemm_f32acc(a, b)), (row, ksteps, split, k_rot, group)


@pytest.mark.parametrize("row", ["64x128_w1x4_k2", "128x128_w2x2_k2", "skinny_64x64_k8", "64x128_w1x4_dma"])
def test_starts_further_in_than_the_leading_arguments_hold(row):
    """13 bits of the head are the rotated start.  Values beyond them have to be brought down before it is decided whether the
    K-group rows copy a_scale four K blocks at a time, which takes starts at multiples of four: a cut to 8191 after that
    starts 42 of 56 column tiles off a group."""
    M, N = 200, 1100
    Q.force_config(row)
    for ksteps, split, k_rot in ((16, 1, 8192), (20, 1, 8200), (40, 5, 1 << 20), (17, 2, 8195), (33, 4, 1 << 31)):
        K = 128 * ksteps
        say("launch head", row, (M, N, K), "split", split, "k_rot", k_rot)
        Q.set_option("force_split", split)
        Q.set_option("k_rot", k_rot)
        rng = np.random.default_rng(ksteps)
        a = rng.integers(-3, 4, size=(M, K)).astype(np.float32)
        b = rng.integers(-3, 4, size=(N, K)).astype(np.float32)
        as_ = (2.0 ** rng.integers(-3, 4, size=(M, ksteps))).astype(np.float32)
        bs = (2.0 ** rng.integers(-3, 4, size=((N + 127) // 128, ksteps))).astype(np.float32)
        c = torch.full((M, N), -7.0, dtype=torch.float32, device="cuda")
        Q.scaled_gemm(fp8_tensor(R.encode_fp8(a)), fp8_tensor(R.encode_fp8(b)), dev(as_), dev(bs), c, M, N, K, Q.SCALE_BLOCK128)
        assert Q.last_config().startswith(row), Q.last_config()
        assert np.array_equal(host(c), R.gemm_fp8_block(a, b, as_, bs)), (row, ksteps, split, k_rot)


def test_groups_of_more_row_tiles_than_the_leading_arguments_hold():
    """16 bits of the head are the row tiles of a group: above, the group and its inverses have to be cut together."""
    M, N, K = 16 * 70000 + 3, 300, 48
    say("launch head", (M, N, K), "70001 row tiles")
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    a = torch.randint(-3, 4, (M, K), generator=g, device="cuda", dtype=torch.int8)
    b = torch.randint(-3, 4, (N, K), generator=g, device="cuda", dtype=torch.int8)
    one = dev(np.ones(1, np.float32))
    want = (a.float() @ b.float().t()).bfloat16()                     # (sums below 433: exact in float, rounded once)
    Q.force_config("16x128_w1x2_dma")
    for group in (70000, 65536, 65535, 1 << 40):
        Q.set_option("group_m", group)
        c = torch.full((M, N), -7.0, dtype=torch.bfloat16, device="cuda")
        Q.scaled_gemm(a, b, one, one, c, M, N, K, Q.SCALE_PER_MATRIX)
        assert Q.last_config() == "16x128_w1x2_dma"
        assert torch.equal(c, want), group
