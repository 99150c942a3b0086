"""The workspace and who uses which part of it, on the host: statuses, allocations, events and launches of calls on several
streams, captured or not, with memory and without (tests/host_runtime.py: no kernel runs)."""
import pytest

from tests import host_runtime


@pytest.fixture
def host(tmp_path_factory):
    return lambda script: host_runtime.run(tmp_path_factory, script)


def test_an_eager_quantisation_leaves_room_for_a_captured_one(host):
    """Per-matrix scales, matrices without gaps: one launch without workspace, two passes with it while captured.  Nothing else has
    used the workspace."""
    host("""
for rows, cols in ((129, 1024), (500, 1000), (4096, 4096)):
    lib.qgemm_shutdown()
    runtime.host_capture(64, 1)
    assert quantize(rows, cols, stream=64) == 5                 # (nobody has run the shape)
    assert quantize(rows, cols) == 0 and kernels() == ["quant_whole_matrix_kernel"]
    assert quantize(rows, cols, stream=64) == 0
    assert kernels() == ["quant_amax_kernel", "quant_matrix_kernel"]
    assert quantize(rows, cols) == 0 and not any("malloc" in e for e in events())
runtime.host_budget(0)                                          # without memory the one launch runs all the same
lib.qgemm_shutdown()
assert quantize(500, 1000) == 0 and quantize(500, 1000, stream=64) == 5
""")
