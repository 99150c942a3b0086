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


def test_a_reservation_serves_every_stream(host):
    """No call that needs no more than was reserved allocates, on whichever stream, also above what a stream has for itself."""
    host("""
need = 4 * 4096 * 4096 * 4                                      # planes of four K slices: 256 MiB
assert lib.qgemm_reserve_workspace(need) == 0
events()
for stream in (0, 64, 128, 192, 256, 2):                        # (2: hipStreamPerThread)
    for M, split in ((4096, 4), (192, 4), (4096, 2)):
        assert product(M, 4096, 2048, stream=stream, split=split) == 0 and "splitk%d" % split in config()
assert not any(e.startswith(("malloc", "synchronize")) for e in events())
lib.qgemm_shutdown()
runtime.host_budget(need)                                       # room for the reservation and nothing else
assert lib.qgemm_reserve_workspace(need) == 0
events()
for stream in (0, 64, 128, 192, 256, 2):
    assert product(4096, 4096, 2048, stream=stream, split=4) == 0 and product(192, 4096, 2048, stream=stream, split=4) == 0
assert not any(e.startswith(("malloc", "synchronize")) for e in events())
""")


def test_a_small_reservation(host):
    """It takes no more memory than it says, four times; a call that needs more allocates as if nothing had been reserved."""
    host("""
assert lib.qgemm_reserve_workspace(0) == 0 and events() == []
assert lib.qgemm_reserve_workspace(1 << 20) == 0 and events() == ["malloc 1048576"] * 4
assert product(32, 512, 2048, split=4) == 0 and "splitk4" in config() and all(e.startswith("launch") for e in events())
assert product(192, 4096, 2048, split=4) == 0
assert [e for e in events() if not e.startswith("launch")] == ["malloc %d" % (64 << 20), "malloc %d" % (128 << 20)]
assert lib.qgemm_reserve_workspace(1 << 20) == 0 and events() == []
assert product(192, 4096, 2048, split=4) == 0 and all(e.startswith("launch") for e in events())
""")


def test_whose_block(host):
    """Three streams have a block each and no events; further streams, hipStreamPerThread and calls beyond 128 MiB share one and wait for
    one another; captured calls touch no event."""
    host("""
def block(stream, M=192, split=4):
    assert product(M, 4096, 2048, stream=stream, split=split) == 0
    log = events()
    return [re.search("first (0x[0-9a-f]+)", e).group(1) for e in log if "splitk_reduce" in e][0], [e.split()[0] for e in log if e[:4] in ("wait", "reco")]
own = [block(s) for s in (0, 64, 128)]
shared = block(192)
assert len({b for b, _ in own} | {shared[0]}) == 4 and all(not e for _, e in own) and shared[1] == ["record"]
assert block(192) == (shared[0], ["record"]) and block(256) == (shared[0], ["wait", "record"])
assert block(2) == block(2) == (shared[0], ["wait", "record"])
assert [block(s) for s in (0, 64, 128)] == own
large = block(64, 4096)                                         # (the shared block grows)
assert large[1] == ["wait", "record"] and large[0] not in {b for b, _ in own} | {shared[0]}
assert block(192) == (large[0], ["wait", "record"])
runtime.host_capture(64, 1)
assert block(64) == (large[0], []) and block(64, 4096) == (large[0], [])
runtime.host_capture(64, 0)
assert block(64) == own[1]
""")


def test_without_memory_for_another_block(host):
    """A stream for which there is no block left uses the shared one, which is as large as any call has needed: nothing is waited for on
    the host, and no other stream's block is touched."""
    host("""
runtime.host_budget((64 + 128) << 20)
def call(stream, M=192):
    return product(M, 4096, 2048, stream=stream, split=4), [e.split()[0] for e in events() if not e.startswith("launch")]
assert call(0) == (0, ["malloc", "malloc"])
assert call(64) == (0, ["malloc", "record"])
assert call(64) == (0, ["record"]) and call(128) == (0, ["wait", "record"]) and call(0) == (0, [])
assert call(64, 4096) == (5, ["malloc"]) and call(0, 4096) == (5, ["malloc"])       # (more than the shared block, and none to be had)
assert call(64) == (0, ["wait", "record"])
lib.qgemm_shutdown()
runtime.host_budget(1 << 40)
assert call(64) == (0, ["synchronize", "malloc", "malloc"]) and call(64) == (0, [])
""")


def test_two_streams_exchange_maxima_at_a_time(host):
    """Quantisations whose workgroups wait for one another need room for all of them: two streams launch such kernels, others make two
    passes, until one of the two has not been seen for a while."""
    host("""
WHOLE, PASSES = ["quant_whole_matrix_kernel"], ["quant_amax_kernel", "quant_matrix_kernel"]
def way(stream, rows=2048):
    assert quantize(rows, 4096, stream=stream) == 0
    return kernels()
for _ in range(100):
    assert way(0) == way(64) == WHOLE and way(128) == way(192) == way(2) == PASSES
for _ in range(59):
    assert way(64) == WHOLE
assert way(128) == PASSES                                       # the 63rd call since stream 0's
assert way(128) == WHOLE and way(0) == PASSES and way(64) == WHOLE
assert way(0, 16) == way(128, 16) == ["quant_small_matrix_kernel"]
""")
    host("""
runtime.host_masked_cus(255)
assert quantize(2048, 4096) == 0 and kernels() == ["quant_amax_kernel", "quant_matrix_kernel"]
assert quantize(2048, 4096) == 0 and kernels() == ["quant_amax_kernel", "quant_matrix_kernel"]
runtime.host_masked_cus(0)
assert quantize(2048, 4096, stream=64) == 0 and kernels() == ["quant_whole_matrix_kernel"]
""")


def test_slices_that_the_caller_asks_for(host):
    """Rows that start or end anywhere, split_k = n: n slices wherever another kernel than the any-shape one runs, none while captured or
    on the static scratch, which launch nothing but the product."""
    host("""
import random
rng = random.Random(3)
ran = {"unaligned": 0, "pack": 0}
for i in range(1500):
    dt, mode, slices = rng.choice([I8, F8]), rng.choice([1, 2]), rng.choice([2, 3, 4])
    shape = [int(2 ** rng.uniform(0, 12)), int(2 ** rng.uniform(6, 13)), int(2 ** rng.uniform(7.1, 13))]
    a, b = (1 << 32) + rng.choice([0, 1, 4, 8]), (1 << 33) + rng.choice([0, 2, 16])
    call = dict(dt=dt, mode=mode, out=rng.choice([F32, BF16]), split=slices, a=a, b=b)
    assert product(*shape, **call) == 0
    way = config()
    if not way.startswith(("unaligned+", "pack+")):
        continue
    ran[way.split("+")[0]] += 1
    steps = (shape[2] + 127) // 128
    each = -(-steps // min(slices, steps))
    got = int(way.split("_splitk")[1]) if "_splitk" in way else 1
    assert got in (-(-steps // each), -(-(steps - 1) // -(-(steps - 1) // min(slices, steps - 1 or 1)))), (shape, call, way)
    events()
    runtime.host_capture(0, 1)
    assert product(*shape, **call) == 0 and "_splitk" not in config() and not config().startswith("pack+"), config()
    runtime.host_capture(0, 0)
    assert all(e.startswith("launch") for e in events())
    assert product(*shape, static=True, **call) == 0 and "_splitk" not in config() and not config().startswith("pack+"), config()
assert min(ran.values()) > 30, ran
option("force_split", 3)
found = 0
for i in range(300):
    assert product(rng.randrange(17, 129), rng.randrange(512, 8192), rng.randrange(1000, 8000), dt=I8, out=BF16) == 0
    if config().startswith("unaligned+"):
        found += 1
        assert config().endswith("_splitk3"), config()
assert found > 10
""")
