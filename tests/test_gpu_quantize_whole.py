"""Per-matrix quantisation in one launch, whose workgroups exchange their maxima: at the sizes where a lane holds one piece more
and where the launch gives way to others, against the CPU oracle bit for bit; also where the workgroups do not wait for one
another (each then takes the maximum of the whole matrix), and on several streams at once."""
import time

import numpy as np
import pytest
import torch

import qgemm_amd as Q
from oracle import cpu_ref as R
from qgemm_amd import lib as L
from tests.util import host, say

pytestmark = pytest.mark.gpu

LANES = 256 * 1024


@pytest.fixture(autouse=True)
def _reset_options():
    yield
    Q.set_option("quant_wait", -2)


def _check(x, xf):
    for qt, ref in ((torch.int8, R.quantize_int8), (torch.float8_e4m3fn, R.quantize_fp8)):
        q, s = ref(xf)
        for wait in (2000, 0, -1):
            Q.set_option("quant_wait", wait)
            g, gs = Q.quantize(x, qt, Q.QUANT_PER_MATRIX)
            assert host(gs).view(np.uint32)[0] == np.array([s], np.float32).view(np.uint32)[0], (qt, wait)
            assert np.array_equal(g.view(torch.uint8).cpu().numpy(), q.view(np.uint8)), (qt, wait)


@pytest.mark.parametrize("dt,vec", [(torch.bfloat16, 8), (torch.float16, 8), (torch.float32, 4)])
@pytest.mark.parametrize("elements", ["small", "first", "groups", 1, 2, 4, 8])
def test_either_side_of_every_form(dt, vec, elements):
    """`small`: the last matrix whose maximum every workgroup takes by itself; `groups`: the first that needs all workgroups; n: the
    last of n pieces a lane."""
    at = {"small": 16384 * vec, "first": 17 * 1024 * vec, "groups": (LANES - 1024) * vec}.get(elements) or elements * LANES * vec
    for n in (at - 1, at, at + 1, at + vec):
        say("quantize whole", dt, n)
        x = torch.from_numpy(R.fill_normal((1, n), 71)).to(dt).cuda()
        x[0, n - 1] = 9.0                                   # the largest: in the last piece, cut short or whole
        _check(x, x.float().cpu().numpy())


@pytest.mark.parametrize("special", [float("nan"), float("inf")])
@pytest.mark.parametrize("rows,cols", [(301, 1031), (1024, 1024)])
def test_special_values(rows, cols, special):
    x = torch.from_numpy(R.fill_normal((rows, cols), 73)).bfloat16().cuda()
    for at in ((rows - 1, cols - 1), (rows // 2, 5)):
        say("quantize whole special", rows, cols, special, at)
        y = x.clone()
        y[at] = special
        yf = y.float().cpu().numpy()
        q, s = R.quantize_fp8(yf)
        for wait in (2000, 0):
            Q.set_option("quant_wait", wait)
            g, gs = Q.quantize(y, torch.float8_e4m3fn, Q.QUANT_PER_MATRIX)
            assert np.array_equal(host(gs).view(np.uint32), np.array([s]).view(np.uint32))
            assert np.array_equal(g.view(torch.uint8).cpu().numpy(), q)


@pytest.mark.parametrize("offset", [0, 1, 2, 3])
def test_addresses(offset):
    """Sources that start anywhere: at odd multiples of two bytes the two passes."""
    flat = torch.from_numpy(R.fill_normal((1, 300 * 1000 + 8), 75)).to(torch.float16).cuda()
    x = flat[0, offset:offset + 300 * 1000].view(300, 1000)
    say("quantize whole offset", offset)
    _check(x, x.float().cpu().numpy())


def test_in_a_capture():
    """Captured, the two passes: a replay on new values, several times, with eager launches between."""
    say("quantize whole captured")
    x = torch.from_numpy(R.fill_normal((500, 1000), 77)).bfloat16().cuda()
    Q.quantize(x, torch.int8, Q.QUANT_PER_MATRIX)
    Q.set_option("quant_wait", -1)
    Q.quantize(x, torch.int8, Q.QUANT_PER_MATRIX)            # (the workspace, outside the capture)
    Q.set_option("quant_wait", 2000)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        g, gs = Q.quantize(x, torch.int8, Q.QUANT_PER_MATRIX)
    for i in range(4):
        x.mul_(1.5 if i % 2 else 0.25)
        graph.replay()
        torch.cuda.synchronize()
        e, es = Q.quantize(x, torch.int8, Q.QUANT_PER_MATRIX)
        assert torch.equal(g, e) and torch.equal(gs, es), i


def test_in_a_capture_after_one_eager_call():
    """An eager call with the options as they are is all that a capture needs, also where nothing has used the workspace."""
    say("quantize whole, eager, captured, replayed")
    x = torch.from_numpy(R.fill_normal((500, 1000), 78)).bfloat16().cuda()
    torch.cuda.synchronize()
    L.check(L.load_library().qgemm_shutdown())
    Q.quantize(x, torch.int8, Q.QUANT_PER_MATRIX)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        g, gs = Q.quantize(x, torch.int8, Q.QUANT_PER_MATRIX)
    for i in range(4):
        x.mul_(1.5 if i % 2 else 0.25)
        graph.replay()
        torch.cuda.synchronize()
        e, es = Q.quantize(x, torch.int8, Q.QUANT_PER_MATRIX)
        assert torch.equal(g, e) and torch.equal(gs, es), i


def test_several_streams():
    """More launches than there are sets of words, on five streams with no synchronisation in between."""
    say("quantize whole, five streams")
    jobs = []
    for i in range(5):
        x = torch.from_numpy(R.fill_normal((700 + 100 * i, 1001), 80 + i)).bfloat16().cuda() * (i + 1)
        q, s = R.quantize_int8(x.float().cpu().numpy())
        jobs.append((x, q, s, torch.cuda.Stream(), []))
    torch.cuda.synchronize()
    for _ in range(30):
        for x, _, _, stream, got in jobs:
            with torch.cuda.stream(stream):
                got.append(Q.quantize(x, torch.int8, Q.QUANT_PER_MATRIX))
    torch.cuda.synchronize()
    for x, q, s, _, got in jobs:
        for g, gs in got:
            assert gs.cpu().numpy()[0] == s and np.array_equal(g.cpu().numpy(), q)


def test_launches_do_not_crowd_one_another_out():
    """Quantisations that take the whole chip each, on four streams, beside products on a fifth: with a wait of a quarter of a second
    a single launch that waited in vain would take longer than all of them together."""
    say("quantize whole, four streams, whole chip")
    n, rounds = 2048, 40
    xs = [torch.from_numpy(R.fill_normal((n, 4096), 90 + i)).bfloat16().cuda() for i in range(4)]
    want = [R.quantize_int8(x.float().cpu().numpy()) for x in xs]
    w = torch.zeros(4096, 4096, dtype=torch.int8, device="cuda")
    c, one = torch.empty(4096, 4096, dtype=torch.int32, device="cuda"), torch.ones(1, device="cuda")
    streams = [torch.cuda.Stream() for _ in range(5)]
    Q.set_option("quant_wait", 250000)
    for x, stream in zip(xs, streams):                      # (first launches of every kernel, and the workspace)
        with torch.cuda.stream(stream):
            Q.quantize(x, torch.int8, Q.QUANT_PER_MATRIX)
    Q.int8_mm(w, w, one, one, c)
    torch.cuda.synchronize()
    start = time.perf_counter()
    got = [[] for _ in xs]
    for _ in range(rounds):
        with torch.cuda.stream(streams[4]):
            Q.int8_mm(w, w, one, one, c)
        for i, x in enumerate(xs):
            with torch.cuda.stream(streams[i]):
                got[i].append(Q.quantize(x, torch.int8, Q.QUANT_PER_MATRIX))
    torch.cuda.synchronize()
    assert time.perf_counter() - start < 0.25
    for (q, s), results in zip(want, got):
        for g, gs in results:
            assert gs.cpu().numpy()[0] == s and np.array_equal(g.cpu().numpy(), q)
