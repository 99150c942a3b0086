"""What a launch leaves behind in the HIP runtime's last error, and what it takes from there: nothing either way."""
import ctypes as C
import re

import pytest
import torch

import qgemm_amd as Q
from qgemm_amd import lib as L
from tests.util import say

pytestmark = pytest.mark.gpu
HIP_OK, CAPTURE_RELAXED = 0, 2
STATUS_LAUNCH = 4


@pytest.fixture
def hip():
    """The runtime that the library and torch are running on."""
    torch.zeros(1, device="cuda")
    Q.load_library().qgemm_init()
    path = {m.group(1) for m in re.finditer(r"(/\S*libamdhip64\S*)", open("/proc/self/maps").read())}
    assert len(path) == 1, path
    lib = C.CDLL(path.pop())
    torch.cuda.synchronize()
    lib.hipGetLastError()
    yield lib
    lib.hipGetLastError()


def test_a_refused_launch_leaves_no_error_behind(hip):
    """A stream whose capture has been invalidated takes no launch.  The call says so; whoever asks the runtime next hears nothing."""
    say("refused launch")
    x = torch.randn(16, 256, device="cuda").bfloat16()
    q, s = Q.quantize(x, torch.float8_e4m3fn, Q.QUANT_BLOCK_1x128)
    torch.cuda.synchronize()
    stream = C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == HIP_OK
    assert hip.hipStreamBeginCapture(stream, CAPTURE_RELAXED) == HIP_OK
    assert hip.hipStreamSynchronize(stream) != HIP_OK                 # (not allowed while capturing: the capture is void)
    hip.hipGetLastError()
    status = L.load_library().qgemm_quantize(Q.DT_BF16, Q.DT_F8E4M3, Q.QUANT_BLOCK_1x128, x.data_ptr(), 256, 16, 256, q.data_ptr(), 256,
                                             s.data_ptr(), 2, 1, stream)
    left = hip.hipPeekAtLastError()
    graph = C.c_void_p()
    hip.hipStreamEndCapture(stream, C.byref(graph))
    assert hip.hipStreamDestroy(stream) == HIP_OK
    assert status == STATUS_LAUNCH
    assert left == HIP_OK


def test_an_error_that_somebody_left_is_not_taken_for_a_launch_of_ours(hip):
    """hipSetDevice of a device that is not there leaves an error in the runtime.  Calls behind it answer for their own launches, and
    leave that error where it is."""
    calls = []
    bf16 = lambda *shape: torch.randint(-3, 4, shape, device="cuda").bfloat16()                                                                  # noqa: E731
    for name, M, N, K, layout in (("short", 3, 5, 2, "nk"), ("any-shape kernel", 300, 500, 101, "nk"), ("few rows", 5, 500, 1001, "nk"), ("packed", 600, 2000, 4001, "nk"),
                                  ("transposed", 512, 512, 8192, "kn")):
        a, b, c = bf16(M, K), bf16(N, K), torch.zeros(M, N, device="cuda", dtype=torch.bfloat16)
        stored = b if layout == "nk" else b.t().contiguous()
        calls.append((name, lambda a=a, stored=stored, c=c, layout=layout: Q.gemm(a, stored, c, layout), c, lambda a=a, b=b: (a.float() @ b.float().t()).bfloat16()))
    for dtype in (torch.int8, torch.bfloat16, torch.float32):
        x, y = torch.randint(-9, 10, (130, 77), device="cuda").to(dtype), torch.zeros(77, 130, device="cuda", dtype=dtype)
        calls.append(("transpose", lambda x=x, y=y: Q.matrix_transpose(x, y), y, lambda x=x: x.t()))
    x = torch.randn(640, 2048, device="cuda").bfloat16()
    want = Q.quantize(x, torch.float8_e4m3fn, Q.QUANT_PER_MATRIX)[0].view(torch.uint8).clone()
    out = []
    calls.append(("quantise", lambda: out.append(Q.quantize(x, torch.float8_e4m3fn, Q.QUANT_PER_MATRIX)[0]), None, None))
    for name, run, c, ref in calls:
        run()                                                        # (kernels loaded, workspace there)
        torch.cuda.synchronize()
        if c is not None:
            c.zero_()
            torch.cuda.synchronize()
        hip.hipGetLastError()
        say("error of somebody else", name)
        assert hip.hipSetDevice(1 << 20) != HIP_OK
        left = hip.hipPeekAtLastError()
        run()
        after = hip.hipGetLastError()
        torch.cuda.synchronize()
        assert left != HIP_OK and after == left, (name, Q.last_config())
        got, expected = (c, ref()) if c is not None else (out[-1].view(torch.uint8), want)
        assert torch.equal(got, expected), (name, Q.last_config())
