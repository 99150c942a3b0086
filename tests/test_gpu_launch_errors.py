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
