"""Runs the library's host code, launches included, without a device: a process of its own, in which
tests/host_runtime/host_runtime.cpp stands for the HIP runtime.  A script has `lib` (the C ABI), `events()` (what the library asked
of the runtime since the last call: malloc, launch, record, wait, synchronize lines), `kernels()` (the kernels among them) and the
runtime's switches."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_HEAD = """
import ctypes as C, importlib.util, re
runtime = C.CDLL({runtime!r}, mode=C.RTLD_GLOBAL)
spec = importlib.util.spec_from_file_location("qgemm_lib", {lib!r})
L = importlib.util.module_from_spec(spec)
spec.loader.exec_module(L)
lib = L.load_library()
runtime.host_events.restype = C.c_char_p
runtime.host_budget.argtypes = [C.c_size_t]
runtime.host_capture.argtypes = [C.c_void_p, C.c_int]
F32, BF16, F16, I8, F8, I32 = {dtypes}
def events():
    text = runtime.host_events().decode().splitlines()
    runtime.host_clear()
    return text
def kernels():
    return [re.match("launch _ZN5qgemm[0-9]+([a-z0-9_]+?_kernel)", e).group(1) for e in events() if e.startswith("launch ")]
def option(key, value):
    assert lib.qgemm_set_option(key.encode(), value) == 0
def config():
    buf = C.create_string_buffer(160)
    assert lib.qgemm_last_config(buf, 160) == 0
    return buf.value.decode()
def quantize(rows, cols, stream=0, mode=1, ld=0, x=1 << 32, dt=BF16, out=I8):
    return lib.qgemm_quantize(dt, out, mode, x, ld or cols, rows, cols, 1 << 33, cols, 1 << 34, 1, 1, stream)
def product(M, N, K, stream=0, dt=I8, out=I32, mode=1, layout=0, split=0, a=1 << 32, b=1 << 33, static=False, ldc=0):
    f = lib.qgemm_scaled_gemm_static if static else lib.qgemm_scaled_gemm
    return f(dt, out, mode, layout, a, b, 1 << 34, 1 << 35, 1 << 36, ldc or N, M, N, K, split, stream)
def plain(M, N, K, stream=0, dt=BF16, out=BF16, layout=1, a=1 << 32, b=1 << 33, lda=0, ldb=0):
    return lib.qgemm_gemm(dt, out, layout, a, lda or K, b, ldb or (K if layout else N), 1 << 36, N, M, N, K, stream)
"""


def run(tmp_path_factory, script, library=None):
    gxx = shutil.which("g++")
    if gxx is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime_api.h"):
        pytest.skip("no g++ or no HIP headers")
    out = os.path.join(str(tmp_path_factory.getbasetemp()), "host_runtime.so")
    if not os.path.exists(out):
        subprocess.run([gxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", out,
                        os.path.join(ROOT, "tests", "host_runtime", "host_runtime.cpp")], check=True, timeout=300)
    import qgemm_amd as Q
    from qgemm_amd import lib as L
    head = _HEAD.format(runtime=out, lib=L.__file__, 
                        dtypes=(Q.DT_F32, Q.DT_BF16, Q.DT_F16, Q.DT_I8, Q.DT_F8E4M3, Q.DT_I32))
    env = dict(os.environ, QGEMM_LIBRARY=library or L.library_path())
    done = subprocess.run([sys.executable, "-c", head + script], capture_output=True, text=True, timeout=300, env=env, cwd=ROOT)
    assert done.returncode == 0, done.stdout[-2000:] + done.stderr[-4000:]
    return done.stdout
