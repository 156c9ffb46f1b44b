"""libvk_gemm.so's own launch code on the host, over a stand-in HIP runtime
(tests/native/hip_stub.cpp) that logs launches instead of running them."""
import json
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STUB = os.path.join(ROOT, "tests", "native", "hip_stub.cpp")
LIB = os.path.join(ROOT, "vibekernel_amd", "lib", "libvk_gemm.so")

# In a process of its own: the stand-in has to be there before any HIP runtime.
CHILD = """
import ctypes, json, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
stub.stub_log.restype = ctypes.c_char_p
lib = ctypes.CDLL(sys.argv[2])
lib.vk_gemm.argtypes = [ctypes.c_int] * 3 + [ctypes.c_size_t] * 3 + [ctypes.c_void_p] * 4
done, out = 0, []
for dtype, version, m, n, k in json.loads(sys.argv[3]):
    status = lib.vk_gemm(version, dtype, dtype, m, n, k, 4096, 4096, 4096, None)
    lines = stub.stub_log().decode().splitlines()
    out.append([status, lines[done:]])
    done = len(lines)
print(json.dumps(out))
"""


def build_stub(folder):
    """The stand-in runtime, built in `folder`."""
    assert os.path.exists(LIB), f"{LIB} is not built"
    stub = os.path.join(str(folder), "libhip_stub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", STUB, "-o", stub], check=True, timeout=300)
    return stub


def launches(stub, calls):
    """[(status, launch lines)] of calls [dtype, version, m, n, k] (dtype 1: fp16,
    2: fp32, in and out) in a fresh process."""
    r = subprocess.run([sys.executable, "-c", CHILD, stub, LIB, json.dumps(calls)], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return json.loads(r.stdout.splitlines()[-1])
