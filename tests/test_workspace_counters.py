"""The library workspace's counters on the host: libvk_gemm.so's own launch code
over a stand-in HIP runtime (tests/native/hip_stub.cpp) that logs launches.
Fresh and reused memory holds garbage there, so a launch that counts arrivals
must find its counters at zero, whatever calls came before it and whether they
split K, copied operands to the workspace's start or left it alone.  The GPU
counterpart is tests/test_gpu_workspace_counters.py."""
import json
import os
import subprocess
import sys

import pytest

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


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    """[(status, launch lines)] of a list of calls (dtype 1: fp16, 2: fp32) in a
    fresh process."""
    if not os.path.exists(LIB):
        pytest.fail(f"{LIB} is not built")
    stub = str(tmp_path_factory.mktemp("stub") / "libhip_stub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", STUB, "-o", stub], check=True, timeout=300)

    def run(calls):
        r = subprocess.run([sys.executable, "-c", CHILD, stub, LIB, json.dumps(calls)], capture_output=True, text=True,
                           timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr
        return json.loads(r.stdout.splitlines()[-1])

    return run


def v15(*shape):
    return [1, 15, *shape]


def v3(*shape):
    return [2, 3, *shape]


HEAD = v15(32, 50257, 4096)      # few rows, unsplit
HEAD2 = v15(100, 8193, 1024)     # the same above 64 rows
SPLIT = v15(16, 4095, 4096)      # few rows, K split
COPIES = v15(4096, 4095, 4096)   # copies of B at the workspace's start
ANY = v15(1000, 1001, 999)       # no workspace used
F32_HEAD = v3(16, 4096, 256)     # few rows, unsplit (too few k-steps)
F32_HEAD2 = v3(16, 18432, 4096)  # the same (enough column blocks)
F32_SPLIT = v3(16, 4096, 4096)   # few rows, K split
F32_TILES = v3(100, 512, 1024)   # tiles, K split

SEQUENCES = {
    "fresh, unsplit, split": [HEAD, SPLIT],
    "copies, unsplit, split": [COPIES, HEAD2, SPLIT],
    "split, copies, unsplit, split": [HEAD, SPLIT, COPIES, HEAD, SPLIT],
    "copies, any, split": [COPIES, ANY, SPLIT],
    "another version between": [SPLIT, F32_SPLIT, HEAD2, SPLIT],
    "fp32: fresh, unsplit, split": [F32_HEAD2, F32_HEAD, F32_SPLIT],
    "fp32: copies, unsplit, split": [COPIES, F32_HEAD, F32_SPLIT],
    "fp32: copies, unsplit, split tiles": [COPIES, F32_HEAD, F32_TILES],
    "fp32: tiles and few rows": [F32_TILES, F32_SPLIT, COPIES, F32_HEAD2, F32_SPLIT, F32_TILES],
}


@pytest.mark.parametrize("name", SEQUENCES)
def test_counting_launches_find_zeroed_counters(launches, name):
    calls = SEQUENCES[name]
    out = launches(calls)
    for call, (status, lines) in zip(calls, out):
        assert status == 0
        assert not any("counters=dirty" in x for x in lines), (call, lines)
        if call in (SPLIT, F32_SPLIT, F32_TILES):
            assert any("counters=clean" in x for x in lines), (call, lines)
        else:
            assert not any("counters=clean" in x for x in lines), (call, lines)


@pytest.mark.parametrize("calls", [[SPLIT, HEAD, SPLIT], [SPLIT, ANY, HEAD2, SPLIT],
                                   [F32_SPLIT, F32_HEAD, F32_TILES, F32_HEAD, F32_SPLIT]])
def test_calls_that_leave_the_workspace_alone_cost_no_clear(launches, calls):
    """Once the workspace is large enough, the counters stay known to be zero
    past calls that do not touch them."""
    warm = [max(calls, key=lambda c: c[2] * c[3] * c[4])] + calls[:1]
    out = launches(warm + calls)
    assert not any("zero_fill" in x for _, lines in out[len(warm):] for x in lines), out
