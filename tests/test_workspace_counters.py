"""The library workspace's counters on the host: libvk_gemm.so's own launch code
over a stand-in HIP runtime that logs launches (host_launches.py).  Fresh and
reused memory holds garbage there, so a launch that counts arrivals must find
its counters at zero, whatever calls came before it and whether they split K,
copied operands to the workspace's start or left it alone.  The GPU counterpart
is tests/test_gpu_workspace_counters.py."""
import pytest

import host_launches


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    stub = host_launches.build_stub(tmp_path_factory.mktemp("stub"))
    return lambda calls: host_launches.launches(stub, calls)


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
