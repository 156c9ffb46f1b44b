"""Launches stay within the runtime's limits, on the host: libvk_gemm.so's own
launch code over a stand-in HIP runtime that logs launches (host_launches.py).
HIP takes grid.y up to 65535 and fewer than 2^32 threads along x; the shapes are
tall or wide enough that a grid of tile rows and columns would not fit.  The GPU
counterpart is tests/test_gpu_long_sides.py."""
import re

import pytest

import host_launches

F16, F32 = 1, 2


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    stub = host_launches.build_stub(tmp_path_factory.mktemp("stub"))
    return lambda calls: host_launches.launches(stub, calls)


# (dtype, version, m, n, k), all accepted by vk_gemm_check
SHAPES = [(F16, 15, 9000000, 9, 8), (F16, 15, 65535 * 128 + 1, 1, 100), (F16, 15, 65535 * 128, 9, 8),
          (F16, 1, 65535 * 128, 9, 8), (F32, 1, 65535 * 128, 3, 5),
          (F32, 1, 65, 2 ** 30, 1), (F32, 1, 1, 2 ** 30 + 77, 1), (F32, 1, 70, 2 ** 29 + 5, 2)]


@pytest.mark.parametrize("shape", SHAPES)
def test_grids_fit(launches, shape):
    (status, lines), = launches([list(shape)])
    assert status == 0 and lines
    for line in lines:
        x, y, z, block = map(int, re.search(r"grid=(\d+),(\d+),(\d+) block=(\d+)", line).groups())
        assert y <= 65535 and z <= 65535 and x * block < 2 ** 32, line
