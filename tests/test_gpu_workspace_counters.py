"""Versions 15 and fp32 3 on one library workspace, in orders where a call that
does not split K stands between one that leaves operand copies at the
workspace's start (or a new allocation) and one that counts arrivals there:
exact on integer inputs, every element written.  The host side alone is
tests/test_workspace_counters.py."""
import numpy as np
import pytest

from gpu_util import make_inputs, run_gemm

pytestmark = pytest.mark.gpu

HEAD = (15, 32, 50257, 4096)     # few rows, unsplit
HEAD2 = (15, 100, 8193, 1024)    # the same above 64 rows
SPLIT = (15, 16, 4095, 4096)     # few rows, K split
COPIES = (15, 4096, 4095, 4096)  # copies of B at the workspace's start (256 whole tiles)
ANY = (15, 1000, 1001, 999)      # no workspace used
F32_HEAD = (3, 16, 4096, 256)    # few rows, unsplit
F32_SPLIT = (3, 16, 4096, 4096)  # few rows, K split
F32_TILES = (3, 100, 512, 1024)  # tiles, K split


@pytest.fixture(scope="module")
def cases():
    """Inputs and the exact product of a call, made once."""
    made = {}

    def get(call):
        if call not in made:
            version, m, n, k = call
            A, B = make_inputs(m, n, k, "int", seed=m + n + k, dtype=np.float32 if version == 3 else np.float16)
            B[0, :] = 3  # the copies' first row, where the counters are, holds no zero
            made[call] = A, B, A.astype(np.float32) @ B.astype(np.float32)
        return made[call]

    return get


@pytest.mark.parametrize("calls", [
    [HEAD, SPLIT],
    [COPIES, HEAD2, SPLIT, SPLIT],
    [SPLIT, COPIES, HEAD, ANY, SPLIT],
    [COPIES, F32_HEAD, F32_SPLIT, F32_SPLIT],
    [COPIES, F32_HEAD, F32_TILES, F32_SPLIT, F32_TILES],
], ids=lambda calls: "-".join("x".join(map(str, c[1:])) for c in calls))
def test_products_after_untouched_workspaces(gpu, cases, calls):
    from vibekernel_amd import _abi
    _abi.release()  # the first call of the sequence allocates
    for call in calls:
        A, B, exact = cases(call)
        assert np.abs(exact).max() < 2 ** 24
        assert np.array_equal(run_gemm(call[0], A, B, "f32"), exact), call
