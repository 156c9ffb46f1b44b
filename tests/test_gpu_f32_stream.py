"""GPU parity of fp32 version 3's path for up to 64 rows (B streamed once):
every count of 16-row blocks at its edges, column blocks of 4 to 64 columns,
K below one 16-deep step and with remainders of 4, 8 and 12, whole and split
over workgroups.  Integer inputs exact, random ones within 2 k u |A||B| of the
exact (fp64) product; values past an edge in memory and memory outside C stay
out of it; repeats are bitwise equal (whichever piece arrives last)."""
import numpy as np
import pytest

from gpu_util import announce, check_f32_out, make_inputs, run_gemm

pytestmark = pytest.mark.gpu

SHAPES = [(1, 4, 4), (1, 4096, 4096), (15, 60, 12), (16, 64, 16), (17, 68, 1000), (32, 132, 1028), (33, 4096, 2056),
          (48, 1000, 8408), (49, 2052, 4100), (64, 50260, 172), (63, 520, 16388), (64, 8, 2064), (2, 64, 100)]


@pytest.mark.parametrize("shape", SHAPES)
def test_random_and_integer(gpu, oracle, shape):
    m, n, k = shape
    A, B = make_inputs(m, n, k, "uniform", seed=m + 3 * n + k, dtype=np.float32)
    C = run_gemm(3, A, B, "f32")
    check_f32_out(C, A, B, oracle.dgemm(A, B))
    for _ in range(3):
        assert np.array_equal(run_gemm(3, A, B, "f32"), C)
    A, B = make_inputs(m, n, k, "int", seed=m + n + k, dtype=np.float32)
    assert np.array_equal(run_gemm(3, A, B, "f32").astype(np.float64), A.astype(np.float64) @ B.astype(np.float64))


@pytest.mark.parametrize("shape", [(5, 68, 20), (40, 4100, 2076)])
def test_values_past_the_edges_and_guards(gpu, shape):
    """A[1][0] is what row 0 reads past K, B[k-1][0] what row k-2 reads past
    N: infinite, they may only reach row 1 and column 0."""
    import torch
    import vibekernel_amd as vk
    m, n, k = shape
    A, B = make_inputs(m, n, k, "int", seed=m + n, dtype=np.float32)
    A[1, 0] = np.inf
    B[k - 1, 0] = np.inf
    pad = 4096
    buf = torch.full((pad + m * n + pad,), float("nan"), dtype=torch.float32, device="cuda:0")
    C = buf[pad:pad + m * n].view(m, n)
    announce(f"f32 version=3 few rows guarded m={m} n={n} k={k}")
    vk.matmul(m, n, k, torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda(), C, 3)
    torch.cuda.synchronize()
    assert torch.isnan(buf[:pad]).all() and torch.isnan(buf[pad + m * n:]).all()
    keep = np.ones((m, n), dtype=bool)
    keep[1, :] = False
    keep[:, 0] = False
    A[1, 0] = 0
    B[k - 1, 0] = 0
    exact = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(C.cpu().numpy()[keep].astype(np.float64), exact[keep])
