"""GPU parity of version 15's path for up to 128 rows with N or K off the
multiples of 8 and K >= 1024 (B streamed at any row alignment), through the C
ABI: every count of 16-row blocks at its edges, column blocks of 8 to 128
columns, K with and without a remainder of the 32-deep steps, whole and split
over 2 to 32 workgroups.

* integer inputs: exact; random inputs: within the fp32 accumulation bound of
  the exact (fp64) product;
* values past an edge in memory (the next row of A or B) never reach C, and
  nothing outside C is written;
* results do not depend on the arrival order of a split (repeats are equal),
  nor on what used the library workspace before."""
import numpy as np
import pytest

from gpu_util import announce, check_f16_out, check_f32_out, make_inputs, run_gemm

pytestmark = pytest.mark.gpu

SHAPES = [(1, 9, 1024), (3, 8, 1031), (16, 129, 1057), (17, 127, 1088), (32, 135, 1999), (33, 1001, 1024),
          (48, 257, 1055), (49, 1001, 2048), (64, 4095, 2049), (80, 263, 4097), (96, 12, 4095), (100, 519, 1111),
          (112, 777, 4104), (113, 2001, 1600), (127, 1003, 8190), (2, 15, 16391), (128, 50257, 1030)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("out", ["f16", "f32"])
def test_random_and_integer(gpu, oracle, shape, out):
    m, n, k = shape
    A, B = make_inputs(m, n, k, "uniform", seed=m + 3 * n + k)
    (check_f16_out if out == "f16" else check_f32_out)(run_gemm(15, A, B, out), A, B,
                                                       oracle.dgemm(A.astype(np.float32), B.astype(np.float32)))
    if out == "f32":
        A, B = make_inputs(m, n, k, "int", seed=m + n + k)
        exact = A.astype(np.float64) @ B.astype(np.float64)
        assert np.array_equal(run_gemm(15, A, B, out).astype(np.float64), exact)


@pytest.mark.parametrize("shape", [(5, 131, 1030), (40, 1001, 2060)])
def test_values_past_the_edges_and_guards(gpu, shape):
    """A[1][0] is what row 0 reads past K, B[k][0] what row k-1 reads past N:
    infinite, they may only reach row 1 and column 0."""
    import torch
    import vibekernel_amd as vk
    m, n, k = shape
    A, B = make_inputs(m, n, k, "int", seed=m + n)
    A[1, 0] = np.inf
    B[k - 1, 0] = np.inf
    pad = 4096
    buf = torch.full((pad + m * n + pad,), float("nan"), dtype=torch.float32, device="cuda:0")
    C = buf[pad:pad + m * n].view(m, n)
    announce(f"version=15 few rows guarded m={m} n={n} k={k}")
    vk.matmul(m, n, k, torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda(), C, 15)
    torch.cuda.synchronize()
    assert torch.isnan(buf[:pad]).all() and torch.isnan(buf[pad + m * n:]).all()
    got = C.cpu().numpy().astype(np.float64)
    keep = np.ones((m, n), dtype=bool)
    keep[1, :] = False
    keep[:, 0] = False
    A[1, 0] = 0
    B[k - 1, 0] = 0
    exact = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(got[keep], exact[keep])


def test_repeats_and_shared_workspace(gpu):
    """A split shape between calls whose workspace holds copies there (past
    2^33 multiply-adds, 256 whole tiles: the copy of B is at its start)."""
    A, B = make_inputs(33, 1001, 4097, "normal", seed=3)
    A2, B2 = make_inputs(4096, 4095, 1032, "normal", seed=4)
    ref, ref2 = run_gemm(15, A, B, "f32"), run_gemm(15, A2, B2, "f32")
    for _ in range(3):
        assert np.array_equal(run_gemm(15, A, B, "f32"), ref)
        assert np.array_equal(run_gemm(15, A, B, "f32"), ref)
        assert np.array_equal(run_gemm(15, A2, B2, "f32"), ref2)


# K one past the whole 32-deep steps: the last element of A ends the last
# fragment's dword where the last row is odd, and is past it where it is even
@pytest.mark.parametrize("shape", [(1, 40, 1025), (2, 40, 1025), (11, 40, 1025), (16, 40, 1025), (31, 136, 1057),
                                   (32, 136, 1057), (47, 264, 2049), (64, 264, 2049), (95, 129, 1089), (96, 129, 1089),
                                   (127, 72, 4129), (128, 72, 4129)])
def test_odd_k(gpu, shape):
    m, n, k = shape
    A, B = make_inputs(m, n, k, "int", seed=m + n + k)
    exact = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(run_gemm(15, A, B, "f32").astype(np.float64), exact)
