"""GPU parity of fp16 version 1 (any shape, any 2-byte alignment): at the edges
of its 64 x 64 and 128 x 128 tiles and of its 128- and 64-deep k-tiles, N or K
below one 16-byte chunk, operands off the 16-byte boundaries; integer inputs
exact, random ones within the fp32 accumulation bound of the exact (fp64)
product, nothing written outside C, values past an edge in memory kept out of
it."""
import numpy as np
import pytest

from gpu_util import announce, check_f16_out, check_f32_out, make_inputs

pytestmark = pytest.mark.gpu

# from (1990, 2047, 33) on: 128 x 128 tiles (256 CUs)
SHAPES = [(1, 1, 1), (2, 7, 9), (5, 9, 7), (63, 65, 128), (64, 64, 127), (65, 63, 129), (1, 129, 255), (129, 12, 257),
          (200, 130, 640), (64, 67, 512), (100, 300, 70), (1990, 2047, 33), (2047, 1985, 130), (1601, 1600, 191),
          (1600, 1609, 320), (25000, 5, 65), (25000, 70, 6), (200, 7, 300), (65, 1, 129),
          (64, 5, 256), (130, 3, 1023), (67000, 7, 200)]


def _run(A, B, out, shift):
    import torch
    import vibekernel_amd as vk
    m, k = A.shape
    n = B.shape[1]

    def put(x):  # `shift` halves past a 16-byte boundary
        buf = torch.empty(x.size + shift, dtype=torch.float16, device="cuda:0")
        buf[shift:] = torch.from_numpy(x).reshape(-1)
        return buf[shift:].view(x.shape)

    pad = 1024
    dt = torch.float16 if out == "f16" else torch.float32
    buf = torch.full((pad + shift + m * n + pad,), float("nan"), dtype=dt, device="cuda:0")
    C = buf[pad + shift:pad + shift + m * n].view(m, n)
    announce(f"f16 version=1 m={m} n={n} k={k} out={out} shift={shift}")
    vk.matmul(m, n, k, put(A), put(B), C, 1)
    torch.cuda.synchronize()
    assert torch.isnan(buf[:pad + shift]).all() and torch.isnan(buf[pad + shift + m * n:]).all()
    return C.cpu().numpy()


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("out,shift", [("f16", 0), ("f16", 3), ("f32", 1)])
def test_random_and_integer(gpu, oracle, shape, out, shift):
    m, n, k = shape
    A, B = make_inputs(m, n, k, "uniform", seed=m + 2 * n + 3 * k)
    (check_f16_out if out == "f16" else check_f32_out)(_run(A, B, out, shift), A, B,
                                                       oracle.dgemm(A.astype(np.float32), B.astype(np.float32)))
    if out == "f32":
        A, B = make_inputs(m, n, k, "int", seed=m + n + k)
        assert np.array_equal(_run(A, B, out, shift).astype(np.float64), A.astype(np.float64) @ B.astype(np.float64))


# C in whole rows through LDS or not, at both sides of half a tile; 128 x 128 tiles from (63, 65603, 9) on
@pytest.mark.parametrize("shape", [(31, 33, 40), (32, 31, 40), (32, 33, 40), (33, 39, 7), (95, 41, 70), (63, 65603, 9),
                                   (64, 65603, 9), (70001, 63, 9), (70001, 65, 9), (65, 65543, 5)])
@pytest.mark.parametrize("shift", [0, 1])
def test_rows_of_c(gpu, oracle, shape, shift):
    m, n, k = shape
    A, B = make_inputs(m, n, k, "int", seed=m + n + k)  # sums of at most 4 k: exact in fp16
    assert np.array_equal(_run(A, B, "f16", shift).astype(np.float32), A.astype(np.float32) @ B.astype(np.float32))


@pytest.mark.parametrize("shape", [(3, 5, 35), (70, 67, 130), (1700, 1603, 260), (70, 5, 200), (70, 67, 5)])
def test_values_past_the_edges_never_reach_c(gpu, shape):
    """A[1][0] is what row 0 reads past K, B[k-1][0] what row k-2 reads past
    N: infinite, they may only reach row 1 and column 0."""
    m, n, k = shape
    A, B = make_inputs(m, n, k, "int", seed=m + k)
    A[1, 0] = np.inf
    B[k - 1, 0] = np.inf
    C = _run(A, B, "f32", 0)
    keep = np.ones((m, n), dtype=bool)
    keep[1, :] = False
    keep[:, 0] = False
    A[1, 0] = 0
    B[k - 1, 0] = 0
    exact = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(C[keep].astype(np.float64), exact[keep])
