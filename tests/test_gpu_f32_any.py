"""GPU parity of fp32 version 1's matrix-core path (any shape, any 4-byte
alignment): bits equal to the oracle's fused multiply-add chain, at the edges
of its 64 x 64 and 128 x 128 tiles and of its 64- and 32-deep k-tiles, N or K
below one 16-byte chunk, operands off the 16-byte boundaries; values past an
edge in memory and memory outside C stay out of it."""
import numpy as np
import pytest

from gpu_util import announce, make_inputs

pytestmark = pytest.mark.gpu

# the last two on 128 x 128 tiles (256 CUs)
SHAPES = [(1, 1, 3), (2, 3, 64), (5, 2, 7), (63, 65, 64), (64, 64, 63), (65, 63, 129), (1, 129, 191), (129, 1, 193),
          (200, 130, 320), (64, 67, 256), (1990, 2047, 33), (2047, 1985, 130)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("shift", [0, 1])
def test_bits_equal_to_the_oracle(gpu, oracle, shape, shift):
    import torch
    import vibekernel_amd as vk
    m, n, k = shape
    A, B = make_inputs(m, n, k, "uniform", seed=m + 2 * n + 3 * k, dtype=np.float32)

    def put(x):  # `shift` floats past a 16-byte boundary
        buf = torch.empty(x.size + shift, dtype=torch.float32, device="cuda:0")
        buf[shift:] = torch.from_numpy(x).reshape(-1)
        return buf[shift:].view(x.shape)

    pad = 1024
    buf = torch.full((pad + shift + m * n + pad,), float("nan"), dtype=torch.float32, device="cuda:0")
    C = buf[pad + shift:pad + shift + m * n].view(m, n)
    announce(f"f32 version=1 m={m} n={n} k={k} shift={shift}")
    vk.matmul(m, n, k, put(A), put(B), C, 1)
    torch.cuda.synchronize()
    assert torch.isnan(buf[:pad + shift]).all() and torch.isnan(buf[pad + shift + m * n:]).all()
    assert np.array_equal(C.cpu().numpy(), oracle.sgemm(A, B))


# K within one k-tile of 32 or 64, two of 64, and any K with N below 4: at the
# 16-deep groups and the 16-row blocks that are left out when they hold nothing
@pytest.mark.parametrize("mn", [(1, 5), (16, 3), (17, 16), (33, 67), (48, 17), (70, 130)], ids=lambda mn: "%dx%d" % mn)
@pytest.mark.parametrize("shift", [0, 1])
def test_small_k(gpu, oracle, mn, shift):
    m, n = mn
    for k in (1, 2, 3, 4, 5, 15, 16, 17, 31, 32, 33, 48, 50, 63, 64, 65, 80, 83, 112, 127, 128):
        test_bits_equal_to_the_oracle(gpu, oracle, (m, n, k), shift)


@pytest.mark.parametrize("shape", [(1, 1, 129), (64, 3, 192), (65, 2, 200), (47, 3, 257), (130, 1, 1023)])
@pytest.mark.parametrize("shift", [0, 1])
def test_few_columns(gpu, oracle, shape, shift):
    test_bits_equal_to_the_oracle(gpu, oracle, shape, shift)


@pytest.mark.parametrize("shape", [(3, 5, 35), (70, 67, 130), (70, 67, 30), (18, 40, 61), (34, 65, 100), (33, 2, 200)])
def test_values_past_the_edges_never_reach_c(gpu, shape):
    """A[1][0] is what row 0 reads past K, B[k-1][0] what row k-2 reads past
    N: infinite, they may only reach row 1 and column 0."""
    import torch
    import vibekernel_amd as vk
    m, n, k = shape
    A, B = make_inputs(m, n, k, "int", seed=m + k, dtype=np.float32)
    A[1, 0] = np.inf
    B[k - 1, 0] = np.inf
    C = torch.empty((m, n), dtype=torch.float32, device="cuda:0")
    announce(f"f32 version=1 edges m={m} n={n} k={k}")
    vk.matmul(m, n, k, torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda(), C, 1)
    torch.cuda.synchronize()
    keep = np.ones((m, n), dtype=bool)
    keep[1, :] = False
    keep[:, 0] = False
    A[1, 0] = 0
    B[k - 1, 0] = 0
    exact = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(C.cpu().numpy()[keep].astype(np.float64), exact[keep])
