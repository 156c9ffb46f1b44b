"""GPU parity of version 11's 64 x 256 tiles (grids of 128 x 128 tiles just
past a whole round of the CUs, an odd number of 64-row blocks): bitwise equal
to version 13, which runs the same sums on whole 128 x 128 tiles; integer
inputs exact; nothing written outside C, values past an edge kept out of it.
K of one k-tile, odd and even numbers of them, and remainders; N at the edges
of a tile.  (256 CUs: 258 to 276 square tiles, 195 to 245 wide ones.)"""
import numpy as np
import pytest

from gpu_util import announce, make_inputs, run_gemm

pytestmark = pytest.mark.gpu

SHAPES = [(300, 11008, 256), (257, 11000, 72), (320, 10928, 200), (192, 16640, 64), (150, 17152, 8), (448, 8712, 328),
          (320, 11008, 448), (129, 16648, 1000)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("out", ["f16", "f32"])
def test_bits_of_whole_square_tiles(gpu, shape, out):
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    m, n, k = shape
    if cus == 256:
        assert -(-m // 128) * -(-n // 128) > cus >= -(-m // 64) * -(-n // 256), "the case must take 64 x 256 tiles"
    A, B = make_inputs(m, n, k, "uniform", seed=m + 3 * n + k)
    u = np.uint16 if out == "f16" else np.uint32
    C = run_gemm(11, A, B, out)
    assert not np.isnan(C.astype(np.float32)).any()
    assert np.array_equal(C.view(u), run_gemm(13, A, B, out).view(u))


@pytest.mark.parametrize("shape", [(300, 11000, 72), (192, 16640, 64)])
def test_exact_guards_and_edges(gpu, shape):
    import torch
    import vibekernel_amd as vk
    m, n, k = shape
    A, B = make_inputs(m, n, k, "int", seed=m + n)
    A[1, 0] = np.inf
    B[k - 1, 0] = np.inf
    pad = 4096
    buf = torch.full((pad + m * n + pad,), float("nan"), dtype=torch.float32, device="cuda:0")
    C = buf[pad:pad + m * n].view(m, n)
    announce(f"version=11 wide guarded m={m} n={n} k={k}")
    vk.matmul(m, n, k, torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda(), C, 11)
    torch.cuda.synchronize()
    assert torch.isnan(buf[:pad]).all() and torch.isnan(buf[pad + m * n:]).all()
    keep = np.ones((m, n), dtype=bool)
    keep[1, :] = False
    keep[:, 0] = False
    A[1, 0] = 0
    B[k - 1, 0] = 0
    assert np.array_equal(C.cpu().numpy()[keep].astype(np.float64), (A.astype(np.float32) @ B.astype(np.float32))[keep])
