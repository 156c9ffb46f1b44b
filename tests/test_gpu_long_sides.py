"""Products whose tile rows or columns are more than one side of a grid holds,
exact on integer inputs, every element written.  The grids themselves are
checked in tests/test_launch_limits.py."""
import pytest

from gpu_util import announce

pytestmark = pytest.mark.gpu


def test_tall_f16(gpu):
    """70,313 rows of 128-row tiles, N off the multiples of 8."""
    import torch
    import vibekernel_amd as vk
    m, n, k = 9000000, 9, 8
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(1)
    A = torch.randint(-4, 5, (m, k), generator=gen, device="cuda:0", dtype=torch.int8)
    B = torch.randint(-4, 5, (k, n), generator=gen, device="cuda:0", dtype=torch.int8)
    exact = sum(A[:, i:i + 1].short() * B[i:i + 1].short() for i in range(k))  # at most 128: exact in fp16
    C = torch.full((m, n), float("nan"), dtype=torch.float16, device="cuda:0")
    version = vk.pick_version(m, n, k)
    announce(f"tall version={version} m={m} n={n} k={k}")
    assert version == 15
    vk.matmul(m, n, k, A.half(), B.half(), C, version)
    torch.cuda.synchronize()
    assert torch.equal(C, exact.half())


def test_wide_f32(gpu):
    """One row of 2^30 + 77 columns: more than 2^32 threads in one row of
    tiles."""
    import torch
    import vibekernel_amd as vk
    n = 2 ** 30 + 77
    A = torch.tensor([[3.0]], device="cuda:0")
    B = (torch.arange(n, device="cuda:0", dtype=torch.int32) % 1000003).float().view(1, n)
    C = torch.full((1, n), float("nan"), device="cuda:0")
    version = vk.pick_version(1, n, 1, "f32")
    announce(f"wide f32 version={version} n={n}")
    assert version == 1
    vk.matmul(1, n, 1, A, B, C, version)
    torch.cuda.synchronize()
    assert torch.equal(C, 3 * B)
