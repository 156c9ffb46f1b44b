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
