"""vk_gemm_pick against the rule written out over vk_gemm_check, for shapes at
and around every line of it, on the current device's compute units (256 with
none visible)."""
import itertools
import random

import pytest

from vibekernel_amd import VkError, _abi, pick_version

F16, F32 = 1, 2


def _cus():
    import torch
    if torch.cuda.is_available():
        return torch.cuda.get_device_properties(torch.cuda.current_device()).multi_processor_count
    return 256


def _rule(m, n, k, in_dt, out_dt):
    def takes(v):
        return _abi.check(v, in_dt, out_dt, m, n, k, 4096, 4096, 4096) == 0

    if in_dt == F32:
        return next((v for v in (2, 3, 1) if takes(v)), None)
    cus, tiles = _cus(), -(-m // 128) * -(-n // 128)
    on_grid = m % 256 == 0 and n % 256 == 0 and k % 64 == 0
    v11 = tiles <= cus if on_grid else 2 * tiles <= 3 * cus
    v14 = m <= 128 and n <= 4096 and not (m <= 32 and k > 12288) and (
        (n > 2048 or (m <= 8 and n > 1024 and k <= 8192)) if m <= 64 else k <= 8192)
    for v in (14, 8, 4, 11, 9, 7, 10, 6, 5, 3, 2, 15, 1):
        if (v == 14 and not v14) or (v == 8 and m > 128 and v11 and takes(11)) or (v == 11 and not v11):
            continue
        if (v == 9 and _abi.workspace_bytes(9, in_dt, m, n, k) == 0) or (v == 15 and m * n * k < 1 << 24):
            continue
        if takes(v):
            return v
    return None


MS = [0, 1, 8, 9, 16, 32, 33, 64, 65, 128, 129, 255, 256, 257, 512, 2048, 4096, 1 << 24]
NS = [0, 1, 7, 8, 300, 1024, 1032, 2048, 2056, 4096, 4104, 8192, 50257, 1 << 22]
KS = [0, 1, 32, 70, 1024, 4095, 4096, 8192, 8224, 12288, 14336, (1 << 31) - 1]
OVER = [(1 << 31, 8, 8), (8, 1 << 31, 8), (8, 8, 1 << 31), ((1 << 31) - 1,) * 3, ((1 << 64) - 1, 64, 64)]


@pytest.mark.parametrize("dtype,out", [("f16", "f16"), ("f16", "f32"), ("f32", "f32"), ("f32", "f16")])
def test_pick_equals_the_rule(dtype, out):
    rng = random.Random(5)
    drawn = [tuple(int(2 ** (13 * rng.random())) for _ in range(3)) for _ in range(1500)]
    codes = {"f16": F16, "f32": F32}
    for m, n, k in itertools.chain(itertools.product(MS, NS, KS), OVER, drawn):
        want = _rule(m, n, k, codes[dtype], codes[out])
        if want is None:
            with pytest.raises(VkError) as e:
                pick_version(m, n, k, dtype, out)
            assert e.value.status == -3
        else:
            assert pick_version(m, n, k, dtype, out) == want, (m, n, k, dtype, out)
