"""Which kernel a call launches, on the host: libvk_gemm.so's own launch code
over a stand-in HIP runtime that logs launches (host_launches.py; 256 CUs).
Each case lies on one side of a rule whose two sides are measured where it
stands in the source."""
import pytest

import host_launches

F16, F32 = 1, 2


@pytest.fixture(scope="module")
def kernel(tmp_path_factory):
    """The (mangled) name of the last kernel that one call launches."""
    stub = host_launches.build_stub(tmp_path_factory.mktemp("stub"))

    def run(*call):
        (status, lines), = host_launches.launches(stub, [list(call)])
        assert status == 0, call
        return lines[-1].split()[0]

    return run


# C's rows on 16-byte boundaries or not: the last template argument
@pytest.mark.parametrize("call,name", [
    ((F16, 10, 520, 520, 64), "f16_pp16_edge_kernelIDF16_Lb0EE"),
    ((F16, 10, 1000, 1000, 4000), "f16_pp16_sk_kernelIDF16_Lb1ELb0EE"),
    ((F16, 15, 4096, 4096, 4095), "f16_pp16_edge_kernelIDF16_Lb0EE"),
    ((F16, 15, 4096, 4095, 4096), "f16_pp16_edge_kernelIDF16_Lb1EE"),
    ((F16, 15, 300, 201, 4095), "f16_pp16_sk_kernelIDF16_Lb1ELb1EE"),
])
def test_rows_of_c_in_version_10(kernel, call, name):
    assert name in kernel(*call)


# version 11's 64 x 256 tiles (the last template argument) by rounds of the CUs
@pytest.mark.parametrize("call,wide", [
    ((F16, 11, 300, 11008, 16384), True),   # 2 -> 1
    ((F16, 11, 320, 22016, 1024), True),    # 3 -> 2
    ((F16, 11, 320, 22016, 2048), False),
    ((F16, 11, 192, 65536, 512), True),     # 4 -> 3
    ((F16, 11, 192, 65536, 4096), False),
    ((F16, 11, 320, 65536, 256), True),     # 6 -> 5
    ((F16, 11, 320, 65536, 2048), False),
    ((F16, 11, 64, 98304, 4096), True),     # 3 -> 2, half of each square tile empty
    ((F16, 11, 1024, 4096, 4096), False),   # one round of square tiles
    ((F16, 11, 256, 16512, 4096), False),   # two rounds either way
    ((F16, 11, 256, 16512, 64), False),
    ((F16, 11, 129, 16640, 4096), True),
])
def test_wide_tiles_of_version_11(kernel, call, wide):
    name = kernel(*call)
    assert ("f16_pp128n_kernel" in name and "ELb0ELb1EE" in name) == wide, name


# few rows of version 15: A by whole dwords where K is odd and M above 9 (the last template argument)
@pytest.mark.parametrize("call,name", [((F16, 15, 16, 4095, 4096), "f16_stream_kernelILi1EDF16_Lb0EE"),
                                       ((F16, 15, 16, 4095, 4095), "f16_stream_kernelILi1EDF16_Lb1EE"),
                                       ((F16, 15, 10, 4095, 4095), "f16_stream_kernelILi1EDF16_Lb1EE"),
                                       ((F16, 15, 9, 4095, 4095), "f16_stream_kernelILi1EDF16_Lb0EE"),
                                       ((F16, 15, 128, 4096, 4094), "f16_stream_kernelILi4EDF16_Lb0EE"),
                                       ((F16, 15, 128, 4096, 4095), "f16_stream_kernelILi4EDF16_Lb1EE")])
def test_odd_k_of_few_rows(kernel, call, name):
    assert name in kernel(*call)


# version 15 through registers or through copies and version 10
@pytest.mark.parametrize("call,name", [
    ((F16, 15, 1000, 1001, 999), "f16_any"),
    ((F16, 15, 500, 500, 12287), "f16_any"),       # few tiles: odd K up to 12288
    ((F16, 15, 500, 500, 12289), "f16_pp16"),
    ((F16, 15, 700, 700, 16385), "f16_any"),       # and 8 tiles of 256 x 256
    ((F16, 15, 5825, 33, 14805), "f16_any"),
    ((F16, 15, 500, 500, 16382), "f16_any"),       # even K up to 16384
    ((F16, 15, 500, 500, 16386), "f16_pp16"),
    ((F16, 15, 1987, 128, 17674), "f16_any"),
    ((F16, 15, 13398, 30, 17198), "f16_any"),
    ((F16, 15, 700, 697, 13312), "f16_any"),       # K a multiple of 8 up to 13312
    ((F16, 15, 700, 697, 13320), "f16_pp16"),
    ((F16, 15, 697, 700, 13320), "f16_any"),       # N up to M
    ((F16, 15, 14946, 29, 14024), "f16_any"),
    ((F16, 15, 300, 200, 1023), "f16_any"),        # fewer still: K up to 1024
    ((F16, 15, 300, 200, 4095), "f16_pp16"),
    ((F16, 15, 1000, 2001, 4096), "f16_any"),      # more tiles than CUs
    ((F16, 15, 2461, 411, 4608), "f16_any"),
    ((F16, 15, 2461, 411, 4616), "f16_pp16"),
    ((F16, 15, 2461, 412, 6144), "f16_any"),       # rows of B that start on dwords
    ((F16, 15, 2461, 412, 6152), "f16_pp16"),
    ((F16, 15, 413, 2535, 5584), "f16_any"),       # N above 2 M
    ((F16, 15, 2764, 365, 6144), "f16_any"),       # more than 21 of 256 x 256
    ((F16, 15, 2764, 365, 6152), "f16_pp16"),
    ((F16, 15, 365, 2764, 6152), "f16_any"),
    ((F16, 15, 16567, 35, 14450), "f16_any"),      # both copied
    ((F16, 15, 8000, 257, 3072), "f16_any"),       # two per CU
    ((F16, 15, 763, 3761, 2696), "f16_any"),
    ((F16, 15, 128, 50001, 1023), "f16_any"),      # half-empty 256 x 256 tiles
    ((F16, 15, 100000, 65, 513), "f16_any"),
    ((F16, 15, 100000, 65, 512), "f16_pp16"),
    ((F16, 15, 46840, 1, 688), "f16_pp16"),        # N below 8
    ((F16, 15, 46840, 1, 383), "f16_any"),
    ((F16, 15, 100000, 7, 128), "f16_pp16"),
    ((F16, 15, 100000, 7, 120), "f16_any"),
    ((F16, 15, 2000, 1, 688), "f16_any"),
    ((F16, 15, 2000, 1, 776), "f16_pp16"),
    ((F16, 15, 16000, 401, 512), "f16_pp16"),      # only B copied
    ((F16, 15, 236, 16964, 1024), "f16_any"),      # and its rows start on dwords
    ((F16, 15, 512, 4978, 3368), "f16_any"),
    ((F16, 15, 400, 15001, 512), "f16_any"),       # few rows
    ((F16, 15, 401, 15001, 264), "f16_pp16"),
    ((F16, 15, 3000, 1500, 1700), "f16_any"),      # even K
    ((F16, 15, 3000, 1500, 1281), "f16_pp16"),
    ((F16, 15, 3000, 1500, 1279), "f16_any"),
    ((F16, 15, 384, 14001, 1401), "f16_any"),      # narrow
    ((F16, 15, 14001, 384, 1401), "f16_any"),
    ((F16, 15, 14001, 385, 1401), "f16_pp16"),
    ((F16, 15, 11118, 1328, 21), "f16_any"),       # small K, one residency
    ((F16, 15, 281, 41448, 46), "f16_any"),
    ((F16, 15, 11118, 1328, 129), "f16_pp16"),
    ((F16, 15, 239, 74678, 144), "f16_any"),       # few rows
    ((F16, 15, 239, 74679, 144), "f16_pp16"),
    ((F16, 15, 50000, 305, 64), "f16_pp16"),
    ((F16, 15, 300, 50001, 130), "f16_any"),
    ((F16, 15, 1000, 8001, 1023), "f16_any"),      # two 128 x 128 tiles per CU
    ((F16, 15, 1500, 3001, 1801), "f16_pp16"),
    ((F16, 15, 50000, 304, 191), "f16_any"),       # few columns
    ((F16, 15, 50000, 304, 257), "f16_pp16"),
    ((F16, 15, 50000, 400, 65), "f16_pp16"),
    ((F16, 15, 300, 50000, 129), "f16_any"),       # few rows, aligned columns
    ((F16, 15, 300, 50001, 129), "f16_pp16"),
    ((F16, 15, 4096, 8192, 255), "f16_pp16"),
    ((F16, 15, 2049, 2051, 2052), "f16_pp16"),     # past 2^33
    ((F16, 15, 129, 9, 4097), "f16_pp16_sk"),
    ((F16, 15, 300, 201, 4095), "f16_pp16_sk"),
    ((F16, 15, 4000, 4001, 33), "f16_pp16_edge"),
    ((F16, 15, 4096, 4095, 1032), "f16_pp16_edge"),
])
def test_copies_of_version_15(kernel, call, name):
    assert name in kernel(*call)


# fp32 version 1 off its asm kernel: tile rows / 64, k-tile depth, k-tiles (0: any number, 3: any, N below 4)
@pytest.mark.parametrize("call,name", [
    ((F32, 1, 1000, 1001, 32), "f32_any_kernelILi1ELi32ELi1EE"),
    ((F32, 1, 1000, 1001, 33), "f32_any_kernelILi1ELi64ELi1EE"),
    ((F32, 1, 1000, 1001, 64), "f32_any_kernelILi1ELi64ELi1EE"),
    ((F32, 1, 1000, 1001, 65), "f32_any_kernelILi1ELi64ELi2EE"),
    ((F32, 1, 1000, 1001, 128), "f32_any_kernelILi1ELi64ELi2EE"),
    ((F32, 1, 1000, 1001, 129), "f32_any_kernelILi1ELi64ELi0EE"),
    ((F32, 1, 1000, 3, 129), "f32_any_kernelILi1ELi64ELi3EE"),
    ((F32, 1, 1000, 3, 128), "f32_any_kernelILi1ELi64ELi2EE"),
    ((F32, 1, 1990, 2047, 33), "f32_any_kernelILi2ELi32ELi0EE"),
])
def test_small_k_of_fp32_version_1(kernel, call, name):
    assert name in kernel(*call)


# few rows of fp32 version 3: small whole k-tiles, and a second round of column blocks from 33 rows, keep the tiles
@pytest.mark.parametrize("call,name", [
    ((F32, 3, 32, 16384, 64), "f32_mfma4"), ((F32, 3, 32, 16384, 80), "f32_stream"),
    ((F32, 3, 32, 16384, 128), "f32_stream"), ((F32, 3, 32, 20000, 96), "f32_mfma4"),
    ((F32, 3, 32, 32768, 64), "f32_stream"), ((F32, 3, 16, 16384, 64), "f32_mfma4"),
    ((F32, 3, 16, 20000, 64), "f32_stream"), ((F32, 3, 64, 262144, 64), "f32_mfma4"),
    ((F32, 3, 64, 262144, 96), "f32_stream"), ((F32, 3, 48, 262144, 64), "f32_stream"),
    ((F32, 3, 64, 16384, 4096), "f32_stream"), ((F32, 3, 64, 16388, 4096), "f32_mfma4"),
    ((F32, 3, 33, 32640, 1024), "f32_mfma4"), ((F32, 3, 33, 32644, 1024), "f32_stream"),
    ((F32, 3, 32, 20000, 4096), "f32_stream"),
])
def test_few_rows_of_fp32_version_3(kernel, call, name):
    assert name in kernel(*call)


# fp16 version 1: tile rows / 64, N or K below 8, C in whole rows
@pytest.mark.parametrize("call,name", [
    ((F16, 1, 32, 33, 40), "f16_any_kernelILi1EDF16_Lb0ELb1EE"),
    ((F16, 1, 31, 33, 40), "f16_any_kernelILi1EDF16_Lb0ELb0EE"),
    ((F16, 1, 32, 31, 40), "f16_any_kernelILi1EDF16_Lb0ELb0EE"),
    ((F16, 1, 33, 39, 7), "f16_any_kernelILi1EDF16_Lb1ELb1EE"),
    ((F16, 1, 64, 65603, 9), "f16_any_kernelILi2EDF16_Lb0ELb1EE"),
    ((F16, 1, 63, 65603, 9), "f16_any_kernelILi2EDF16_Lb0ELb0EE"),
    ((F16, 1, 70001, 65, 9), "f16_any_kernelILi2EDF16_Lb0ELb1EE"),
    ((F16, 1, 70001, 63, 9), "f16_any_kernelILi2EDF16_Lb0ELb0EE"),
    ((F16, 1, 4000, 4002, 9), "f16_any_kernelILi2EDF16_Lb0ELb0EE"),
    ((F16, 1, 4000, 4001, 9), "f16_any_kernelILi2EDF16_Lb0ELb1EE"),
])
def test_rows_of_c_in_fp16_version_1(kernel, call, name):
    assert name in kernel(*call)
