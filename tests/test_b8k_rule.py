"""Which 8-bit products take the kernel whose waves cut K (qmm_gemm_b8k_shape): host work only. Times in us, the kernels
before / this one, measured on an MI355X: weights from HBM, in the entries below the first comment the geometric mean of
weights from HBM and in the caches."""
import pytest

from onednn_amd import _capi, memory

dt = memory.data_type


def shape(M, K, N, src=dt.s8, post_ops=0):
    return _capi.lib().qmm_gemm_b8k_shape(src, M, N, K, post_ops)


@pytest.mark.parametrize("M,K,N,want", [
    (64, 4096, 14336, 0x44),  # 24.1 / 20.0
    (16, 12288, 2048, 0x12),  # 15.7 / 15.3
    (195, 6912, 3296, 0x44),  # 28.7 / 18.4
    (256, 4096, 4096, 0x44),  # 19.7 / 14.9
    (1, 12032, 9248, 0x14),  # 28.1 / 25.9
    (1, 4096, 14336, 0),  # 14.2 / 15.1
    (894, 2944, 12624, 0),  # 61 / 108
    (16384, 1024, 128, 0),  # 13.7 / 16.9
    (4096, 4096, 14336, 0),
    # few k or many columns: the kernels of 256 rows
    (2059, 256, 768, 0),  # 10.8 / 14.2
    (74, 6016, 49408, 0),  # 84.0 / 121.0
    (86, 2688, 39168, 0),  # 42.8 / 55.2
    (403, 512, 3776, 0),  # 12.4 / 15.5
    (202, 3584, 8448, 0),  # 32.5 / 34.2
    (714, 1024, 2368, 0),  # 15.3 / 17.2
    # three rows of tiles that find their weights in L2
    (1851, 6656, 1216, 0),  # 48.2 / 56.3
    (1582, 6400, 1792, 0),  # 45.9 / 51.5
    (1169, 12544, 2560, 0x44),  # 84.9 / 75.6
    # what the streaming kernel requests at once, and where that is no gain
    (25, 1536, 21808, 0),  # 12.6 / 13.6
    (28, 1664, 117056, 0),  # 51 / 59
    (2, 3200, 65072, 0x14),  # 42 / 36
    # one row of workgroups
    (23, 3584, 124496, 0x22),  # in 32 x 64 results 99.5, so 86.1
    (56, 384, 126800, 0x44),  # in 32 x 32 results 69.4, so 60.0
])
def test_integers(M, K, N, want):
    assert shape(M, K, N) == want


@pytest.mark.parametrize("M,K,N,want", [
    (413, 12672, 3584, 0x44),  # 84 / 54
    (350, 8704, 1472, 0x24),  # 30 / 17.5
    (967, 8576, 4064, 0),  # 66 / 83
    (1, 4096, 14336, 0),  # 13.5 / 15.5
    (8192, 8192, 8192, 0),
    # few k: 256 x 256 tiles
    (65, 640, 62464, 0),  # 21.2 / 50.1
    (129, 768, 35584, 0),  # 24.8 / 51.5
    (1102, 640, 4608, 0),  # 20.6 / 45.3
    (204, 640, 18944, 0),  # 21.0 / 39.7
    (279, 1280, 16640, 0),  # 28.0 / 52.1
    (40, 384, 56928, 0),  # 21.4 / 27.1
    # rows that no L2 holds
    (1921, 7168, 1040, 0),  # 53.7 / 72.5
])
def test_fp8(M, K, N, want):
    assert shape(M, K, N, dt.f8_e4m3, 1) == want


def test_u8_sources():
    assert shape(256, 1024, 1024, dt.u8) == 0x22  # 6.4 / 5.9
    # the others' pre-pass pays over many tiles
    assert shape(1934, 14336, 4112, dt.u8, 1) == 0  # 184 / 284
    assert shape(404, 128, 3808, dt.u8) == 0x44  # 15.9 / 11.6


def test_other_arguments_take_nothing():
    assert not shape(64, 4160, 4096) and not shape(0, 4096, 4096) and not shape(64, 1 << 40, 4096)
    assert not shape(64, 4096, 4096, dt.f16)
