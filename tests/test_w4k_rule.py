"""Which workgroups 17 and more rows of f16 / bf16 activations take under 4- and 8-bit weights (qmm_gemm_w4k_shape): host
work only. Times in us, the kernels that walk K in one chain / this one, measured on an MI355X."""
import pytest

from onednn_amd import _capi, memory

dt = memory.data_type


def shape(M, K, N, bits=4, src=dt.f16, per_column=0):
    return _capi.lib().qmm_gemm_w4k_shape(src, bits, per_column, M, N, K)


@pytest.mark.parametrize("M,K,N,want", [
    (164, 6528, 3552, 0x34),  # 54.3 / 19.4
    (64, 4096, 4096, 0x22),  # 20.2 / 8.3
    (89, 4480, 4304, 0x24),  # 39.4 / 11.3
    (563, 2048, 1248, 0x34),  # 22.7 / 11.5
    (33, 1280, 1408, 0x22),  # 8.1 / 5.1
    (30, 3584, 1072, 0),  # 6.7 / 7.1
    (19, 7040, 1536, 0),  # 8.5 / 10.0
    (925, 3840, 3024, 0),  # 57.3 / 60.9
    (1000, 4096, 14336, 0),  # 159 / 276
    (488, 1152, 6464, 0),  # 26.6 / 33.6
    (33, 256, 65544, 0), (16, 4096, 4096, 0), (64, 4160, 4096, 0),
])
def test_4_bit_weights_under_f16(M, K, N, want):
    assert shape(M, K, N) == want


@pytest.mark.parametrize("M,K,N,want", [
    (204, 12928, 2176, 0x24),  # 110.8 / 25.0
    (48, 11904, 3712, 0x22),  # 38.7 / 16.8
    (711, 9088, 3520, 0x24),  # 131.1 / 102.4
    (1310, 3968, 1488, 0),  # 45.3 / 51.8
    (361, 10112, 16288, 0),  # 188.8 / 240.4
    (1324, 13824, 2544, 0),  # 191.4 / 219.1
    (400, 6784, 9872, 0x24),  # 134.7 / 114.2
])
def test_4_bit_weights_under_bf16(M, K, N, want):
    assert shape(M, K, N, src=dt.bf16) == want


@pytest.mark.parametrize("M,K,N,want", [
    (148, 12800, 1424, 0x22),  # 76.9 / 19.0
    (112, 10880, 3664, 0x24),  # 104.9 / 27.1
    (68, 11008, 7488, 0x34),  # 118.7 / 32.9
    (20, 3968, 1760, 0),  # 7.3 / 8.5
])
def test_8_bit_weights(M, K, N, want):
    assert shape(M, K, N, 8, per_column=1) == want


def test_groups_of_8_bit_weights_take_no_tall_tile():
    assert shape(68, 11008, 7488, 8) in (0x22, 0x24) and shape(68, 11008, 7488, 8, dt.bf16, 1) in (0x22, 0x24)


def test_other_arguments_take_nothing():
    assert shape(0, 1024, 1024) == 0 and shape(100, 1024, 4096, 2) == 0 and shape(100, 1024, 4096, src=dt.s8) == 0
    assert shape(100, 1 << 40, 4096) == 0


@pytest.mark.parametrize("M,K,N,bits,src,want", [
    (16, 1280, 4160, 8, dt.f16, 0x22),  # 13.1 / 6.1
    (14, 8704, 11712, 8, dt.f16, 0x24),  # 45.5 / 27.9
    (15, 3456, 5408, 4, dt.f16, 0x22),  # 11.7 / 7.8
    (12, 2432, 12432, 4, dt.bf16, 0x24),  # 17.5 / 9.3
    (14, 7808, 3440, 4, dt.f16, 0),  # 9.9 / 11.5
    (8, 4096, 14336, 4, dt.f16, 0), (9, 4096, 4096, 8, dt.f16, 0),
    # very wide 4-bit weights with few k: the tall tiles
    (10, 128, 95648, 4, dt.bf16, 0),  # 10.3 / 21.6
    (10, 256, 76352, 4, dt.bf16, 0),  # 12.2 / 19.2
    (15, 512, 78560, 4, dt.bf16, 0),  # 18.0 / 21.9
    (12, 512, 69472, 4, dt.f16, 0),  # 16.7 / 19.9
    (16, 256, 65590, 4, dt.bf16, 0),
])
def test_9_to_16_rows(M, K, N, bits, src, want):
    assert shape(M, K, N, bits, src, per_column=bits == 8) == want
