"""Which kernel 17 and more rows of f16 / bf16 activations take under 4- and 8-bit weights (qmm_gemm_w4f_tiled): host work
only. Times in us, the decode kernel once per 16 rows / the tiled one, measured on an MI355X."""
import pytest

from onednn_amd import _capi, memory

dt = memory.data_type


def tiled(M, K, N, bits=4, src=dt.f16):
    return bool(_capi.lib().qmm_gemm_w4f_tiled(src, bits, M, N, K))


@pytest.mark.parametrize("M,K,N,want", [
    # up to 4096 k a pass of the decode kernel takes the same time
    (20, 512, 12288, True),  # 29.1 / 7.9
    (24, 2048, 4096, False), (100, 1024, 4096, True),  # 29.7 / 15.2
    (50, 2048, 8192, True),  # 27.3 / 22.3
    (50, 4096, 8192, False),  # 29.3 / 36.3
    (100, 4096, 4096, False),  # 29.1 / 35.9
    (100, 4096, 6144, True),  # 43.9 / 36.0
    (20, 4096, 12288, True),  # 30.3 / 26.3
    # ... and past it more by another step
    (100, 4608, 4096, True),  # 53.8 / 39.5
    (200, 4608, 2560, True),  # 67.0 / 39.4
    (50, 5120, 8192, True),  # 48.8 / 43.3
    (100, 6144, 4096, True),  # 53.4 / 50.0
    (100, 8192, 4096, False),  # 53.5 / 63.9
    (20, 8192, 12288, False),  # 41.8 / 48.6
    (20, 8192, 16384, False),  # 43.5 / 49.3
    (50, 8192, 8192, False),  # 49.3 / 64.5
    (50, 11008, 8192, False),  # 67.0 / 84.0
    (20, 14336, 16384, False),  # 72.9 / 82.8
    (20, 14336, 10240, False),  # 58.1 / 82.1
    (100, 14336, 5120, True),  # 135.5 / 106.0
    # a last block of few rows; a second round of the tiled kernel
    (17, 8192, 12304, False),  # 40.6 / 48.8
    (18, 1408, 4480, False),  # 10.7 / 12.5
    (24, 1408, 4480, True),  # 12.6 / 12.1
    (33, 3840, 12336, True),  # 35.8 / 33.8
    (32, 8192, 43008, True),  # 132.7 / 96.5
    (24, 4096, 65536, True),  # 126.9 / 53.5
])
def test_4_bit_weights_under_f16(M, K, N, want):
    assert tiled(M, K, N) == want


@pytest.mark.parametrize("M,K,N,want", [
    (50, 1024, 8192, True),  # 26.0 / 18.1
    (50, 4096, 8192, False),  # 27.6 / 43.1
    (50, 8192, 8192, False),  # 48.1 / 76.7
    (50, 14336, 8192, False),  # 84.9 / 127.0
    (200, 6144, 2560, True),  # 68.4 / 59.5
    (200, 8192, 2560, False),  # 67.8 / 76.2
])
def test_4_bit_weights_under_bf16(M, K, N, want):
    assert tiled(M, K, N, src=dt.bf16) == want


@pytest.mark.parametrize("M,K,N,want", [
    (20, 1024, 12288, True),  # 27.3 / 12.9
    (24, 2048, 8192, False),  # 20.1 / 20.5
    (20, 4096, 12288, False),  # 29.0 / 35.9
    (20, 4096, 16384, True),  # 38.7 / 36.2
    (100, 4096, 4096, False),  # 36.5 / 47.9
    (100, 4608, 4096, True),  # 65.5 / 53.0
    (20, 8192, 12288, False),  # 54.0 / 66.5
    (50, 8192, 8192, False),  # 74.2 / 88.6
    (100, 14336, 4096, False),  # 129 / 148
    (200, 11008, 3072, True),  # 144 / 116
    (18, 3840, 12336, False),  # 31.2 / 34.5
    (28, 3840, 12336, True),  # 36.1 / 34.1
])
def test_8_bit_weights(M, K, N, want):
    assert tiled(M, K, N, 8) == want


def test_other_arguments_take_nothing():
    assert not tiled(16, 1024, 65536) and not tiled(0, 1024, 1024) and not tiled(100, 1024, 4096, 2)
    assert not tiled(100, 1024, 4096, src=dt.s8) and not tiled(100, 1 << 40, 4096)
