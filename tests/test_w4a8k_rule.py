"""Which workgroups s8 activations under s4 weights with scales per 128 k take (qmm_gemm_w4a8k_shape): host work only.
Times in us, the kernels before / this one, measured
on an MI355X with weights in the caches (from HBM both are slower: 1 x 4096 x 14336 10.5 / 10.3)."""
import pytest

from onednn_amd import _capi, memory


@pytest.mark.parametrize("M,K,N,want", [
    (1, 4096, 14336, 0x14),  # 9.3 / 8.5
    (1, 13312, 1312, 0x12),  # 10.4 / 8.7
    (8, 4096, 4096, 0x12),  # 16.1 / 5.7
    (32, 4096, 14336, 0x24),  # 16.1 / 10.5
    (64, 12288, 2048, 0x12),  # 21.1 / 9.5
    (128, 12288, 2048, 0x14),  # 85.4 / 12.9
    (200, 12288, 2048, 0x24),  # 84.9 / 16.5
    (640, 12288, 2048, 0x34),  # 86.5 / 41.2
    (200, 4096, 14336, 0),  # 37.6 / 42.3
    (1000, 4096, 4096, 0),  # 37.5 / 57.9
    (1941, 4096, 14336, 0),  # 161.8 / 341.2
    (1267, 14336, 2768, 0),  # 106.0 / 128.1
])
def test_shape(M, K, N, want):
    assert _capi.lib().qmm_gemm_w4a8k_shape(M, N, K) == want


def test_up_to_64_rows_always():
    for M in (1, 4, 5, 16, 17, 32, 33, 64):
        for N in (1, 16, 1000, 4096, 128256):
            for K in (128, 1024, 14336):
                # (but a few rows of weights larger than the caches)
                assert bool(_capi.lib().qmm_gemm_w4a8k_shape(M, N, K)) == (M > 4 or N * K < 1 << 27)


def test_the_tall_tiles_tests_run_the_tall_tiles():
    """Sizes at which the kernel of qmm_gemm_g128.hip is tested stay with it."""
    f = _capi.lib().qmm_gemm_w4a8k_shape
    for M, N, K in ((129, 16650, 128), (193, 16642, 384), (700, 14330, 256), (640, 14336, 512), (1100, 3400, 128),
                    (1160, 7150, 128), (257, 14350, 256), (129, 16640, 256), (640, 16640, 256)):
        assert f(M, N, K) == 0 and _capi.lib().qmm_gemm_g128_rows(memory.data_type.s8, M, N, K)


def test_other_arguments_take_nothing():
    f = _capi.lib().qmm_gemm_w4a8k_shape
    assert not f(0, 1024, 1024) and not f(8, 1024, 1088) and not f(8, 1 << 40, 1024) and not f(8, 1024, 64)
