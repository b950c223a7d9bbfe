"""Which f16 x 8-bit-weights products take the kernel whose waves cut K (qmm_gemm_f16w8k_shape): host work only. Times in us,
256 x 256 tiles / this kernel, measured on an MI355X."""
import pytest

from onednn_amd import _capi


@pytest.mark.parametrize("M,K,N,want", [
    (263, 1280, 3040, 0x44),  # 43.4 / 12.6
    (300, 1024, 1168, 0x24),  # 38.7 / 7.7
    (424, 2816, 5344, 0x34),  # 63.3 / 39.8
    (614, 1664, 10400, 0),  # 56.0 / 70.2
    (1922, 2304, 2864, 0),  # 62.9 / 82.2
    (4096, 1024, 1024, 0),  # 36.3 / 42.4
    (3000, 1024, 1024, 0x44),  # 42.8 / 32.1
    # long rows that no L2 holds
    (1473, 14464, 1344, 0),  # 106.3 / 124.2
    (2102, 9216, 816, 0),  # 74.9 / 80.9
    (885, 12160, 1472, 0x34),  # 90.3 / 69.3
    # columns in multiples of 128, which the tiles store faster
    (331, 256, 8960, 0),  # 21.8 / 23.8
    (1283, 512, 2816, 0),  # 25.7 / 27.5
    (1031, 640, 3840, 0),
    (344, 256, 12528, 0x44),  # with a swish 87 / 38
    (2176, 4096, 14336, 0), (300, 1056, 1168, 0), (0, 1024, 1168, 0), (300, 1 << 40, 1168, 0),
])
def test_shape(M, K, N, want):
    assert _capi.lib().qmm_gemm_f16w8k_shape(M, N, K) == want
