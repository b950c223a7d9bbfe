"""The sizes that the tiled kernel for 4-bit weights with groups of 128 k takes (qmm_gemm_g128_rows): host work only.

Times in us, the other kernels / the tiled one, 4096 k unless said otherwise, measured on an MI355X."""
import pytest

from onednn_amd import _capi, memory

dt = memory.data_type


def rows(code, M, N, K):
    return _capi.lib().qmm_gemm_g128_rows(code, M, N, K)


@pytest.mark.parametrize("code", [dt.f16, dt.bf16], ids=["f16", "bf16"])
@pytest.mark.parametrize("M,N,K,taken", [
    # more than 65536 columns: one row of tiles is past the block count from which the kernel is worth it
    (1, 128256, 4096, False),  # 49 / 84
    (8, 128256, 4096, False),  # 74 / 85
    (16, 128256, 4096, True),  # 119 / 87
    (32, 128256, 4096, True),  # 109 / 91
    (1, 65552, 4096, False),  # 28 / 83
    (16, 65552, 4096, False),  # 69 / 84
    (33, 65552, 4096, True),  # 121 / 87
    (1, 262144, 8192, False),  # 185 / 339
    (1, 128256, 1024, True),  # 39 / 25
    (16, 65552, 1024, True),  # 73 / 26
    # up to 65536 columns: the block count alone
    (1, 16384, 4096, False), (64, 65536, 4096, False), (65, 32800, 4096, True), (256, 16384, 4096, False),
    (257, 14336, 4096, True),
])
def test_rows_and_columns_from_which_16bit_activations_take_it(code, M, N, K, taken):
    assert (rows(code, M, N, K) > 0) == taken


@pytest.mark.parametrize("M,N,tile", [(64, 128256, 0), (65, 128256, 128), (129, 16650, 64), (128, 16384, 0), (640, 14336, 128)])
def test_s8_tiles(M, N, tile):
    assert rows(dt.s8, M, N, 4096) == tile


def test_other_arguments_take_nothing():
    assert rows(dt.f32, 4096, 4096, 4096) == 0
    assert rows(dt.f16, 0, 1 << 20, 4096) == 0
    assert rows(dt.f16, 1 << 40, 1 << 20, 4096) == 0
