"""Which kernel and which blocks int8 / fp8 products take: host work only. Times in us, measured on an MI355X."""
import collections

import pytest

from onednn_amd import _capi, memory

dt = memory.data_type


def tile(code, M, K, N, batch=1, post_ops=0):
    return _capi.lib().qmm_gemm_b8_tile(code, batch, M, N, K, post_ops)


@pytest.mark.parametrize("M,K,N,post_ops,want", [
    # 64 x 64 tiles / the streaming kernel
    (256, 1024, 2048, 1, 32),  # 10.4 / 7.6
    (256, 1024, 2816, 1, 64),  # 10.3 / 11.4
    (256, 2048, 2816, 1, 32),  # 13.0 / 11.9
    (256, 2048, 3552, 1, 64),  # 12.9 / 14.3
    (226, 3712, 3552, 1, 64),  # 18.4 / 19.2
    (226, 4096, 3552, 0, 32),  # 19.8 / 18.3
    (226, 1024, 3552, 0, 64),  # 10.4 / 11.6
    (128, 8192, 8000, 0, 64),  # 32.5 / 36.6
    (2000, 1024, 288, 0, 64),  # 9.9 / 11.6
    # as they were
    (64, 4096, 14336, 0, 32), (256, 1024, 1024, 1, 32), (256, 4096, 4096, 0, 32), (384, 4096, 4096, 0, 256),
    (300, 1024, 4096, 0, 128), (4096, 4096, 14336, 1, 256),
])
def test_s8(M, K, N, post_ops, want):
    assert tile(dt.s8, M, K, N, 1, post_ops) == want


@pytest.mark.parametrize("M,K,N,want", [
    # tiles / the streaming kernel
    (33, 4096, 16384, 32),  # 31.1 / 22.9
    (64, 4096, 24576, 32),  # 36.8 / 33.7
    (64, 8192, 24576, 32),  # 69.1 / 62.2
    (33, 14336, 24576, 128),  # 97.8 / 114.1
    (33, 4096, 32768, 128),  # 34.6 / 41.5
    (64, 14336, 32768, 128),  # 113.9 / 150.1
    (100, 4096, 16384, 32),  # 37.7 / 36.8
    (100, 6144, 16384, 128),  # 46.0 / 55.9
    (32, 14336, 65536, 32), (16, 64, 64, 32),
    (226, 1024, 3552, 64),  # 10.2 / 12.1
    (384, 2048, 1800, 32),  # 13.1 / 11.7
    (226, 2048, 3552, 64),  # 12.9 / 13.2
])
def test_fp8_few_results(M, K, N, want):
    assert tile(dt.f8_e4m3, M, K, N) == want


@pytest.mark.parametrize("batch,M,K,N,want", [
    # tiles of 128 (below 64 of them: 64) / 256 x 256
    (2, 128, 512, 1024, 64),  # 8.2 / 18.0
    (2, 128, 2048, 1024, 64),  # 12.8 / 28.6
    (32, 128, 1024, 128, 64),  # 9.2 / 19.7
    (3, 500, 1024, 520, 64),  # 10.8 / 48.2
    (8, 16, 512, 1024, 128),  # 9.6 / 14.6
    (64, 200, 512, 256, 128),  # 24.6 / 44.0
    (40, 256, 1024, 512, 128),  # 31.7 / 49.8
    (4, 500, 2048, 2048, 128),  # 30.4 / 39.8
    (8, 64, 512, 1024, 256),  # 19.1 / 14.6
    (12, 384, 2048, 1024, 256),  # 43.5 / 33.3
    (16, 64, 2048, 4096, 256),  # 41.6 / 37.8
    (8, 128, 4096, 1024, 128),  # 37.8 / 44.4
    # one matrix
    (1, 1500, 4096, 3000, 128),  # 42.4 / 67.0
    (1, 512, 8192, 8192, 128),  # 55.2 / 75.3
    (1, 1024, 4096, 4096, 128),  # 38.9 / 45.9
    (1, 2048, 4096, 4096, 256),  # 51.5 / 47.4
    (1, 1152, 1024, 6144, 256),  # 26.9 / 24.0
    (1, 1000, 2048, 6144, 128),  # 32.5 / 37.3
    (1, 700, 8192, 14336, 256),  # 124.8 / 87.7
    (1, 1746, 2048, 5856, 128),  # 44.0 / 52.7
    (1, 1746, 8192, 5856, 256),  # 113.2 / 96.8
    (1, 100, 8192, 43008, 256),  # 110.5 / 98.3
    (1, 33, 2048, 32768, 128),  # 23.6 / 30.7
    (1, 256, 1024, 2816, 64),  # 9.8, streaming 11.7
    (1, 256, 2048, 2816, 32),  # 12.6, streaming 11.8
    (1, 256, 2048, 3584, 64),  # 12.6, streaming 13.6
    (1, 8192, 8192, 8192, 256),
])
def test_fp8_tiles(batch, M, K, N, want):
    assert tile(dt.f8_e4m3, M, K, N, batch) == want


def test_other_arguments_take_nothing():
    assert tile(dt.f32, 64, 64, 64) == 0 and tile(dt.s8, 0, 64, 64) == 0 and tile(dt.s8, 64, 40, 64) == 0


def blocks(M, N):
    lib = _capi.lib()
    rows, cols = (M + 31) // 32, (N + 31) // 32
    end = rows * (cols // 8 * 8 + 8)
    found = [(w, lib.qmm_gemv_b8_block(M, N, w)) for w in range(end)]
    assert lib.qmm_gemv_b8_block(M, N, end) == -1
    return [(w, b >> 32, b & 0xffffffff) for w, b in found if b >= 0]


@pytest.mark.parametrize("M,N", [(33, 1), (64, 32), (1024, 33), (16384, 64), (43008, 32), (97, 257), (300, 4096), (200, 1000),
                                 (992, 225), (993, 225), (2000, 288)])
def test_every_block_once(M, N):
    found = blocks(M, N)
    assert sorted((r, c) for _, r, c in found) == [(r, c) for r in range(0, M, 32) for c in range((N + 31) // 32)]
    per_xcd = collections.Counter(w % 8 for w, _, _ in found)
    if M > 992:  # 32 row blocks and more: every XCD an eighth
        assert max(per_xcd.values()) == (len(found) + 7) // 8


def test_blocks_of_a_column_share_an_xcd():
    lib = _capi.lib()
    xcds = collections.defaultdict(set)
    for w in range(8 * 32):  # 256 x 1024: 8 row blocks, 32 column blocks
        xcds[lib.qmm_gemv_b8_block(256, 1024, w) & 0xffffffff].add(w % 8)
    assert all(len(x) == 1 for x in xcds.values()) and len(xcds) == 32


def test_a_workgroup_outside_the_grid_has_nothing():
    lib = _capi.lib()
    assert lib.qmm_gemv_b8_block(32, 1024, 0) == -1 and lib.qmm_gemv_b8_block(64, 1024, -1) == -1
