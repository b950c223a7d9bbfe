"""Which kernel and which blocks int8 / fp8 products take: host work only."""
import collections

import pytest

from onednn_amd import _capi


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
