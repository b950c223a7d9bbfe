"""Which kernel and which blocks int8 / fp8 products take: host work only."""
import collections

import pytest

from onednn_amd import _capi


@pytest.mark.parametrize("M,N", [(33, 1), (64, 32), (1024, 33), (16384, 64), (43008, 32), (97, 257), (300, 4096), (200, 1000), (1000, 225)])
def test_every_xcd_takes_an_eighth_of_the_blocks(M, N):
    lib = _capi.lib()
    rows, cols = (M + 31) // 32, (N + 31) // 32
    per_xcd, seen = collections.Counter(), set()
    for w in range(8 * ((rows * cols + 7) // 8)):
        b = lib.qmm_gemv_b8_block(M, N, w)
        if b >= 0:
            seen.add((b >> 32, b & 0xffffffff))
            per_xcd[w % 8] += 1
    assert seen == {(32 * r, c) for r in range(rows) for c in range(cols)} and sum(per_xcd.values()) == rows * cols
    assert max(per_xcd.values()) == (rows * cols + 7) // 8
    assert lib.qmm_gemv_b8_block(M, N, 8 * ((rows * cols + 7) // 8)) == -1


def test_blocks_of_a_column_share_an_xcd():
    lib = _capi.lib()
    xcds = collections.defaultdict(set)
    for w in range(8 * 32):  # 256 x 1024: 8 row blocks, 32 column blocks
        xcds[lib.qmm_gemv_b8_block(256, 1024, w) & 0xffffffff].add(w % 8)
    assert all(len(x) == 1 for x in xcds.values()) and len(xcds) == 32


def test_a_workgroup_outside_the_grid_has_nothing():
    lib = _capi.lib()
    assert lib.qmm_gemv_b8_block(32, 1024, 0) == -1 and lib.qmm_gemv_b8_block(64, 1024, -1) == -1
