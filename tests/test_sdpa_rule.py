"""Which of the two attention kernels takes more than 16 queries without an explicit mask (qmm_sdpa_pipelined): host work
only. Times in us, the kernel of 32-key tiles / the pipelined one, measured on an MI355X."""
import pytest

from onednn_amd import _capi


def pipelined(D, causal, heads, queries, keys, kv=None, cache=False):
    return bool(_capi.lib().qmm_sdpa_pipelined(D, causal, heads, kv or heads, queries, keys, cache))


@pytest.mark.parametrize("D,causal,heads,queries,keys,taken", [
    # at most one workgroup to a CU
    (64, 0, 8, 512, 96, False),  # 6.6 / 7.1
    (64, 0, 8, 512, 128, True),  # 7.4 / 6.8
    (128, 0, 32, 512, 64, False),  # 8.3 / 8.6
    (128, 0, 32, 512, 128, True),  # 10.7 / 9.6
    (64, 1, 256, 32, 32, False),  # 5.3 / 5.8
    (64, 1, 256, 64, 64, True),  # 6.5 / 6.0
    # two
    (64, 0, 32, 2048, 320, False),  # 16.2 / 17.2
    (64, 0, 32, 2048, 512, True),  # 22.4 / 21.0
    (64, 1, 256, 256, 256, False),  # 13.7 / 16.8
    (64, 1, 128, 512, 512, True),  # 20.0 / 18.4
    (128, 0, 32, 2048, 256, False),  # 22.5 / 24.4
    (128, 0, 32, 2048, 512, True),  # 34.8 / 33.3
    (128, 1, 512, 128, 128, False),  # 18.0 / 23.7
    (128, 1, 32, 2048, 2048, True),  # 84.9 / 50.1
    # three and more
    (64, 1, 128, 700, 700, False),  # 26.4 / 29.8
    (64, 1, 32, 3000, 3000, True),  # 82.3 / 69.4
    (64, 0, 64, 4096, 32, False),  # 18.2 / 42.1
    (64, 0, 64, 4096, 1024, False),  # 119.7 / 124.0
    (64, 0, 64, 4096, 2048, True),  # 226 / 219
    (64, 1, 512, 512, 512, False),  # 50.7 / 72.1
    (64, 1, 256, 2048, 2048, False),  # 270 / 289
    (64, 1, 128, 4096, 4096, True),  # 470 / 462
    (128, 1, 256, 512, 512, False),  # 46.7 / 61.5
    (128, 1, 64, 2048, 2048, True),  # 109 / 100
    (128, 0, 64, 4096, 700, False),  # 150 / 157
    (128, 0, 64, 4096, 1500, True),  # 288 / 268
])
def test_keys_from_which_the_pipelined_kernel_takes_16_bit_values(D, causal, heads, queries, keys, taken):
    assert pipelined(D, causal, heads, queries, keys) == taken


@pytest.mark.parametrize("D,causal,heads,kv,queries,keys,taken", [
    (64, 0, 8, 8, 256, 4096, False), (128, 0, 32, 8, 257, 16, False),  # 8.3 / 18.1
    (64, 0, 8, 8, 300, 256, False),  # 14.6 / 15.3
    (64, 0, 8, 8, 300, 300, True),  # 17.6 / 16.8
    (64, 1, 128, 32, 400, 400, False),  # 24.3 / 25.2
    (64, 1, 128, 32, 600, 600, True),  # 38.2 / 33.7
    (64, 1, 256, 64, 900, 900, False),  # 92 / 102
    (64, 0, 64, 8, 4096, 384, False),  # 67.9 / 74.2
    (64, 0, 64, 8, 4096, 512, True),  # 85.0 / 84.3
    (128, 0, 32, 8, 300, 150, False),  # 17.1 / 19.2
    (128, 0, 32, 8, 300, 200, True),  # 21.4 / 19.7
    (128, 0, 64, 8, 4096, 128, False),  # 72.8 / 76.0
    (128, 1, 8, 8, 257, 257, True),  # 24.1 / 18.3
])
def test_keys_from_which_an_8_bit_cache_is_dequantized_first(D, causal, heads, kv, queries, keys, taken):
    assert pipelined(D, causal, heads, queries, keys, kv, True) == taken


def test_fewer_keys_than_queries():
    # a causal mask over fewer keys: most workgroups walk all of them
    assert not pipelined(64, 1, 64, 4096, 256) and pipelined(64, 1, 64, 8192, 2560)


def test_other_arguments_take_nothing():
    assert not pipelined(96, 0, 8, 512, 512) and not pipelined(64, 0, 8, 16, 512)
    assert not pipelined(64, 0, 8, 512, 0) and not pipelined(64, 0, 8, 512, 1 << 40) and not pipelined(64, 0, 9, 512, 512, 4)
    assert not pipelined(128, 0, 8, 512, 1 << 23)  # byte offsets in a head past 31 bits
