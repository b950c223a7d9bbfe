"""How attention over few queries is cut over the keys, seen from the scratchpad that a primitive asks for (host work
only): several ranges leave their states there for a second, combining launch; one range needs none."""
import os

import pytest

os.environ.setdefault("DNNL_AMD_DESCRIPTOR_ONLY", "1")

import onednn_amd as dnnl  # noqa: E402
from onednn_amd import memory  # noqa: E402

dt, tag = memory.data_type, memory.format_tag


def scratch_bytes(batch, heads, kv_heads, queries, keys, D, code=dt.f16, cache=None):
    eng = dnnl.engine(dnnl.engine.kind.gpu, 0)
    T = lambda name: 2 + tag._plain.index(name)  # noqa: E731
    attr = dnnl.primitive_attr()
    attr.set_scratchpad_mode(dnnl.scratchpad_mode.user)
    q = memory.desc([batch, heads, queries, D], code, T("abcd"))
    kt = memory.desc([batch, kv_heads, D, keys], cache or code, T("abdc"))
    v = memory.desc([batch, kv_heads, keys, D], cache or code, T("abcd"))
    side = [None, None]
    if cache:
        for i, groups in enumerate(([D, 1], [1, D])):
            side[i] = dnnl.primitive_attr()
            side[i].set_scales(dnnl.DNNL_ARG_WEIGHTS, 0b1111, groups, dt.f16)
    pd = dnnl.sdpa.primitive_desc(eng, q, kt, v, None, code, q, False, kv_heads, False, attr, *side)
    md = pd.scratchpad_desc()
    return 0 if md.is_zero() else md.get_size()


@pytest.mark.parametrize("batch,heads,kv_heads", [(1, 32, 32), (1, 32, 8), (16, 32, 1), (16, 32, 4), (64, 32, 8)])
@pytest.mark.parametrize("D,keys", [(32, 512), (64, 512), (96, 256), (128, 256), (256, 128)])
def test_few_keys_are_one_range(batch, heads, kv_heads, D, keys):
    # 32 keys a tile, four waves: however few workgroups the packed heads leave
    assert scratch_bytes(batch, heads, kv_heads, 1, keys, D) == 0
    # past that, several ranges unless the packed heads fill the chip twice by themselves
    assert (scratch_bytes(batch, heads, kv_heads, 1, keys + 1, D) > 0) == (batch * kv_heads < 512)


def test_an_8_bit_cache_without_packed_dequantization_is_cut_earlier():
    assert scratch_bytes(1, 32, 8, 1, 256, 64, dt.bf16, dt.s8) == 0
    assert scratch_bytes(1, 32, 8, 1, 257, 64, dt.bf16, dt.s8) > 0
    assert scratch_bytes(1, 32, 8, 1, 256, 32, dt.bf16, dt.s8) == 0
    assert scratch_bytes(1, 32, 8, 1, 512, 32, dt.bf16, dt.s8) > 0
    assert scratch_bytes(1, 32, 8, 1, 129, 128, dt.bf16, dt.s8) > 0
    assert scratch_bytes(1, 32, 8, 1, 256, 128, dt.f16, dt.s8) == 0


@pytest.mark.parametrize("D,one,three", [(64, 384, 896), (96, 512, 1280), (128, 640, 1664), (256, 1152, 3200)])
def test_states_lie_on_lines_of_their_own(D, one, three):
    # 20 tiles, five ranges; per query D accumulators, maximum and sum; a range's, up to whole 128-byte lines
    assert scratch_bytes(1, 1, 1, 1, 640, D) == 5 * one
    assert scratch_bytes(2, 4, 2, 3, 640, D) == 2 * 4 * 5 * three
