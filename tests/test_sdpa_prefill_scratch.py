"""The scratchpad that attention over an 8-bit cache asks for: room for the cache in 16 bits where it is written there
first (many queries and keys, no explicit mask, head size 64 or 128), nothing elsewhere (host work only)."""
import os

import pytest

os.environ.setdefault("DNNL_AMD_DESCRIPTOR_ONLY", "1")

import onednn_amd as dnnl  # noqa: E402
from onednn_amd import memory  # noqa: E402

dt, tag = memory.data_type, memory.format_tag


@pytest.mark.parametrize("queries,keys,D,cache,masked,want", [
    (257, 300, 64, dt.s8, False, True), (256, 300, 64, dt.s8, False, False), (4096, 161, 128, dt.u8, False, True),
    (4096, 1, 128, dt.u8, False, False),  # few keys: dequantized while staging (257 queries x 16 keys 8.3 us, through the scratchpad 18.1)
    (300, 300, 96, dt.s8, False, False), (300, 300, 64, dt.f16, False, False), (300, 300, 64, dt.s8, True, False),
    (300, 1 << 17, 128, dt.s8, False, True), (300, (1 << 17) + 1, 128, dt.s8, False, False)])
def test_room_for_the_cache(queries, keys, D, cache, masked, want):
    eng = dnnl.engine(dnnl.engine.kind.gpu, 0)
    T = lambda name: 2 + tag._plain.index(name)  # noqa: E731
    attr = dnnl.primitive_attr()
    attr.set_scratchpad_mode(dnnl.scratchpad_mode.user)
    q = memory.desc([1, 8, queries, D], dt.f16, T("abcd"))
    kt = memory.desc([1, 4, D, keys], cache, T("abdc"))
    v = memory.desc([1, 4, keys, D], cache, T("abcd"))
    mask = memory.desc([1, 1, queries, keys], dt.f16, T("abcd")) if masked else None
    pd = dnnl.sdpa.primitive_desc(eng, q, kt, v, mask, dt.f16, q, False, 4, False, attr)
    md = pd.scratchpad_desc()
    assert (0 if md.is_zero() else md.get_size()) == (2 * 4 * keys * D * 2 if want else 0)


def test_a_primitive_is_created_without_room_for_the_cache():
    """The room only makes the launch faster: where it cannot be had (no device here, no memory elsewhere) the primitive
    is created all the same. The ranges of few queries need theirs."""
    eng = dnnl.engine(dnnl.engine.kind.gpu, 0)
    T = lambda name: 2 + tag._plain.index(name)  # noqa: E731

    def create(queries, keys, cache):
        q = memory.desc([1, 8, queries, 64], dt.f16, T("abcd"))
        pd = dnnl.sdpa.primitive_desc(eng, q, memory.desc([1, 8, 64, keys], cache, T("abdc")),
                                      memory.desc([1, 8, keys, 64], cache, T("abcd")), None, dt.f16, q, False, 8, False)
        return dnnl.sdpa(pd)

    create(300, 400, dt.s8)
    if eng_has_no_device():
        with pytest.raises(dnnl.error):
            create(1, 4096, dt.f16)


def eng_has_no_device():
    import torch
    return not torch.cuda.is_available()
