"""GPU parity of hip:gfx950:decode_w4 where scales and zero points are one per K group for all columns (mask 1 with groups):
every kernel behind the name steps from group to group by one entry there, not by a row of N. Zero points in nibbles then
lie two groups to a byte."""
import numpy as np
import pytest

import onednn_amd as dnnl
import test_gpu_parity as parity
from onednn_amd import _capi
from qmm_harness import dt
from test_gpu_g128 import check_16bit

pytestmark = pytest.mark.gpu
F, B = dict(act_dt=dt.f16), dict(act_dt=dt.bf16)
U8 = dict(wei_dt=dt.u8, zp_dt=dt.u8)


@pytest.fixture(scope="module")
def ctx():
    eng = dnnl.engine(dnnl.engine.kind.gpu, 0)
    return eng, dnnl.stream(eng)


# (runs with K cut over a workgroup's waves, problem)
CASES = {
    # the decode kernels: one, some and 16 rows, one column block a wave and several
    "f16_u4_1_row": (False, dict(M=1, K=512, N=272, **F)),
    "bf16_s4_5_rows": (False, dict(M=5, K=768, N=272, wei_dt=dt.s4, zp_dt=dt.s8, scale_dt=dt.bf16, **B)),
    "f16_u8_8_rows": (False, dict(M=8, K=512, N=320, **U8, **F)),
    "bf16_u4_16_rows": (False, dict(M=16, K=512, N=1040, zp_dt=dt.u8, **B)),
    "f16_u4_2_rows_wide": (False, dict(M=2, K=512, N=32768, **F)),
    "f16_u8_16_rows": (False, dict(M=16, K=640, N=1040, zp_group=128, G=128, **U8, **F)),
    # K cut over the waves
    "f16_u4_40_rows": (True, dict(M=40, K=512, N=2000, **F)),
    "bf16_s4_40_rows": (True, dict(M=40, K=1280, N=2000, wei_dt=dt.s4, zp_dt=dt.s8, zp_group=256, **B)),
    "f16_u8_40_rows": (True, dict(M=40, K=1024, N=1500, G=256, **U8, **F)),
    "bf16_u4_12_rows": (True, dict(M=12, K=512, N=9220, **B)),
    # tiles that walk all of K
    "f16_u4_tiles": (False, dict(M=1100, K=256, N=2048, **F)),
    "bf16_u4_tiles_zp_u8": (False, dict(M=1100, K=512, N=2048, zp_dt=dt.u8, G=256, zp_group=128, **B)),
}


@pytest.mark.parametrize("zero_points", ["grouped", "columns"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_one_scale_per_group_of_k(ctx, name, zero_points):
    print("[case] w4 group scales %s %s" % (name, zero_points), flush=True)
    eng, strm = ctx
    k_cut, kw = CASES[name]
    p = parity.decode_w4(seed=50 + len(name), **kw)
    M, N = kw["M"], kw["N"]
    bits = 8 if p.wei.dt == dt.u8 else 4
    assert bool(_capi.lib().qmm_gemm_w4k_shape(p.src.dt, bits, 0, M, N, kw["K"])) == k_cut
    _, code, groups, v = p.scales["wei"]
    p.scales["wei"] = (3, code, groups, np.repeat(v[:, 7:8] * np.linspace(0.5, 2, len(v))[:, None], N, 1))
    if zero_points == "grouped":
        _, zcode, zgroups, z = p.zps["wei"]
        p.zps["wei"] = (3, zcode, zgroups, np.repeat(z[:, 3:4] + np.arange(len(z))[:, None] % 3, N, 1))
    terms = parity.decode_term_scale(p)
    p.scales["wei"] = (1, code, groups, np.ascontiguousarray(p.scales["wei"][3][:, 0]))
    if zero_points == "grouped":
        p.zps["wei"] = (1, zcode, zgroups, np.ascontiguousarray(p.zps["wei"][3][:, 0]))
    got, pd = p.run_gpu(eng, strm, weights_any=True, return_pd=True)
    assert pd.impl_info_str() == parity.DECODE
    check_16bit(p, M, N, got, name, terms)
