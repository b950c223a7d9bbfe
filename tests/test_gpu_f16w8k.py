"""GPU parity of the kernel that cuts K over a workgroup's waves for f16 x 8-bit weights (qmm_gemm_f16w8k.hip,
hip:gfx950:mfma_f16w8), under the bars of the kernel beside it: rows and columns that end inside a workgroup's blocks, waves
without a tile of 128 k, with an odd and an even number of them, every way scales and zero points are stored. Each case
asserts the shape its sizes take."""
import pytest

import onednn_amd as dnnl
from onednn_amd import _capi
from qmm_harness import dt
from test_gpu_f16w8 import F16W8, check, problem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    eng = dnnl.engine(dnnl.engine.kind.gpu, 0)
    return eng, dnnl.stream(eng)


CASES = {
    "rows32_two_tiles": (0x24, dict(M=257, K=256, N=1001)),
    "rows32_9_tiles_f32_add": (0x24, dict(M=270, K=1152, N=1031, dst_dt=dt.f32, post="add")),
    "rows48_17_tiles_swish": (0x34, dict(M=300, K=2176, N=2050, post="swish")),
    "rows48_3_tiles_s8_pitched": (0x34, dict(M=300, K=384, N=2050, wei_dt=dt.s8, zp_dt=dt.s8, lda=400)),
    "rows64_10_tiles_s8_u8_zero_points": (0x44, dict(M=263, K=1280, N=3043, wei_dt=dt.s8, zp_dt=dt.u8, dst_dt=dt.f32)),
    "rows32_common_zero_point_bf16_scales": (0x24, dict(M=321, K=640, N=2800, zp="common", scale_dt=dt.bf16)),
    "rows48_no_zero_point_common_scale_gelu": (0x34, dict(M=400, K=512, N=2570, zp=None, scale="common", post="gelu")),
    "rows64_no_scale_source_scale": (0x44, dict(M=263, K=512, N=3043, scale=None, src_scale=0.25, dst_dt=dt.f32)),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_f16w8k(ctx, name):
    print("[case] f16w8k %s" % name, flush=True)
    shape, kw = CASES[name]
    eng, strm = ctx
    assert _capi.lib().qmm_gemm_f16w8k_shape(kw["M"], kw["N"], kw["K"]) == shape
    p = problem(seed=60 + len(name), **kw)
    got, pd = p.run_gpu(eng, strm, weights_any=True, return_pd=True)
    assert pd.impl_info_str() == F16W8
    check(p, got, p.run_oracle(), name)
