"""GPU parity of the kernel that cuts K over a workgroup's waves (qmm_gemm_w4k.hip): f16 / bf16 activations under 4- and
8-bit weights from 17 rows on, hip:gfx950:decode_w4. Row and column blocks that end inside a workgroup's, waves without
a tile, with an odd and an even number of them, every way scales and zero points are stored. Each case asserts the shape
its sizes take: the kernels beside this one carry the same implementation name."""
import numpy as np
import pytest

import onednn_amd as dnnl
import test_gpu_parity as parity
from onednn_amd import _capi
from qmm_harness import TensorSpec, dt
from test_gpu_g128 import check_16bit, pitched

pytestmark = pytest.mark.gpu
A = dnnl.algorithm
S22, S24, S34 = 0x22, 0x24, 0x34


@pytest.fixture(scope="module")
def ctx():
    eng = dnnl.engine(dnnl.engine.kind.gpu, 0)
    return eng, dnnl.stream(eng)


def run(ctx, p, shape):
    eng, strm = ctx
    (M, K), N = p.src.dims, p.wei.dims[1]
    bits = 8 if p.wei.dt in (dt.u8, dt.s8) else 4
    assert _capi.lib().qmm_gemm_w4k_shape(p.src.dt, bits, int(p.scales["wei"][2] is None), M, N, K) == shape
    got, pd = p.run_gpu(eng, strm, weights_any=True, return_pd=True)
    assert pd.impl_info_str() == parity.DECODE
    return got


F, B = dict(act_dt=dt.f16), dict(act_dt=dt.bf16)
U8 = dict(wei_dt=dt.u8, zp_dt=dt.u8)
CASES = {
    # one k tile (seven waves without any), one row past a block or short of it, columns past one
    "f16_u4_one_tile": (S22, dict(M=33, K=128, N=2046, **F)),
    "bf16_u4_one_tile_all_but_a_row": (S24, dict(M=63, K=128, N=4998, **B)),
    # 9 tiles: one wave has two; 17: one has three; groups wider than a tile, and other ones for the zero points
    "f16_s4_9_tiles_zp_groups": (S22, dict(M=40, K=1152, N=1362, wei_dt=dt.s4, zp_dt=dt.s8, G=128, zp_group=1152, **F)),
    "bf16_s4_17_tiles": (S22, dict(M=81, K=2176, N=1000, wei_dt=dt.s4, zp_dt=dt.s4, scale_dt=dt.bf16, **B)),
    "bf16_u4_many_rows_swish": (S24, dict(M=230, K=1920, N=1200, **B,
                                          post_ops=[{"kind": "eltwise", "alg": A.eltwise_swish, "alpha": 1.0}])),
    "f16_u4_48_rows": (S34, dict(M=217, K=1152, N=2460, zp_dt=dt.u8, G=128, **F)),
    "f16_u4_per_column_48_rows_f32": (S34, dict(M=200, K=1280, N=2450, per_column=True, dst_dt=dt.f32, **F)),
    "f16_u4_no_zero_points": (S22, dict(M=33, K=2048, N=1500, with_zp=False, **F)),
    "f16_s4_extreme_zero_points": (S22, dict(M=37, K=256, N=1040, wei_dt=dt.s4, zp_dt=dt.s8, **F)),
    # 8-bit weights: one scale per column (sums not folded), groups, both signs
    "f16_u8_per_column": (S22, dict(M=50, K=1280, N=1111, per_column=True, **U8, **F)),
    "f16_s8_per_column_48_rows": (S34, dict(M=149, K=2304, N=3930, wei_dt=dt.s8, zp_dt=dt.s8, per_column=True, **F)),
    "f16_u8_groups": (S22, dict(M=60, K=1024, N=1500, G=256, **U8, **F)),
    "f16_s8_groups_no_zero_points": (S22, dict(M=36, K=1024, N=1500, wei_dt=dt.s8, with_zp=False, **F)),
    "bf16_u8_per_column": (S22, dict(M=65, K=1024, N=1500, per_column=True, **U8, **B)),
    # 9 ... 16 rows: half of a block of 32 repeats the last row
    "f16_u4_9_rows": (S22, dict(M=9, K=1152, N=4100, **F)),
    "bf16_u4_16_rows": (S24, dict(M=16, K=1152, N=9220, **B)),
    "f16_u8_15_rows": (S22, dict(M=15, K=1280, N=4166, per_column=True, **U8, **F)),
    "bf16_s8_groups": (S22, dict(M=39, K=1024, N=2000, wei_dt=dt.s8, zp_dt=dt.s8, **B)),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_w4k(ctx, name):
    print("[case] w4k %s" % name, flush=True)
    shape, kw = CASES[name]
    p = parity.decode_w4(seed=900 + len(name), **kw)
    if "extreme" in name:
        _, code, groups, v = p.zps["wei"]
        p.zps["wei"] = (3, code, groups, np.where(np.arange(v.size) % 2 == 0, -128, 127).reshape(np.shape(v)))
    check_16bit(p, kw["M"], kw["N"], run(ctx, p, shape), name)


def test_pitched_rows_bias_and_binary(ctx):
    """Rows with a gap, an f32 mask added per result: the last block's rows and columns take their own operands."""
    print("[case] w4k pitched", flush=True)
    add = TensorSpec(dt.f32, [50, 1230], None, np.random.default_rng(3).standard_normal((50, 1230)) * 4)
    p = pitched(parity.decode_w4(50, 1024, 1230, 77, act_dt=dt.f16,
                                 post_ops=[{"kind": "binary", "alg": A.binary_add, "src1": add}]), 1096)
    check_16bit(p, 50, 1230, run(ctx, p, S22), "pitched")


def test_a_row_of_infinities_stays_a_row(ctx):
    """Rows share products' registers and LDS pieces, never sums."""
    print("[case] w4k infinities", flush=True)
    p = parity.decode_w4(40, 1024, 1200, 78, act_dt=dt.f16)
    a = p.src.logical().copy()
    clean = p.run_oracle().reshape(40, 1200).copy()
    a[39] = np.inf
    p.src.set(a)
    got = run(ctx, p, S22).reshape(40, 1200)
    import oracle as O
    g = O.to_f32(dt.f16, got[:39].reshape(-1)).astype(np.float64)
    w = O.to_f32(dt.f16, clean[:39].reshape(-1)).astype(np.float64)
    terms = parity.decode_term_scale(parity.decode_w4(40, 1024, 1200, 78, act_dt=dt.f16)).reshape(40, 1200)[:39].reshape(-1)
    assert np.all(np.abs(g - w) <= 2e-5 * terms + np.abs(w) * 2.0 ** -10)
    assert not np.isfinite(O.to_f32(dt.f16, got[39])).any()
