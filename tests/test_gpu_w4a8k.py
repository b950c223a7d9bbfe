"""GPU parity of the kernel that cuts K over a workgroup's waves for s8 activations x s4 weights (qmm_gemm_w4a8k.hip,
hip:gfx950:mfma_w4a8): rows and columns that end inside a workgroup's blocks, waves without a group, with an odd and an
even number of them, scales without rows or columns, pitched rows, huge scales. Power-of-two scales: bit for bit. Each
case asserts the shape its sizes take: the kernels beside this one carry the same implementation name."""
import numpy as np
import pytest

import onednn_amd as dnnl
import oracle as O
from onednn_amd import _capi
from qmm_harness import TensorSpec, assert_bit_exact, assert_f32_close, dt
from test_gpu_g128 import pitched
from test_gpu_w4a8 import W4A8, dynamic_quant

pytestmark = pytest.mark.gpu
A = dnnl.algorithm


@pytest.fixture(scope="module")
def ctx():
    eng = dnnl.engine(dnnl.engine.kind.gpu, 0)
    return eng, dnnl.stream(eng)


def run(ctx, p, shape):
    eng, strm = ctx
    (M, K), N = p.src.dims, p.wei.dims[1]
    assert _capi.lib().qmm_gemm_w4a8k_shape(M, N, K) == shape
    got, pd = p.run_gpu(eng, strm, weights_any=True, return_pd=True)
    assert pd.impl_info_str() == W4A8
    return got


CASES = {
    # one group (seven waves without any); one row
    "one_group": (0x12, dict(M=1, K=128, N=34)),
    # 9 groups: a wave has two; 17: one has three, the others two
    "rows16_9_groups": (0x12, dict(M=16, K=1152, N=162, scale_dt=dt.bf16)),
    "rows17_17_groups": (0x12, dict(M=17, K=2176, N=1090)),
    # 64 columns, a last block of 16 columns of which two are there
    "cols64_m5": (0x14, dict(M=5, K=1280, N=14338, dst_dt=dt.f16)),
    "cols64_m33": (0x14, dict(M=33, K=256, N=4098)),
    "rows32_m63": (0x24, dict(M=63, K=1664, N=5650)),
    "rows32_m97": (0x24, dict(M=97, K=1152, N=4002)),
    "rows48_m145": (0x34, dict(M=145, K=1152, N=4002)),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_exact(ctx, name):
    print("[case] w4a8k %s" % name, flush=True)
    shape, kw = CASES[name]
    p = dynamic_quant(seed=700 + len(name), exact=True, **kw)
    assert_bit_exact(run(ctx, p, shape), p.run_oracle(), name)


@pytest.mark.parametrize("wei_mask,src_mask,pitch", [(1, 3, 256), (3, 2, 256), (1, 2, 272), (3, 3, 320)])
def test_scales_without_columns_or_rows_and_pitched_source(ctx, wei_mask, src_mask, pitch):
    print("[case] w4a8k masks %d %d pitch %d" % (wei_mask, src_mask, pitch), flush=True)
    p = pitched(dynamic_quant(35, 256, 1094, 31, exact=True), pitch)
    _, code, groups, v = p.scales["wei"]
    p.scales["wei"] = (wei_mask, code, groups, v if wei_mask == 3 else np.ascontiguousarray(v[:, 3]))
    _, code, groups, v = p.scales["src"]
    p.scales["src"] = (src_mask, code, groups, v if src_mask == 3 else np.ascontiguousarray(v[5]))
    assert_bit_exact(run(ctx, p, 0x12), p.run_oracle(), "masks")


def test_extreme_sums(ctx):
    print("[case] w4a8k extremes", flush=True)
    p = dynamic_quant(20, 256, 1040, 7, exact=True)
    p.src.set(np.full((20, 256), -128.0))
    p.wei.set(np.where(np.arange(1040) % 2 == 0, -8.0, 7.0)[None].repeat(256, 0))
    assert_bit_exact(run(ctx, p, 0x12), p.run_oracle(), "extremes")


@pytest.mark.parametrize("name", ["bf16_2e110", "f16_inf"])
def test_huge_row_scales_stay_in_their_rows(ctx, name):
    print("[case] w4a8k huge row scales %s" % name, flush=True)
    finite = name == "bf16_2e110"
    M = 40
    p = dynamic_quant(M, 256, 4098, 23, exact=True, scale_dt=dt.bf16 if finite else dt.f16)
    mask, code, group, ss = p.scales["src"]
    ss = np.array(ss, dtype=np.float64)
    ss[5, 0] = ss[M - 1, 1] = 2.0 ** 110 if finite else np.inf
    p.scales["src"] = (mask, code, group, ss)
    got, want = run(ctx, p, 0x14), p.run_oracle()
    got, want = O.to_f32(p.dst.dt, got).reshape(M, -1), O.to_f32(p.dst.dt, want).reshape(M, -1)
    assert np.isfinite(want).all() == finite
    np.testing.assert_array_equal(got, want)


def test_arbitrary_scales_and_post_ops(ctx):
    """An f32 mask per result and an eltwise: every row and column takes its own operand (1e-5 of the summed terms:
    the waves' sums are added in another order than the oracle's)."""
    print("[case] w4a8k post-ops", flush=True)
    M, N = 100, 4010
    add = TensorSpec(dt.f32, [M, N], None, np.random.default_rng(M).standard_normal((M, N)) * 4)
    p = dynamic_quant(M, 1152, N, 19, dst_dt=dt.f32,
                      post_ops=[{"kind": "eltwise", "alg": A.eltwise_relu, "alpha": 0.5},
                                {"kind": "binary", "alg": A.binary_add, "src1": add}])
    assert_f32_close(run(ctx, p, 0x24), p.run_oracle(), rel=1e-5, scale=p.term_scale, what="f32")
