"""GPU parity of the kernel that cuts K over a workgroup's waves for 8-bit operands (qmm_gemm_b8k.hip, hip:gfx950:mfma_b8):
rows and columns that end inside a workgroup's blocks, waves without a tile of 128 k, with an odd and an even number of
them, u8 sources with zero points, scales per row, pitched rows, the loads past the caches. Integer sums are exact, fp8
codes have few bits, so every result is bit for bit. Each case asserts the shape its sizes take: the kernels beside this
one carry the same implementation name."""
import numpy as np
import pytest

import onednn_amd as dnnl
import test_gpu_parity as cases
from onednn_amd import _capi
from qmm_harness import TensorSpec, assert_bit_exact, dt
from test_gpu_b8_stream import fp8_sum
from test_gpu_g128 import pitched

pytestmark = pytest.mark.gpu
A = dnnl.algorithm


@pytest.fixture(scope="module")
def ctx():
    eng = dnnl.engine(dnnl.engine.kind.gpu, 0)
    return eng, dnnl.stream(eng)


def run(ctx, p, shape):
    eng, strm = ctx
    (M, K), N = p.src.dims, p.wei.dims[1]
    assert _capi.lib().qmm_gemm_b8k_shape(p.src.dt, M, N, K, bool(p.post_ops)) == shape
    got, pd = p.run_gpu(eng, strm, weights_any=True, return_pd=True)
    assert pd.impl_info_str() == "hip:gfx950:mfma_b8"
    return got


CASES = {
    "one_tile_one_row": (0x12, dict(M=1, K=128, N=33)),
    "rows16_9_tiles": (0x12, dict(M=17, K=1152, N=1031)),
    "cols64": (0x14, dict(M=5, K=512, N=14339)),
    "rows32_32": (0x22, dict(M=129, K=384, N=7275)),
    "rows32_64_17_tiles": (0x24, dict(M=65, K=2176, N=4203)),
    "rows64_32": (0x42, dict(M=127, K=1152, N=3590)),
    "rows64_64": (0x44, dict(M=190, K=1280, N=2795)),
    "40_mb_of_weights": (0x44, dict(M=63, K=4096, N=10250)),
}


@pytest.mark.parametrize("src", [dt.s8, dt.u8], ids=["s8", "u8"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_integers(ctx, name, src):
    print("[case] b8k %s %d" % (name, src), flush=True)
    shape, kw = CASES[name]
    if src == dt.u8:
        p = cases.int8_linear(seed=40 + len(name), src_dt=src, src_zp=119, dst_dt=dt.s32 if kw["M"] == 1 else dt.f32, **kw)
    else:
        p = cases.int8_linear(seed=40 + len(name), src_dt=src, src_zp=None, per_token=True, dst_dt=dt.bf16, **kw)
    assert_bit_exact(run(ctx, p, shape), p.run_oracle(), name)


def test_pitched_rows_post_ops_and_dst_quantization(ctx):
    print("[case] b8k pitched", flush=True)
    M, K, N = 70, 384, 2050
    add = TensorSpec(dt.f32, [M, N], None, np.random.default_rng(5).standard_normal((M, N)) * 4)
    p = pitched(cases.int8_linear(M, K, N, 3, bias_dt=dt.f32, dst_dt=dt.s8, dst_scale=0.5, dst_zp=[3], src_zp=7, post_ops=[
        {"kind": "binary", "alg": A.binary_add, "src1": add}, {"kind": "eltwise", "alg": A.eltwise_relu, "alpha": 0.5}]), 400)
    assert_bit_exact(run(ctx, p, 0x42), p.run_oracle(), "pitched")


@pytest.mark.parametrize("M,K,N,shape", [(1, 128, 40, 0x12), (33, 1152, 1031, 0x12), (129, 384, 7275, 0x22),
                                         (65, 384, 2050, 0x42), (65, 2176, 4203, 0x24), (190, 1280, 2795, 0x44), (64, 2944, 14338, 0x44)])
def test_fp8_into_a_residual(ctx, M, K, N, shape):
    print("[case] b8k fp8 %d %d %d" % (M, K, N), flush=True)
    assert _capi.lib().qmm_gemm_b8k_shape(dt.f8_e4m3, M, N, K, 1) == shape
    fp8_sum(ctx, M, K, N, M + N, dt.f32)


@pytest.mark.parametrize("M,K,N,shape", [(2, 8192, 16418, 0x12), (33, 3072, 43700, 0x44)])
@pytest.mark.parametrize("kind", ["s8", "u8", "fp8"])
def test_weights_past_the_caches(ctx, kind, M, K, N, shape):
    """128 MB of weights and more, read once: the loads are others. Exact in f32, whatever the order of the sums."""
    import torch
    from onednn_amd import memory
    print("[case] b8k past the caches %s %d %d %d" % (kind, M, K, N), flush=True)
    assert K * N >= 128 << 20
    code = {"s8": dt.s8, "u8": dt.u8, "fp8": dt.f8_e4m3}[kind]
    assert _capi.lib().qmm_gemm_b8k_shape(code, M, N, K, kind == "fp8") == shape
    if kind == "fp8":
        fp8_sum(ctx, M, K, N, M, dt.f32)
        return
    eng, strm = ctx
    g = torch.Generator().manual_seed(M)
    lo, hi, kind_t = (0, 256, torch.uint8) if kind == "u8" else (-127, 128, torch.int8)
    a = torch.randint(lo, hi, (M, K), generator=g, dtype=kind_t)
    b = torch.randint(-127, 128, (K, N), generator=g, dtype=torch.int8)
    T = lambda name: 2 + memory.format_tag._plain.index(name)  # noqa: E731
    pd = dnnl.matmul.primitive_desc(eng, memory.desc([M, K], code, T("ab")), memory.desc([K, N], dt.s8, memory.format_tag.any),
                                    memory.desc([M, N], dt.s32, T("ab")))
    packed = memory(pd.weights_desc(), eng)
    plain = memory(memory.desc([K, N], dt.s8, T("ab")), eng).write(b.numpy())
    dnnl.reorder(plain, packed).execute(strm, plain, packed)
    out = memory(pd.dst_desc(), eng)
    dnnl.matmul(pd).execute(strm, {dnnl.DNNL_ARG_SRC: memory(pd.src_desc(), eng).write(a.numpy()),
                                   dnnl.DNNL_ARG_WEIGHTS: packed, dnnl.DNNL_ARG_DST: out})
    strm.wait()
    want = a.double() @ b.double()
    got = out.read(np.int32, (M, N))
    assert (torch.from_numpy(got.copy()).double() == want).all()
