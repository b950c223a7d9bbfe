"""GPU parity of the tiled kernel for 4-bit weights with groups of 128 k at many rows (qmm_gemm_g128.hip): s8
activations (hip:gfx950:mfma_w4a8) and f16 / bf16 activations (hip:gfx950:decode_w4), at the edges of its tiles.

Sizes are chosen by its rule (gemm_g128_rows): more than 192 (s8) or 256 blocks of 64 rows x 256 columns, and the
taller tile where that needs fewer rounds; every case asserts the tile that its sizes take, since the kernels beside
this one carry the same implementation names. Bars as in the tests of the kernels beside it: bit for bit where every
order of operations gives the same bits, else a share of the summed magnitudes (f32 sums of a few hundred terms).
"""
import numpy as np
import pytest

import onednn_amd as dnnl
import oracle as O
import test_gpu_parity as parity
from onednn_amd import _capi
from qmm_harness import TensorSpec, assert_bf16_within_1ulp, assert_bit_exact, assert_f32_close, dt
from test_gpu_w4a8 import W4A8, dynamic_quant

pytestmark = pytest.mark.gpu
A = dnnl.algorithm


@pytest.fixture(scope="module")
def ctx():
    eng = dnnl.engine(dnnl.engine.kind.gpu, 0)
    return eng, dnnl.stream(eng)


def run(ctx, p, tile, impl):
    """The result, after checking that the sizes take a tile of so many rows (0: one of the other kernels)."""
    eng, strm = ctx
    (M, K), N = p.src.dims, p.wei.dims[1]
    assert _capi.lib().qmm_gemm_g128_rows(p.src.dt, M, N, K) == tile
    if impl == parity.DECODE:  # (the launch asks for this one first)
        assert not _capi.lib().qmm_gemm_w4k_shape(p.src.dt, 4, int(p.scales["wei"][2] is None), M, N, K)
    got, pd = p.run_gpu(eng, strm, weights_any=True, return_pd=True)
    assert pd.impl_info_str() == impl
    return got


def pitched(p, pitch):
    """The same source in rows of `pitch` elements."""
    p.src = TensorSpec(p.src.dt, p.src.dims, [pitch, 1], p.src.logical())
    return p


S8_CASES = {
    # 64-row tiles: row and column tails, one group, an odd number of groups
    "rows64_one_group_tails": (64, dict(M=129, K=128, N=16650)),
    "rows64_three_groups_bf16_scales": (64, dict(M=193, K=384, N=16642, scale_dt=dt.bf16)),
    # 128-row tiles
    "rows128_tails": (128, dict(M=700, K=256, N=14330)),
    "rows128_whole_tiles": (128, dict(M=640, K=512, N=14336, dst_dt=dt.f16)),
    # more than eight tiles of rows: the tile order goes on behind its first eight, with a short last group
    "rows64_18_row_tiles": (64, dict(M=1100, K=128, N=3400)),
    "rows128_10_row_tiles": (128, dict(M=1160, K=128, N=7150)),
}


@pytest.mark.parametrize("name", sorted(S8_CASES))
def test_s8_exact(ctx, name):
    print("[case] g128 s8 %s" % name, flush=True)
    tile, kw = S8_CASES[name]
    p = dynamic_quant(seed=500 + len(name), exact=True, **kw)
    assert_bit_exact(run(ctx, p, tile, W4A8), p.run_oracle(), name)


@pytest.mark.parametrize("wei_mask,src_mask,pitch", [(1, 3, 256), (3, 2, 256), (1, 2, 272), (3, 3, 320)])
def test_s8_scales_without_columns_or_rows_and_pitched_source(ctx, wei_mask, src_mask, pitch):
    """One scale per group for all columns / rows (a stride of 0 in the kernel); source rows with a gap."""
    print("[case] g128 s8 masks %d %d pitch %d" % (wei_mask, src_mask, pitch), flush=True)
    p = pitched(dynamic_quant(257, 256, 14350, 31, exact=True), pitch)
    _, code, groups, v = p.scales["wei"]
    p.scales["wei"] = (wei_mask, code, groups, v if wei_mask == 3 else np.ascontiguousarray(v[:, 3]))
    _, code, groups, v = p.scales["src"]
    p.scales["src"] = (src_mask, code, groups, v if src_mask == 3 else np.ascontiguousarray(v[5]))
    assert_bit_exact(run(ctx, p, 64, W4A8), p.run_oracle(), "masks")


def test_s8_extreme_sums(ctx):
    """The largest sums a group can reach, both signs: 128 * (-128) * (-8) and 128 * (-128) * 7, times 16."""
    print("[case] g128 s8 extremes", flush=True)
    p = dynamic_quant(129, 256, 16640, 7, exact=True)
    p.src.set(np.full((129, 256), -128.0))
    p.wei.set(np.where(np.arange(16640) % 2 == 0, -8.0, 7.0)[None].repeat(256, 0))
    assert_bit_exact(run(ctx, p, 64, W4A8), p.run_oracle(), "extremes")


@pytest.mark.parametrize("name", ["bf16_2e110", "f16_inf"])
@pytest.mark.parametrize("M", [129, 640])
def test_s8_huge_row_scales(ctx, M, name):
    """Row scales whose product with the bias of the sums is no f32 number: finite results stay exact, an infinite
    scale gives infinities of the sums' signs (NaN where a sum is 0)."""
    print("[case] g128 s8 huge row scales %d %s" % (M, name), flush=True)
    finite = name == "bf16_2e110"
    p = dynamic_quant(M, 256, 16640, 23, exact=True, scale_dt=dt.bf16 if finite else dt.f16)
    mask, code, group, ss = p.scales["src"]
    ss = np.array(ss, dtype=np.float64)
    ss[5, 0] = ss[M - 1, 1] = 2.0 ** 110 if finite else np.inf
    p.scales["src"] = (mask, code, group, ss)
    got, want = run(ctx, p, 64 if M == 129 else 128, W4A8), p.run_oracle()
    got, want = O.to_f32(p.dst.dt, got).reshape(M, -1), O.to_f32(p.dst.dt, want).reshape(M, -1)
    assert np.isfinite(want).all() == finite
    if finite:  # (a row's two groups lie 2^100 apart: one of them is lost in the rounding of the sum)
        assert np.abs(want[5]).max() > 2.0 ** 100
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("M,N,tile", [(257, 14350, 64), (700, 14330, 128)])
def test_s8_arbitrary_scales_and_post_ops(ctx, M, N, tile):
    print("[case] g128 s8 arbitrary scales %d" % M, flush=True)
    add = TensorSpec(dt.f32, [1, N], None, np.random.default_rng(M).standard_normal(N) * 4)
    p = dynamic_quant(M, 256, N, 19, dst_dt=dt.f32,
                      post_ops=[{"kind": "eltwise", "alg": A.eltwise_relu, "alpha": 0.5},
                                {"kind": "binary", "alg": A.binary_add, "src1": add}])
    assert_f32_close(run(ctx, p, tile, W4A8), p.run_oracle(), rel=1e-5, scale=p.term_scale, what="f32")


W4_CASES = {
    # 64-row tiles
    "f16_u4_rows64_tails": (64, dict(M=100, K=128, N=32900, act_dt=dt.f16, zp_dt=dt.u4)),
    "bf16_s4_zp_s8_rows64": (64, dict(M=100, K=384, N=32770, wei_dt=dt.s4, zp_dt=dt.s8, scale_dt=dt.bf16)),
    "f16_u4_zp_u8_groups256_f32_dst": (64, dict(M=97, K=512, N=32774, act_dt=dt.f16, zp_dt=dt.u8, G=256, zp_group=128,
                                                dst_dt=dt.f32)),
    "bf16_u4_14_row_tiles": (64, dict(M=870, K=128, N=7150)),
    # 96-row tiles
    "f16_s4_no_zp_rows96_tails": (96, dict(M=190, K=256, N=32700, act_dt=dt.f16, wei_dt=dt.s4, with_zp=False)),
    "bf16_u4_rows96_relu": (96, dict(M=129, K=256, N=22200,
                                     post_ops=[{"kind": "eltwise", "alg": A.eltwise_relu, "alpha": 0.0}])),
    "f16_u4_per_column_rows96": (96, dict(M=65, K=256, N=33000, act_dt=dt.f16, zp_dt=dt.u4, per_column=True)),
    "f16_u4_zp_groups512_10_row_tiles": (96, dict(M=870, K=512, N=9460, act_dt=dt.f16, zp_group=512)),
}


def check_16bit(p, M, N, got, name, terms=None):
    want = p.run_oracle()
    code = p.dst.dt
    terms = (parity.decode_term_scale(p) if terms is None else terms).reshape(M, N)
    if code == dt.bf16:
        assert_bf16_within_1ulp(got, want, name, abs_slack=2e-5 * terms.reshape(-1))
        return
    g, w = O.to_f32(code, got).reshape(M, N), O.to_f32(code, want).reshape(M, N)
    # f32 sums in another order: 2e-5 of the summed magnitudes; an f16 result one step (2^-10) more
    bar = 2e-5 * terms + (np.abs(w) * 2.0 ** -10 if code == dt.f16 else 0)
    assert np.all(np.abs(g.astype(np.float64) - w) <= bar), name


@pytest.mark.parametrize("name", sorted(W4_CASES))
def test_16bit_activations(ctx, name):
    print("[case] g128 %s" % name, flush=True)
    tile, kw = W4_CASES[name]
    p = parity.decode_w4(seed=600 + len(name), **kw)
    check_16bit(p, kw["M"], kw["N"], run(ctx, p, tile, parity.DECODE), name)


@pytest.mark.parametrize("act_dt,pitch,mask", [(dt.f16, 264, 3), (dt.bf16, 320, 3), (dt.f16, 256, 1), (dt.bf16, 256, 1)])
def test_16bit_pitched_source_and_scales_without_columns(ctx, act_dt, pitch, mask):
    print("[case] g128 16 bit pitch %d mask %d" % (pitch, mask), flush=True)
    p = pitched(parity.decode_w4(129, 256, 22200, 640 + pitch, act_dt=act_dt), pitch)
    _, code, groups, v = p.scales["wei"]
    if mask == 1:
        v = np.repeat(v[:, 7:8], 22200, 1)
        p.scales["wei"] = (3, code, groups, v)
    terms = parity.decode_term_scale(p)
    if mask == 1:
        p.scales["wei"] = (1, code, groups, np.ascontiguousarray(v[:, 0]))
    check_16bit(p, 129, 22200, run(ctx, p, 96, parity.DECODE), "pitched", terms)


# One row of tiles over more than 65536 columns: the tiled kernel where it is the faster one, else the decode kernels.
FEW_ROWS = {
    "f16_1_row_decode": (dict(M=1, K=2048, N=65552, act_dt=dt.f16), 0),
    "bf16_8_rows_decode": (dict(M=8, K=2048, N=65552), 0),
    "f16_5_rows_tiled": (dict(M=5, K=128, N=65552, act_dt=dt.f16), 64),
    "bf16_16_rows_tiled": (dict(M=16, K=256, N=65590, with_zp=False, wei_dt=dt.s4), 64),
    "f16_33_rows_tiled": (dict(M=33, K=256, N=65544, act_dt=dt.f16), 64),
}


@pytest.mark.parametrize("name", sorted(FEW_ROWS))
def test_few_rows_of_wide_weights(ctx, name):
    print("[case] g128 few rows %s" % name, flush=True)
    kw, tile = FEW_ROWS[name]
    p = parity.decode_w4(seed=700 + len(name), **kw)
    check_16bit(p, kw["M"], kw["N"], run(ctx, p, tile, parity.DECODE), name)
