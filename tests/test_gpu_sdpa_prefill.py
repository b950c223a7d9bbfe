"""The many-queries attention kernel (two groups of waves over the keys, 128 queries a workgroup and 64 keys a tile)
at the sizes where its tiles end, against float64 attention under the reference test's rule."""
import numpy as np
import pytest

import onednn_amd as dnnl
import oracle as O
from onednn_amd import memory
from qmm_harness import T, dt
from test_gpu_sdpa import attention64, ctx, f16, f16_to_f64, reference_rule, run_sdpa, say  # noqa: F401

pytestmark = pytest.mark.gpu
THR = {dt.f16: 0.001466, dt.bf16: 0.0079}


def check(got, q, k, v, qdt, scale, causal, rep):
    gold = attention64(f16_to_f64(q, qdt), np.swapaxes(f16_to_f64(k, qdt), -1, -2), f16_to_f64(v, qdt), scale, None, causal,
                       rep)
    bad, total, worst = reference_rule(f16_to_f64(got, qdt), gold, THR[qdt])
    print("[sdpa prefill] %d of %d outside, max diff %.2e" % (bad, total, worst))
    assert bad <= total * 0.0006


CASES = [
    # heads, kv heads, queries, keys, D, causal: one tile and less; one row past the 32 queries of a wave and the 128
    # of a workgroup; 32 / 64 / 128 keys and one more or less; fewer keys than queries and more. (The fewest keys are the
    # other kernel's, see below.)
    (2, 2, 17, 1, 64, False), (2, 1, 31, 31, 128, True), (3, 3, 33, 64, 64, True), (2, 2, 32, 65, 128, False),
    (1, 1, 128, 127, 128, True), (4, 2, 129, 129, 64, True), (2, 2, 129, 400, 128, False), (2, 2, 300, 63, 128, True),
    (2, 2, 65, 192, 64, False), (2, 2, 257, 513, 64, True), (1, 1, 1100, 1100, 128, True), (2, 2, 600, 2305, 64, False),
    (2, 1, 17, 97, 64, False), (2, 2, 31, 128, 128, False), (2, 2, 32, 129, 64, False), (1, 1, 65, 65, 128, True),
    # more workgroups than CUs: a second round, a partial third one
    (40, 8, 1000, 1000, 64, True), (40, 40, 1000, 130, 128, False), (100, 4, 700, 70, 64, True),
]


@pytest.mark.parametrize("qdt", [dt.f16, dt.bf16], ids=["f16", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_ends_of_tiles(ctx, case, qdt):  # noqa: F811
    H, KV, Qn, S, D, causal = case
    say("sdpa prefill %s %r" % (qdt, case))
    r = np.random.default_rng(Qn * 3 + S)
    q = f16(r.standard_normal((1, H, Qn, D)), qdt)
    k, v = f16(r.standard_normal((1, KV, S, D)), qdt), f16(r.standard_normal((1, KV, S, D)), qdt)
    got = run_sdpa(ctx, q, k, v, scale=0.125, causal=causal, kv_heads=KV, qdt=qdt)
    check(got, q, k, v, qdt, 0.125, causal, H // KV)


@pytest.mark.parametrize("qdt", [dt.f16, dt.bf16], ids=["f16", "bf16"])
@pytest.mark.parametrize("case", [
    # the sizes at which one kernel takes over from the other: 96 and 97 keys (causal 32 and 33) with at most one
    # workgroup to a CU, and one head more than 256 workgroups
    (2, 2, 40, 96, 128, False), (2, 1, 40, 97, 128, False), (2, 2, 33, 32, 64, True), (2, 2, 33, 33, 64, True),
    (256, 8, 20, 40, 64, True), (257, 257, 20, 40, 64, True), (130, 13, 300, 420, 64, False), (130, 13, 300, 421, 64, False)], ids=str)
def test_either_side_of_the_rule(ctx, case, qdt):  # noqa: F811
    test_ends_of_tiles(ctx, case, qdt)


@pytest.mark.parametrize("scale", [-0.125, 4.0], ids=str)
def test_scales_that_are_not_the_usual(ctx, scale):  # noqa: F811
    """A negative scale (the maximum of the raw products is not that of the scores); scores far apart, so that the
    running maximum grows late and the probabilities before it vanish."""
    H, Qn, S, D = 2, 160, 4200, 64
    say("sdpa prefill scale %g" % scale)
    r = np.random.default_rng(3)
    q = f16(r.standard_normal((1, H, Qn, D)))
    k = r.standard_normal((1, H, S, D))
    k *= np.linspace(0.05, 1.0, S)[:, None]
    k, v = f16(k), f16(r.standard_normal((1, H, S, D)))
    got = run_sdpa(ctx, q, k, v, scale=scale)
    check(got, q, k, v, dt.f16, scale, False, 1)


def test_rows_of_all_heads_side_by_side(ctx):  # noqa: F811
    """Q, K, V and dst as [token][head][D] buffers."""
    eng, strm = ctx
    H, Qn, S, D = 3, 150, 140, 128
    say("sdpa prefill interleaved heads")
    r = np.random.default_rng(9)
    q, k, v = (f16(r.standard_normal((1, n, H, D))) for n in (Qn, S, S))
    q_md = memory.desc([1, H, Qn, D], dt.f16, T("acbd"))
    kt_md = memory.desc([1, H, D, S], dt.f16, T("adbc"))
    v_md = memory.desc([1, H, S, D], dt.f16, T("acbd"))
    out = memory(q_md, eng)
    pd = dnnl.sdpa.primitive_desc(eng, q_md, kt_md, v_md, None, dt.undef, q_md, False, 0, True)
    dnnl.sdpa(pd).execute(strm, {dnnl.DNNL_ARG_QUERIES: memory(q_md, eng).write(q), dnnl.DNNL_ARG_KEYS: memory(kt_md, eng).write(k),
                                 dnnl.DNNL_ARG_VALUES: memory(v_md, eng).write(v), dnnl.DNNL_ARG_DST: out})
    strm.wait()
    got = np.swapaxes(out.read(np.uint16, (1, Qn, H, D)), 1, 2)
    q, k, v = (np.swapaxes(x, 1, 2) for x in (q, k, v))
    check(got, q, k, v, dt.f16, 1.0, True, 1)


def test_infinite_values_stay_with_the_queries_that_see_them(ctx):  # noqa: F811
    """An infinite value at the last key, not a multiple of anything: queries that cannot see the key in a tile of
    their own stay finite, those that do are infinite, and none is NaN through the keys past the end."""
    H, Qn, S, D = 2, 200, 101, 64
    say("sdpa prefill infinite value")
    r = np.random.default_rng(11)
    q, k, v = (f16(r.standard_normal((1, H, n, D))) for n in (Qn, S, S))
    v[:, :, S - 1, 0] = 0x7C00
    got = f16_to_f64(run_sdpa(ctx, q, k, v, scale=0.125))
    assert np.isposinf(got[..., 0]).all() and np.isfinite(got[..., 1:]).all()
    got = f16_to_f64(run_sdpa(ctx, q, k, v, scale=0.125, causal=True))
    assert np.isposinf(got[:, :, S - 1:, 0]).all() and np.isfinite(got[..., 1:]).all()
    assert np.isfinite(got[:, :, :64]).all()  # whole tiles of 64 keys


@pytest.mark.parametrize("kv_dt,sdt,zdt", [(dt.s8, dt.f16, dt.s8), (dt.u8, dt.f16, dt.u8), (dt.s8, dt.f16, None), (dt.s8, dt.f32, dt.s32)], ids=str)
@pytest.mark.parametrize("Qn,S,D,qdt", [(257, 100, 128, dt.f16), (300, 301, 64, dt.bf16), (260, 65, 64, dt.f16),
                                        (257, 195, 128, dt.f16), (390, 281, 64, dt.f16), (290, 333, 128, dt.bf16)], ids=str)
def test_8_bit_cache_under_many_queries(ctx, Qn, S, D, qdt, kv_dt, sdt, zdt):  # noqa: F811
    """From 161 keys a workgroup (head size 64: 281) on the cache is written in the queries' type to the scratchpad first:
    the oracle's reorder gives the same values."""
    MB, H, KV = 2, 4, 2
    say("sdpa prefill 8-bit cache %r" % ((Qn, S, D, qdt, kv_dt, sdt, zdt),))
    r = np.random.default_rng(Qn + D)
    q = f16(r.standard_normal((MB, H, Qn, D)), qdt)
    lo, hi, npdt = (-128, 128, np.int8) if kv_dt == dt.s8 else (0, 256, np.uint8)
    kq, vq = (r.integers(lo, hi, (MB, KV, S, D)).astype(npdt) for _ in range(2))
    scale = [r.uniform(0.005, 0.02, (KV, S)) for _ in range(2)]
    ksc, vsc = [f16(x) if sdt == dt.f16 else x.astype(np.float32) for x in scale]
    znp = {dt.s8: np.int8, dt.u8: np.uint8, dt.s32: np.int32, None: np.int8}[zdt]
    kzp, vzp = [(r.integers(-6, 7, (KV, S)) + (100 if zdt == dt.u8 else 0)).astype(znp) for _ in range(2)]
    side = [(0b1110, g, sdt, sc, zdt, zp if zdt is not None else None)
            for g, sc, zp in (((D, 1), ksc, kzp), ((1, D), vsc, vzp))]
    got = run_sdpa(ctx, q, kq, vq, scale=0.125, causal=True, kv_heads=KV, kv_dt=kv_dt, k_q=side[0], v_q=side[1], qdt=qdt)
    kd, vd = np.zeros((MB, KV, S, D), np.uint16), np.zeros((MB, KV, S, D), np.uint16)
    for raw, sc, zp, outd in ((kq, ksc, kzp, kd), (vq, vsc, vzp, vd)):
        O.reorder(O.Tensor(kv_dt, [MB, KV, S, D], raw), O.Tensor(qdt, [MB, KV, S, D], outd),
                  src_scale=O.Quant(0b1110, sdt, sc, (1, D)),
                  src_zp=O.Quant(0b1110, zdt, zp, (1, D)) if zdt is not None else None)
    check(got, q, kd, vd, qdt, 0.125, True, H // KV)


@pytest.mark.parametrize("qdt", [dt.f16, dt.bf16], ids=["f16", "bf16"])
def test_a_late_key_that_outweighs_the_rest(ctx, qdt):  # noqa: F811
    """Past 2048 keys one key's weight is 2^6.3 ... 2^7.7 of the largest before it. Its probability is exactly 1, as that
    of every maximum, so the result is off by its own rounding and by what the other keys' rounded weights add: together
    0.07 of the result (2^-6.3 and 4350 x 2^-16), each within half a unit of its own last place and independent of the
    others. Against the float64 result rounded to the type that is at most sqrt(1 + 0.07^2) = 1.003 of the error; a
    rounded weight of the late key would be as large as the result's own rounding (1.2 ... 1.4)."""
    H, Qn, S, D = 1, 256, 4352, 64
    say("sdpa prefill late key %s" % qdt)
    r = np.random.default_rng(21)
    q, k = np.zeros((1, H, Qn, D)), np.zeros((1, H, S, D))
    q[..., 0] = np.linspace(0.9, 1.1, Qn)
    k[..., 0] = -16 * np.log(2.0)
    k[:, :, 5, 0] = 0.0
    k[:, :, 66 * 64 + 10, 0] = 7 * np.log(2.0)  # (tiles of 64 keys go to two groups of waves in turn: the same group)
    q, k, v = f16(q, qdt), f16(k, qdt), f16(r.standard_normal((1, H, S, D)), qdt)
    got = f16_to_f64(run_sdpa(ctx, q, k, v, scale=1.0, qdt=qdt), qdt)
    gold = attention64(f16_to_f64(q, qdt), np.swapaxes(f16_to_f64(k, qdt), -1, -2), f16_to_f64(v, qdt), 1.0, None, False, 1)
    off, own = np.linalg.norm(got - gold), np.linalg.norm(f16_to_f64(f16(gold, qdt), qdt) - gold)
    print("[sdpa prefill] error %.3e, rounding alone %.3e" % (off / np.linalg.norm(gold), own / np.linalg.norm(gold)))
    assert off <= 1.01 * own


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bits", [0x7C00, 0x7E00], ids=["inf", "nan"])
def test_values_past_a_block_of_32_keys_stay_out(ctx, D, bits):  # noqa: F811
    """A causal mask hides the second 32 of a tile's 64 keys from a wave's 32 queries, whatever the values there hold
    (rows of a cache that are not written yet): those queries' results are finite and the same."""
    H, Qn, S = 2, 96, 160
    say("sdpa prefill hidden block %d %x" % (D, bits))
    r = np.random.default_rng(31)
    q, k, v = (f16(r.standard_normal((1, H, n, D))) for n in (Qn, S, S))
    for first in (32, 96):
        want = run_sdpa(ctx, q, k, v, scale=0.125, causal=True)
        bad = v.copy()
        bad[:, :, first:] = bits
        got = run_sdpa(ctx, q, k, bad, scale=0.125, causal=True)
        assert (got[:, :, :first] == want[:, :, :first]).all()
