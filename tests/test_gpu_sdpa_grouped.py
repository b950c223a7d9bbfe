"""Few queries against a grouped K / V cache: the heads of a group share a workgroup, their queries the 16 columns of
one MFMA (as many whole divisors of the group as fit). Against float64 attention under the comparison rule of the
reference's own SDPA test, as the cases beside this file."""
import numpy as np
import pytest

import onednn_amd as dnnl
from qmm_harness import dt
from test_gpu_sdpa import attention64, f16, f16_to_f64, reference_rule, run_sdpa

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    eng = dnnl.engine(dnnl.engine.kind.gpu, 0)
    return eng, dnnl.stream(eng)


@pytest.mark.parametrize("qdt", [dt.f16, dt.bf16], ids=["f16", "bf16"])
@pytest.mark.parametrize("rep,Qn,S,D,mkind,quant", [
    (16, 1, 1, 64, "none", None), (5, 3, 700, 128, "per_head", None), (6, 4, 300, 96, "causal", None),
    (7, 1, 2049, 128, "per_head", "f16"), (4, 4, 33, 32, "none", "f32"), (8, 1, 4100, 256, "none", "f16"),
    (32, 1, 640, 128, "per_head", "f32"), (3, 9, 129, 64, "causal", None),
], ids=str)
def test_heads_of_a_group_share_a_workgroup(ctx, rep, Qn, S, D, mkind, quant, qdt):
    print("[case] sdpa grouped rep=%d Qn=%d S=%d D=%d %s %s %s" % (rep, Qn, S, D, mkind, quant, qdt), flush=True)
    MB, KH = 2, 2
    H = KH * rep
    r = np.random.default_rng(rep * 100 + S)
    q = f16(r.standard_normal((MB, H, Qn, D)), qdt)
    scale = 1.0 / np.sqrt(D)
    mask = None
    if mkind == "per_head":
        mask = (r.standard_normal((1, H, Qn, S)) * 2).astype(np.float32)
        mask[..., 1::6] = -np.inf
    kw = dict(scale=scale, mask=mask, causal=mkind == "causal", kv_heads=KH, qdt=qdt)
    if quant is None:
        k, v = f16(r.standard_normal((MB, KH, S, D)), qdt), f16(r.standard_normal((MB, KH, S, D)), qdt)
        got = run_sdpa(ctx, q, k, v, **kw)
        k64, v64 = f16_to_f64(k, qdt), f16_to_f64(v, qdt)
    else:
        k = r.integers(-128, 128, (MB, KH, S, D)).astype(np.int8)
        v = r.integers(-128, 128, (MB, KH, S, D)).astype(np.int8)
        sdt, zdt, znp = (dt.f16, dt.s8, np.int8) if quant == "f16" else (dt.f32, dt.s32, np.int32)
        side = []
        for x, groups in ((k, (D, 1)), (v, (1, D))):
            sc = r.uniform(0.005, 0.02, (KH, S)).astype(np.float32)
            raw = f16(sc) if quant == "f16" else sc
            val = f16_to_f64(raw) if quant == "f16" else sc.astype(np.float64)
            zp = r.integers(-6, 7, (KH, S)).astype(znp)
            # the cache as the reorder to the queries' type gives it
            x64 = f16_to_f64(f16((x - zp[None, ..., None].astype(np.float64)) * val[None, ..., None], qdt), qdt)
            side.append((x64, (0b1110, groups, sdt, raw, zdt, zp)))
        got = run_sdpa(ctx, q, k, v, kv_dt=dt.s8, k_q=side[0][1], v_q=side[1][1], **kw)
        k64, v64 = side[0][0], side[1][0]
    s_eff = float(f16_to_f64(f16(np.array([scale]), qdt), qdt)[0])
    gold = attention64(f16_to_f64(q, qdt), np.swapaxes(k64, -1, -2), v64, s_eff,
                       None if mask is None else mask.astype(np.float64), mkind == "causal", rep)
    bad, total, worst = reference_rule(f16_to_f64(got, qdt), gold, 0.001466 if qdt == dt.f16 else 0.0079)
    print("[sdpa grouped] %d of %d outside the threshold, max diff %.2e" % (bad, total, worst))
    assert bad <= total * 0.0006


@pytest.mark.parametrize("ranges", [3, 4, 5, 6, 7, 8, 9, 15, 16, 17, 23])
@pytest.mark.parametrize("H,KH,Qn", [(2, 2, 1), (8, 2, 2), (15, 3, 1)], ids=str)
def test_every_count_of_ranges_is_combined(ctx, ranges, H, KH, Qn):
    """128 keys a range at these head counts; the combining kernel adds eight ranges at a time, then the rest."""
    print("[case] sdpa combine ranges=%d H=%d KH=%d Qn=%d" % (ranges, H, KH, Qn), flush=True)
    MB, D, S = 2, 128, 128 * ranges - 5
    r = np.random.default_rng(ranges * 10 + H)
    q = f16(r.standard_normal((MB, H, Qn, D)))
    k, v = f16(r.standard_normal((MB, KH, S, D))), f16(r.standard_normal((MB, KH, S, D)))
    scale = 1.0 / np.sqrt(D)
    got = run_sdpa(ctx, q, k, v, scale=scale, kv_heads=KH)
    s_eff = float(f16_to_f64(f16(np.array([scale])))[0])
    gold = attention64(f16_to_f64(q), np.swapaxes(f16_to_f64(k), -1, -2), f16_to_f64(v), s_eff, None, False, H // KH)
    bad, total, worst = reference_rule(f16_to_f64(got), gold, 0.001466)
    print("[sdpa combine] %d of %d outside the threshold, max diff %.2e" % (bad, total, worst))
    assert bad <= total * 0.0006


@pytest.mark.parametrize("H,KH,Qn", [(32, 4, 1), (24, 2, 1), (12, 1, 2), (14, 2, 1), (4, 1, 3)], ids=str)
@pytest.mark.parametrize("S", [256, 257, 2048, 2049])
def test_heads_in_a_pack_by_the_number_of_keys(ctx, H, KH, Qn, S):
    """Fewer heads share a workgroup up to 2048 keys in several ranges (more than 256 keys here) than past either end."""
    print("[case] sdpa packs H=%d KH=%d Qn=%d S=%d" % (H, KH, Qn, S), flush=True)
    D = 128
    r = np.random.default_rng(H * 100 + S)
    q = f16(r.standard_normal((1, H, Qn, D)))
    k, v = f16(r.standard_normal((1, KH, S, D))), f16(r.standard_normal((1, KH, S, D)))
    scale = 1.0 / np.sqrt(D)
    got = run_sdpa(ctx, q, k, v, scale=scale, kv_heads=KH)
    s_eff = float(f16_to_f64(f16(np.array([scale])))[0])
    gold = attention64(f16_to_f64(q), np.swapaxes(f16_to_f64(k), -1, -2), f16_to_f64(v), s_eff, None, False, H // KH)
    bad, total, worst = reference_rule(f16_to_f64(got), gold, 0.001466)
    print("[sdpa packs] %d of %d outside the threshold, max diff %.2e" % (bad, total, worst))
    assert bad <= total * 0.0006


@pytest.mark.parametrize("Qn,H", [(1, 4), (1, 8), (64, 4)], ids=str)
def test_u8_cache_with_negative_zero_points(ctx, Qn, H):
    """Zero points of the other sign than the cache's type: 1024 + z lies below the range of the bytes' own exponent, and
    every difference is still an exact f16 number (the whole range -128 ... 127 in turn)."""
    print("[case] sdpa u8 cache s8 zero points Qn=%d H=%d" % (Qn, H), flush=True)
    KH, S, D = 4, 260, 128
    r = np.random.default_rng(Qn + H)
    q = f16(r.standard_normal((1, H, Qn, D)))
    zp = ((np.arange(KH * S).reshape(KH, S) * 5) % 256 - 128).astype(np.int8)
    side = []
    for groups in ((D, 1), (1, D)):
        # bytes around their zero point where the type holds them, so that the scores stay of order one
        x = np.clip(zp[..., None].astype(np.int64) + r.integers(-60, 61, (KH, S, D)), 0, 255).astype(np.uint8)[None]
        sc = f16(r.uniform(0.005, 0.02, (KH, S)))
        x64 = f16_to_f64(f16((x - zp[None, ..., None].astype(np.float64)) * f16_to_f64(sc)[None, ..., None]))
        side.append((x, x64, (0b1110, groups, dt.f16, sc, dt.s8, zp)))
    scale = 1.0 / np.sqrt(D)
    got = run_sdpa(ctx, q, side[0][0], side[1][0], scale=scale, kv_heads=KH, kv_dt=dt.u8, k_q=side[0][2], v_q=side[1][2])
    s_eff = float(f16_to_f64(f16(np.array([scale])))[0])
    gold = attention64(f16_to_f64(q), np.swapaxes(side[0][1], -1, -2), side[1][1], s_eff, None, False, H // KH)
    bad, total, worst = reference_rule(f16_to_f64(got), gold, 0.001466)
    print("[sdpa u8 zp] %d of %d outside the threshold, max diff %.2e" % (bad, total, worst))
    assert bad <= total * 0.0006
