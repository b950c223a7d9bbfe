"""GPU parity of the kernel for many matrices of a short K (qmm_gemm_b8s.hip, hip:gfx950:mfma_b8): rows and columns that end
inside a wave's 32 x 64, more than 256 rows (the order of the row tiles), scales per column, a bias, a mask for all
matrices or one each, source scales per row. Integer sums, so every result is bit for bit; widths off a multiple of 4 take
this kernel from 64 tiles of 128 x 128 on, which each case asserts: the kernels with tiles carry the same name."""
import numpy as np
import pytest

import onednn_amd as dnnl
from onednn_amd import _capi
from qmm_harness import Problem, TensorSpec, assert_bit_exact, dt

pytestmark = pytest.mark.gpu
A = dnnl.algorithm


@pytest.fixture(scope="module")
def ctx():
    eng = dnnl.engine(dnnl.engine.kind.gpu, 0)
    return eng, dnnl.stream(eng)


def scores(B, M, N, K, seed, mask=None, columns=False, bias=False, rows=False):
    r = np.random.default_rng(seed)
    q, k = r.integers(-127, 128, (B, M, K)), r.integers(-127, 128, (B, K, N))
    scales = {"src": (6, dt.f32, (1, K), r.uniform(0.005, 0.02, M)) if rows else (0, dt.f32, None, [0.01]),
              "wei": (4, dt.f32, None, r.uniform(0.001, 0.01, N)) if columns else (0, dt.f32, None, [0.012])}
    po = []
    if mask:
        shape = [B if mask == "each" else 1, M if mask != "columns" else 1, N]
        po = [{"kind": "binary", "alg": A.binary_add,
               "src1": TensorSpec(dt.f32, shape, None, r.standard_normal(shape).astype(np.float32) * 8)}]
    return Problem(TensorSpec(dt.s8, [B, M, K], None, q), TensorSpec(dt.s8, [B, K, N], None, k), TensorSpec(dt.f32, [B, M, N]),
                   bias=TensorSpec(dt.f32, [1, 1, N], None, r.integers(-20, 20, N)) if bias else None, scales=scales,
                   post_ops=po)


@pytest.mark.parametrize("B,M,N,K,kw", [
    (16, 129, 129, 64, dict(mask="all")),
    (11, 257, 255, 128, dict(mask="all")),
    (11, 321, 130, 128, dict(mask="each")),
    (11, 150, 321, 64, dict(mask="columns")),
    (4, 600, 385, 64, dict(mask="all", columns=True)),
    (16, 193, 191, 128, dict(columns=True)),
    (8, 130, 447, 64, dict(bias=True, columns=True)),
    (16, 150, 129, 64, dict(rows=True, mask="all")),
    (11, 290, 255, 128, dict(rows=True, columns=True)),
], ids=str)
def test_scores(ctx, B, M, N, K, kw):
    print("[case] b8s %d %d %d %d %r" % (B, M, N, K, kw), flush=True)
    eng, strm = ctx
    # (a bias is not in the query; it does not enter the rule)
    assert _capi.lib().qmm_gemm_b8s_takes(B, M, N, K, N, "mask" in kw)
    p = scores(B, M, N, K, B + M + N, **kw)
    got, pd = p.run_gpu(eng, strm, weights_any=True, return_pd=True)
    assert pd.impl_info_str() == "hip:gfx950:mfma_b8"
    assert_bit_exact(got, p.run_oracle(), "scores")
