"""The streaming kernel of few rows or few results (32 x 32 results a workgroup, K cut over its waves) and the rows that
the tiled kernels store one vector at a time: where blocks of 32 rows, 32 columns and K's fragments end, s8 / u8 / f8
operands, every kind of column and row operand. Integer problems bit for bit against the oracle and against the tiled
kernels (QMM_GEMM_VARIANT), fp8 within the rounding of its sums. Where K is a multiple of 128 and there are no weights
zero points, the default choice of most small problems is the kernel of qmm_gemm_b8k.hip (the same implementation name): the
streaming kernel without row sums runs in test_the_streaming_kernel_itself and test_fp8_streams."""
import numpy as np
import pytest

import onednn_amd as dnnl
import test_gpu_parity as cases
from onednn_amd import _capi
from qmm_harness import assert_bit_exact, dt
from test_gpu_int8_wei_zp import w8a8

pytestmark = pytest.mark.gpu
A = dnnl.algorithm


@pytest.fixture(scope="module")
def ctx():
    eng = dnnl.engine(dnnl.engine.kind.gpu, 0)
    return eng, dnnl.stream(eng)


# M, K, N: one row past a block of 32 and of 64; columns that end inside a quad; fewer fragments than waves, a last
# chunk of one; one past 8 column blocks (the XCD order's last, partial group). The last: the kernel of 33 ... 64 rows over
# more than 4096 columns where waves have no fragment
SHAPES = [(33, 32, 33), (64, 224, 72), (65, 288, 64), (63, 2080, 4130), (96, 512, 257), (97, 1056, 290), (130, 256, 1001),
          (256, 1024, 96), (40, 4096, 4128), (5, 224, 70), (63, 96, 4200)]


@pytest.mark.parametrize("src", [dt.s8, dt.u8], ids=["s8", "u8"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_blocks_of_rows_and_columns(ctx, monkeypatch, shape, src):
    eng, strm = ctx
    M, K, N = shape
    print("[case] stream %s %r" % (src, shape), flush=True)
    kw = dict(src_dt=dt.u8, src_zp=119) if src == dt.u8 else {}
    p = w8a8(seed=M + K + N, M=M, K=K, N=N, **kw)
    want = p.run_oracle()
    assert_bit_exact(p.run_gpu(eng, strm, weights_any=True), want, "stream")
    monkeypatch.setenv("QMM_GEMM_VARIANT", "3")  # 64 x 64 tiles
    assert_bit_exact(p.run_gpu(eng, strm, weights_any=True), want, "tiles")


def streams(monkeypatch, src, M, K, N, post_ops=0):
    """Plans made from here on take the streaming kernel: by default, or up to 64 rows of integers in a variant of the tiles,
    which the kernel that cuts K over its waves is not for."""
    lib = _capi.lib()
    assert lib.qmm_gemm_b8_tile(dt.f8_e4m3 if src == dt.f8_e4m3 else dt.s8, 1, M, N, K, post_ops) == 32
    if lib.qmm_gemm_b8k_shape(src, M, N, K, post_ops):
        assert M <= 64 and src != dt.f8_e4m3
        monkeypatch.setenv("QMM_B8X_VARIANT", "2")


@pytest.mark.parametrize("src", [dt.s8, dt.u8], ids=["s8", "u8"])
@pytest.mark.parametrize("M,K,N", [(33, 32, 33), (63, 2080, 4130), (40, 4096, 4128), (5, 256, 70), (1, 4224, 34), (4, 128, 40),
                                   (17, 1024, 130), (64, 1152, 200), (96, 544, 257), (130, 288, 1001), (256, 1056, 96)], ids=str)
def test_the_streaming_kernel_itself(ctx, monkeypatch, M, K, N, src):
    """... without weights zero points, which by themselves keep a problem off the other kernel."""
    print("[case] stream itself %s %d %d %d" % (src, M, K, N), flush=True)
    kw = dict(src_zp=119) if src == dt.u8 else dict(src_zp=None, per_token=True, dst_dt=dt.bf16)
    p = cases.int8_linear(M, K, N, M + K + N, src_dt=src, **kw)
    streams(monkeypatch, src, M, K, N, bool(p.post_ops))
    eng, strm = ctx
    assert_bit_exact(p.run_gpu(eng, strm, weights_any=True), p.run_oracle(), "stream")


@pytest.mark.parametrize("M,K,N", [(70, 256, 98), (40, 512, 4200), (33, 96, 64), (40, 208, 72), (64, 208, 4130),
                                   (33, 1040, 4130)])
def test_post_ops_row_by_row(ctx, M, K, N):
    """... and, with u8 sources, K that ends inside a fragment of 32."""
    eng, strm = ctx
    print("[case] stream post-ops %d %d %d" % (M, K, N), flush=True)
    p = cases.int8_linear(M, K, N, 3, post_ops=[{"kind": "eltwise", "alg": A.eltwise_relu, "alpha": 0.5},
                                                {"kind": "eltwise", "alg": A.eltwise_linear, "alpha": 2.0, "beta": -1.0}])
    assert_bit_exact(p.run_gpu(eng, strm, weights_any=True), p.run_oracle(), "chain")


def fp8_sum(ctx, M, K, N, seed, dst=dt.bf16, scale=0.125):
    """f8_e4m3 codes with few significant bits: every product and every sum is exact in f32, whatever its order."""
    import torch
    from onednn_amd import memory
    eng, strm = ctx
    g = torch.Generator().manual_seed(seed)
    a = torch.randint(-3, 4, (M, K), generator=g).float()
    b = torch.randint(-3, 4, (K, N), generator=g).float()
    old = torch.randint(-8, 9, (M, N), generator=g).float()
    T = lambda name: 2 + memory.format_tag._plain.index(name)  # noqa: E731
    attr = dnnl.primitive_attr()
    attr.set_scales_mask(dnnl.DNNL_ARG_SRC, 0)
    po = dnnl.post_ops()
    po.append_sum(1.0)
    attr.set_post_ops(po)
    pd = dnnl.matmul.primitive_desc(eng, memory.desc([M, K], dt.f8_e4m3, T("ab")), memory.desc([K, N], dt.f8_e4m3, T("ab")),
                                    memory.desc([M, N], dst, T("ab")), attr=attr)
    f8 = lambda x: x.to(torch.float8_e4m3fn).view(torch.uint8).numpy()  # noqa: E731
    store = old.to(torch.bfloat16).view(torch.int16).numpy() if dst == dt.bf16 else old.numpy()
    out = memory(pd.dst_desc(), eng).write(store)
    sc = np.array([scale], np.float32)
    dnnl.matmul(pd).execute(strm, {
        dnnl.DNNL_ARG_SRC: memory(pd.src_desc(), eng).write(f8(a)),
        dnnl.DNNL_ARG_WEIGHTS: memory(memory.desc([K, N], dt.f8_e4m3, T("ab")), eng).write(f8(b)),
        dnnl.DNNL_ARG_DST: out,
        dnnl.DNNL_ARG_ATTR_SCALES | dnnl.DNNL_ARG_SRC: memory(memory.desc([1], dt.f32, T("a")), eng).write(sc)})
    strm.wait()
    want = a.double() @ b.double() * scale + old.double()
    if dst == dt.bf16:
        got = torch.from_numpy(out.read(np.int16, (M, N)).copy()).view(torch.bfloat16)
        want = want.float().to(torch.bfloat16)
    else:
        got, want = torch.from_numpy(out.read(np.float32, (M, N)).copy()), want.float()
    bad = (got != want).sum().item()
    assert bad == 0, "%d of %d differ" % (bad, M * N)


@pytest.mark.parametrize("dst", [dt.bf16, dt.f32], ids=["bf16", "f32"])
@pytest.mark.parametrize("M,K,N", [(3, 64, 40), (33, 128, 33), (300, 64, 70), (257, 1920, 130), (100, 448, 999)])
def test_fp8_into_a_residual(ctx, M, K, N, dst):
    """The streaming kernel: pairs of fragments, one pair in all and an odd number of them per wave."""
    print("[case] fp8 stream %d %d %d" % (M, K, N), flush=True)
    fp8_sum(ctx, M, K, N, M + N, dst)


@pytest.mark.parametrize("M,K,N", [(3, 64, 40), (33, 192, 33), (257, 1856, 130), (100, 448, 999), (16, 2112, 2050)])
def test_fp8_streams(ctx, monkeypatch, M, K, N):
    print("[case] fp8 streams %d %d %d" % (M, K, N), flush=True)
    streams(monkeypatch, dt.f8_e4m3, M, K, N, 1)
    fp8_sum(ctx, M, K, N, M + N, dt.f32)


@pytest.mark.parametrize("B,M,K,N", [(8, 64, 512, 1024), (2, 130, 384, 257), (3, 33, 512, 64), (20, 64, 512, 640)])
def test_fp8_batches(ctx, B, M, K, N):
    """The default choice on either side of its lines: 256 x 256 tiles, 64 x 64 ones, more batches than the former take."""
    import torch
    from onednn_amd import memory
    eng, strm = ctx
    print("[case] fp8 batches %d %d %d %d" % (B, M, K, N), flush=True)
    g = torch.Generator().manual_seed(B + M)
    a, b = (torch.randint(-3, 4, s, generator=g).float() for s in ((B, M, K), (B, K, N)))  # (sums below 2^24: exact)
    T = lambda name: 2 + memory.format_tag._plain.index(name)  # noqa: E731
    f8 = lambda x: x.to(torch.float8_e4m3fn).view(torch.uint8).numpy()  # noqa: E731
    mds = [memory.desc(d, t, T("abc")) for d, t in (([B, M, K], dt.f8_e4m3), ([B, K, N], dt.f8_e4m3), ([B, M, N], dt.f32))]
    pd = dnnl.matmul.primitive_desc(eng, *mds)
    out = memory(mds[2], eng)
    dnnl.matmul(pd).execute(strm, {dnnl.DNNL_ARG_SRC: memory(mds[0], eng).write(f8(a)),
                                   dnnl.DNNL_ARG_WEIGHTS: memory(mds[1], eng).write(f8(b)), dnnl.DNNL_ARG_DST: out})
    strm.wait()
    got = torch.from_numpy(out.read(np.float32, (B, M, N)).copy())
    assert (got == torch.bmm(a, b)).all()


@pytest.mark.parametrize("variant", [2, 3, 6])
@pytest.mark.parametrize("M,K,N,dst", [(300, 512, 520, dt.bf16), (255, 384, 257, dt.bf16), (190, 640, 390, dt.f32),
                                       (64, 384, 130, dt.f32), (449, 512, 513, dt.f32)], ids=str)
def test_fp8_tiles_that_end_inside(ctx, monkeypatch, M, K, N, dst, variant):
    """Whole and partial halves of a wave's rows, columns that end inside a quad, rows at any alignment."""
    print("[case] fp8 tiles %d %d %d variant %d" % (M, K, N, variant), flush=True)
    monkeypatch.setenv("QMM_GEMM_VARIANT", str(variant))
    fp8_sum(ctx, M, K, N, M + N, dst)


@pytest.mark.parametrize("tokens,d", [(131, 64), (257, 128), (150, 64), (321, 64), (64, 128)])
def test_scores_of_any_width(ctx, tokens, d):
    """Batched s8 x s8 scores with a mask added, rows that start at any 4-byte boundary."""
    import torch
    from onednn_amd import memory
    eng, strm = ctx
    print("[case] scores %d %d" % (tokens, d), flush=True)
    g = torch.Generator().manual_seed(tokens)
    H = 12
    q, k = (torch.randint(-127, 128, (H, tokens, d), generator=g, dtype=torch.int8) for _ in range(2))
    k = k.transpose(1, 2).contiguous()
    mask = torch.randint(-4, 5, (1, tokens, tokens), generator=g).float()
    T = lambda name: 2 + memory.format_tag._plain.index(name)  # noqa: E731
    attr = dnnl.primitive_attr()
    mask_md = memory.desc([1, tokens, tokens], dt.f32, T("abc"))
    po = dnnl.post_ops()
    po.append_binary(A.binary_add, mask_md)
    attr.set_post_ops(po)
    pd = dnnl.matmul.primitive_desc(eng, memory.desc([H, tokens, d], dt.s8, T("abc")), memory.desc([H, d, tokens], dt.s8, T("abc")),
                                    memory.desc([H, tokens, tokens], dt.f32, T("abc")), attr=attr)
    out = memory(pd.dst_desc(), eng)
    dnnl.matmul(pd).execute(strm, {
        dnnl.DNNL_ARG_SRC: memory(pd.src_desc(), eng).write(q.numpy()),
        dnnl.DNNL_ARG_WEIGHTS: memory(memory.desc([H, d, tokens], dt.s8, T("abc")), eng).write(k.numpy()),
        dnnl.DNNL_ARG_ATTR_MULTIPLE_POST_OP(0) | dnnl.DNNL_ARG_SRC_1: memory(mask_md, eng).write(mask.numpy()),
        dnnl.DNNL_ARG_DST: out})
    strm.wait()
    want = (torch.bmm(q.double(), k.double()) + mask.double()).float()  # below 2^24: exact
    assert (torch.from_numpy(out.read(np.float32, (H, tokens, tokens)).copy()) == want).all()
