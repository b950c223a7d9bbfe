"""Attention of many queries over an 8-bit cache with and without the scratchpad that it asks for: a user's buffer (whatever
it held), none, one off the 16-byte boundaries, and launches that are recorded into graphs."""
import numpy as np
import pytest

import onednn_amd as dnnl
from onednn_amd import memory
from qmm_harness import T, dt
from test_gpu_sdpa import attention64, ctx, f16, f16_to_f64, reference_rule, say  # noqa: F401

pytestmark = pytest.mark.gpu
H, KV, Qn, S, D = 4, 2, 300, 333, 64


class Problem:
    def __init__(self, ctx, seed, scratchpad):
        self.eng, _ = ctx
        r = np.random.default_rng(seed)
        self.q = f16(r.standard_normal((1, H, Qn, D)))
        self.k, self.v = (r.integers(-128, 128, (1, KV, S, D)).astype(np.int8) for _ in range(2))
        self.sc = [f16(r.uniform(0.005, 0.02, (KV, S))) for _ in range(2)]
        attr = dnnl.primitive_attr()
        attr.set_scratchpad_mode(scratchpad)
        side = []
        for groups in ((D, 1), (1, D)):
            a = dnnl.primitive_attr()
            a.set_scales(dnnl.DNNL_ARG_WEIGHTS, 0b1110, list(groups), dt.f16)
            side.append(a)
        q_md = memory.desc([1, H, Qn, D], dt.f16, T("abcd"))
        kt_md = memory.desc([1, KV, D, S], dt.s8, T("abdc"))
        v_md = memory.desc([1, KV, S, D], dt.s8, T("abcd"))
        self.pd = dnnl.sdpa.primitive_desc(self.eng, q_md, kt_md, v_md, None, dt.f16, q_md, False, KV, True, attr, *side)
        self.out = memory(q_md, self.eng)
        vec = lambda raw: memory(memory.desc([raw.nbytes], dt.u8, T("a")), self.eng).write(raw)  # noqa: E731
        self.args = {dnnl.DNNL_ARG_QUERIES: memory(q_md, self.eng).write(self.q), dnnl.DNNL_ARG_KEYS: memory(kt_md, self.eng).write(self.k),
                     dnnl.DNNL_ARG_VALUES: memory(v_md, self.eng).write(self.v), dnnl.DNNL_ARG_DST: self.out,
                     dnnl.DNNL_ARG_SCALE: memory(memory.desc([1], dt.f16, T("a")), self.eng).write(f16(np.array([0.125]))),
                     dnnl.DNNL_ARG_ATTR_SCALES | dnnl.DNNL_ARG_KEYS: vec(self.sc[0]),
                     dnnl.DNNL_ARG_ATTR_SCALES | dnnl.DNNL_ARG_VALUES: vec(self.sc[1])}

    def check(self, what):
        kd, vd = (f16_to_f64(f16(x.astype(np.float64) * f16_to_f64(s)[None, :, :, None])) for x, s in zip((self.k, self.v), self.sc))
        gold = attention64(f16_to_f64(self.q), np.swapaxes(kd, -1, -2), vd, 0.125, None, True, H // KV)
        got = f16_to_f64(self.out.read(np.uint16, (1, H, Qn, D)))
        bad, total, worst = reference_rule(got, gold)
        print("[sdpa scratch] %s: %d of %d outside, max diff %.2e" % (what, bad, total, worst))
        assert bad <= total * 0.0006


@pytest.mark.parametrize("given", [False, True, "off"], ids=["none", "nan_filled", "off_the_boundary"])
def test_a_user_scratchpad_or_none(ctx, given):  # noqa: F811
    import torch
    say("sdpa scratchpad %s" % given)
    p = Problem(ctx, 5, dnnl.scratchpad_mode.user)
    md = p.pd.scratchpad_desc()
    assert md.get_size() == 2 * KV * S * D * 2
    if given:
        buf = torch.full((md.get_size() // 2 + 8,), float("nan"), dtype=torch.float16, device="cuda")
        torch.cuda.synchronize()
        p.args[dnnl.DNNL_ARG_SCRATCHPAD] = memory(md, p.eng, buf.data_ptr() + (2 if given == "off" else 0))
    dnnl.sdpa(p.pd).execute(ctx[1], p.args)
    ctx[1].wait()
    p.check(str(given))
    if given:
        assert torch.isnan(buf).all() if given == "off" else not torch.isnan(buf[:-8]).any()


def test_graphs_of_one_primitive_side_by_side(ctx):  # noqa: F811
    """Two graphs recorded from one primitive in library mode, with operands of their own, replayed at the same time on two
    streams after the primitive is gone: neither holds the library's scratchpad."""
    import gc
    import torch
    say("sdpa graphs side by side")
    probs = [Problem(ctx, seed, dnnl.scratchpad_mode.library) for seed in (5, 6)]
    prim = dnnl.sdpa(probs[0].pd)
    prim.execute(ctx[1], probs[0].args)
    ctx[1].wait()
    probs[0].check("eager")
    streams, graphs = [torch.cuda.Stream() for _ in probs], []
    for p, s in zip(probs, streams):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            prim.execute(dnnl.stream(p.eng, hip_stream=s.cuda_stream), p.args)
        graphs.append(g)
    del prim
    gc.collect()
    for turn in range(4):
        for p in probs:
            p.out.write(np.full((1, H, Qn, D), 0x7E00, np.uint16))
        torch.cuda.synchronize()
        for g, s in zip(graphs, streams):
            with torch.cuda.stream(s):
                for _ in range(20):
                    g.replay()
        torch.cuda.synchronize()
        for i, p in enumerate(probs):
            p.check("turn %d graph %d" % (turn, i))
