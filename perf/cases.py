"""The work this library is used for, one case per kind of call, for timing it end to end.

Every case is one execute() of a primitive through the public entry points (the `onednn_amd` mirror of `dnnl.hpp`) on
tensors that already live in device memory, as a PyTorch-ROCm program holds them: weights prepacked once through
`format_tag::any` and the reorder primitive, memory objects around the tensors' pointers, the primitive and its
argument table kept, torch's current stream. Kinds:

  w8a8    s8 / u8 activations x s8 weights, s32 accumulation: a scale per token (u8: one scale and zero point for the
          tensor), a scale per column, optional swish; bf16 or f32 result
  fp8     f8_e4m3 x f8_e4m3, one scale each, the result added to the bf16 tensor it is stored to (`sum`: a residual)
  w4      bf16 / f16 activations x u4 weights, groups of 128 k with an f16 scale and a u4 zero point
  w8      f16 activations x u8 weights, an f16 scale and a u8 zero point per column, optional swish
  w4a8    dynamic quantization: s8 activations x s4 weights, f16 scales per row and 128 k and per 128 k and column
  scores  batched s8 Q x s8 K^T, one scale each, f32 scores + the causal mask as a binary post-op
  sdpa    fused attention, K / V cache in the queries' type or 8 bit with an f16 scale and zero point per key; causal
          prefill, or one query per head against a long cache; grouped heads
"""
import math

import torch

import onednn_amd as dnnl
from onednn_amd import memory

dt, tag = memory.data_type, memory.format_tag
GROUP = 128
ELEM = {"s8": 1, "u8": 1, "bf16": 2, "f16": 2, "f32": 4}
DTYPE = {"s8": dt.s8, "u8": dt.u8, "bf16": dt.bf16, "f16": dt.f16, "f32": dt.f32}
TORCH = {"s8": torch.int8, "u8": torch.uint8, "bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _tag(letters):
    return 2 + tag._plain.index(letters)


def listed():
    return [
        # a small quantized layer, u8 activations with a zero point: 0.5 GOP, where latency and launches count
        dict(name="int8_small", kind="w8a8", m=256, k=1024, n=1024, src="u8", dst="f32", swish=False),
        # the up / gate projection of an LLM layer, W8A8, over a 4096-token prompt: the headline configuration
        dict(name="w8a8_prefill", kind="w8a8", m=4096, k=4096, n=14336, src="s8", dst="bf16", swish=True),
        # the same layer in a decode step of 64 sequences
        dict(name="w8a8_decode_batch", kind="w8a8", m=64, k=4096, n=14336, src="s8", dst="bf16", swish=False),
        # a large square fp8 product into a residual: the largest problem
        dict(name="fp8_residual", kind="fp8", m=8192, k=8192, n=8192),
        # one token through a 4-bit attention projection: the smallest call
        dict(name="w4_decode", kind="w4", m=1, k=4096, n=4096, src="bf16"),
        # a ragged 1000-token prompt through a 4-bit layer
        dict(name="w4_prefill", kind="w4", m=1000, k=4096, n=14336, src="f16"),
        # a 2176-token prompt through an 8-bit weights-only layer
        dict(name="w8_prefill", kind="w8", m=2176, k=4096, n=14336, dst="f16", swish=True),
        # one token, then the prompt, through a dynamically quantized layer with 4-bit weights
        dict(name="w4a8_decode", kind="w4a8", m=1, k=4096, n=14336),
        dict(name="w4a8_prefill", kind="w4a8", m=2176, k=4096, n=14336),
        # unfused attention scores of 32 heads over 2048 tokens
        dict(name="attention_scores", kind="scores", heads=32, tokens=2048, d=128),
        # causal attention over the same prompt, fused
        dict(name="attention_prefill", kind="sdpa", heads=32, kv_heads=32, queries=2048, keys=2048, d=128, src="f16",
             cache="native", causal=True),
        # one decode step of 32 heads against 8191 cached tokens in 8 bits
        dict(name="attention_decode", kind="sdpa", heads=32, kv_heads=32, queries=1, keys=8191, d=128, src="f16",
             cache="s8", causal=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(rng, lo, hi, of):
    return max(lo, _log(rng, lo, hi) // of * of)


MOST_FLOPS = 2.0 * 8192 ** 3 / 2  # half of the largest listed case


def draw(rng):
    kind = rng.choice(["w8a8", "fp8", "w4", "w8", "w4a8", "scores", "sdpa"])
    if kind == "scores":
        return dict(kind=kind, heads=rng.randint(4, 32), tokens=_log(rng, 64, 2048), d=rng.choice([64, 128]))
    if kind == "sdpa":
        d = rng.choice([64, 128])
        kv = rng.choice([4, 8, 16, 32])
        heads = kv * rng.choice([1, 1, 2, 4, 8])
        heads, kv = (heads, kv) if heads <= 40 else (32, kv)
        cache = rng.choice(["native", "native", "s8"])
        src = "f16" if cache == "s8" else rng.choice(["f16", "bf16"])
        if rng.random() < 0.5:
            q = _log(rng, 64, 4096)
            return dict(kind=kind, heads=heads, kv_heads=kv, queries=q, keys=q, d=d, src=src, cache=cache, causal=True)
        return dict(kind=kind, heads=heads, kv_heads=kv, queries=1, keys=_log(rng, 128, 32768), d=d, src=src, cache=cache,
                    causal=False)
    k = _multiple(rng, 1024, 14336, GROUP)
    n = _multiple(rng, 1024, 16384, 16)
    lo, hi = {"w8a8": (1, 4096), "fp8": (256, 8192), "w4": (1, 2048), "w8": (1, 4096), "w4a8": (1, 4096)}[kind]
    m = min(_log(rng, lo, hi), max(1, int(MOST_FLOPS / (2.0 * k * n))))
    c = dict(kind=kind, m=m, k=k, n=n)
    if kind == "w8a8":
        c.update(src=rng.choice(["s8", "s8", "u8"]), dst=rng.choice(["bf16", "bf16", "f32"]), swish=rng.random() < 0.5)
        c["n"] += rng.choice([0, 0, 0, 7])  # now and then a width that is not a multiple of anything
    elif kind == "w4":
        c.update(src=rng.choice(["bf16", "f16"]))
    elif kind == "w8":
        c.update(dst=rng.choice(["f16", "f16", "f32"]), swish=rng.random() < 0.5)
    return c


class _State:
    """A primitive, its stream, the argument table of one pass and the tensors behind it."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.eng = dnnl.engine(dnnl.engine.kind.gpu, 0)
        self.stream = dnnl.stream(self.eng, hip_stream=torch.cuda.current_stream().cuda_stream)
        self.args, self.keep, self.out = {}, [], None
        self.plain = None  # exact() sets a dict here, which then gets every operand as it was before any prepacking

    def normal(self, shape, std=1.0):
        return torch.randn(shape, generator=self.gen, device="cuda") * std

    def codes(self, shape, std, dtype=torch.int8):
        """round(N(0, 1) * std), clipped to +-127 (u8: around 128)."""
        x = self.normal(shape, std).round_().clamp_(-127, 127)
        return (x + 128).to(torch.uint8) if dtype == torch.uint8 else x.to(torch.int8)

    def integers(self, lo, hi, shape, dtype):
        return torch.randint(lo, hi, shape, generator=self.gen, device="cuda", dtype=dtype)

    def uniform(self, lo, hi, shape, dtype=torch.float32):
        return (torch.rand(shape, generator=self.gen, device="cuda") * (hi - lo) + lo).to(dtype)

    def memory(self, md, tensor):
        self.keep.append(tensor)
        return memory(md, self.eng, tensor.data_ptr())

    def bind(self, arg, md, tensor):
        if self.plain is not None:
            self.plain.setdefault(arg, tensor)
        self.args[arg] = self.memory(md, tensor)

    def vector(self, arg, code, tensor):
        self.bind(arg, memory.desc([tensor.numel()], code, _tag("a")), tensor)

    def packed(self, pd, plain_md, tensor):
        """Weights in the layout the primitive asked for, written by the reorder primitive."""
        if self.plain is not None:
            self.plain[dnnl.DNNL_ARG_WEIGHTS] = tensor
        md = pd.weights_desc()
        self.bind(dnnl.DNNL_ARG_WEIGHTS, md, torch.empty(md.get_size(), dtype=torch.uint8, device="cuda"))
        plain = memory(plain_md, self.eng, tensor.data_ptr())
        dnnl.reorder(plain, self.args[dnnl.DNNL_ARG_WEIGHTS]).execute(self.stream, plain, self.args[dnnl.DNNL_ARG_WEIGHTS])
        self.stream.wait()


SCALE_SRC = dnnl.DNNL_ARG_ATTR_SCALES | dnnl.DNNL_ARG_SRC
SCALE_WEI = dnnl.DNNL_ARG_ATTR_SCALES | dnnl.DNNL_ARG_WEIGHTS
ZERO_SRC = dnnl.DNNL_ARG_ATTR_ZERO_POINTS | dnnl.DNNL_ARG_SRC
ZERO_WEI = dnnl.DNNL_ARG_ATTR_ZERO_POINTS | dnnl.DNNL_ARG_WEIGHTS


def _linear(s, c):
    kind, m, k, n = c["kind"], c["m"], c["k"], c["n"]
    attr = dnnl.primitive_attr()
    po = dnnl.post_ops()
    f8 = torch.float8_e4m3fn
    src_dt, wei_dt, dst = {"w8a8": (c.get("src"), dt.s8, c.get("dst")), "fp8": ("fp8", dt.f8_e4m3, "bf16"),
                           "w4": (c.get("src"), dt.u4, c.get("src")), "w8": ("f16", dt.u8, c.get("dst")),
                           "w4a8": ("s8", dt.s4, "f16")}[kind]
    groups = k // GROUP
    plain_bytes = (k, n) if kind not in ("w4", "w4a8") else (k * n // 2,)
    out = None
    if kind == "w8a8":
        src = s.codes((m, k), 32, TORCH[src_dt])
        wei = s.integers(-127, 128, plain_bytes, torch.int8)
        if src_dt == "u8":
            attr.set_scales_mask(dnnl.DNNL_ARG_SRC, 0)
            attr.set_zero_points_mask(dnnl.DNNL_ARG_SRC, 0)
            s.vector(SCALE_SRC, dt.f32, s.uniform(0.015, 0.025, (1,)))
            s.vector(ZERO_SRC, dt.s32, torch.full((1,), 128, dtype=torch.int32, device="cuda"))
        else:
            attr.set_scales(dnnl.DNNL_ARG_SRC, 3, [1, k], dt.f32)
            s.vector(SCALE_SRC, dt.f32, s.uniform(0.005, 0.05, (m,)))
        attr.set_scales_mask(dnnl.DNNL_ARG_WEIGHTS, 2)
        s.vector(SCALE_WEI, dt.f32, s.uniform(0.0005, 0.005, (n,)))
    elif kind == "fp8":
        src = s.normal((m, k), 4).clamp_(-448, 448).to(f8)
        wei = s.normal((k, n), 4).clamp_(-448, 448).to(f8)
        attr.set_scales_mask(dnnl.DNNL_ARG_SRC, 0)
        attr.set_scales_mask(dnnl.DNNL_ARG_WEIGHTS, 0)
        s.vector(SCALE_SRC, dt.f32, torch.full((1,), 0.5, device="cuda"))
        s.vector(SCALE_WEI, dt.f32, torch.full((1,), 0.25, device="cuda"))
        po.append_sum(1.0)
        out = s.normal((m, n)).to(torch.bfloat16)
    elif kind == "w4":
        src = s.normal((m, k)).to(TORCH[src_dt])
        wei = s.integers(0, 256, plain_bytes, torch.uint8)  # two uniform nibbles a byte
        attr.set_fpmath_mode(dnnl.fpmath_mode.f16 if src_dt == "f16" else dnnl.fpmath_mode.bf16, True)
        attr.set_scales(dnnl.DNNL_ARG_WEIGHTS, 3, [GROUP, 1], dt.f16)
        attr.set_zero_points(dnnl.DNNL_ARG_WEIGHTS, 3, [GROUP, 1], dt.u4)
        s.vector(SCALE_WEI, dt.f16, s.uniform(0.005, 0.02, (groups, n), torch.float16))
        z = s.integers(6, 10, (groups * n // 2, 2), torch.uint8)
        s.vector(ZERO_WEI, dt.u8, z[:, 0] | (z[:, 1] << 4))
    elif kind == "w8":
        src = s.normal((m, k)).to(torch.float16)
        wei = s.integers(0, 256, plain_bytes, torch.uint8)
        attr.set_fpmath_mode(dnnl.fpmath_mode.f16, True)
        attr.set_scales(dnnl.DNNL_ARG_WEIGHTS, 2, [], dt.f16)
        attr.set_zero_points(dnnl.DNNL_ARG_WEIGHTS, 2, [], dt.u8)
        s.vector(SCALE_WEI, dt.f16, s.uniform(0.0005, 0.002, (n,), torch.float16))
        s.vector(ZERO_WEI, dt.u8, s.integers(100, 156, (n,), torch.uint8))
    else:
        src = s.codes((m, k), 40)
        wei = s.integers(0, 256, plain_bytes, torch.uint8)
        attr.set_scales(dnnl.DNNL_ARG_SRC, 3, [1, GROUP], dt.f16)
        attr.set_scales(dnnl.DNNL_ARG_WEIGHTS, 3, [GROUP, 1], dt.f16)
        s.vector(SCALE_SRC, dt.f16, s.uniform(0.005, 0.05, (m, groups), torch.float16))
        s.vector(SCALE_WEI, dt.f16, s.uniform(0.002, 0.02, (groups, n), torch.float16))
    if c.get("swish"):
        po.append_eltwise(dnnl.algorithm.eltwise_swish, 1.0, 0.0)
    if po.len():
        attr.set_post_ops(po)
    src_code = dt.f8_e4m3 if kind == "fp8" else DTYPE[src_dt]
    pd = dnnl.matmul.primitive_desc(s.eng, memory.desc([m, k], src_code, _tag("ab")), memory.desc([k, n], wei_dt, tag.any),
                                    memory.desc([m, n], DTYPE[dst], _tag("ab")), attr=attr)
    s.out = out if out is not None else torch.empty((m, n), dtype=TORCH[dst], device="cuda")
    s.bind(dnnl.DNNL_ARG_SRC, pd.src_desc(), src)
    s.bind(dnnl.DNNL_ARG_DST, pd.dst_desc(), s.out)
    s.packed(pd, memory.desc([k, n], wei_dt, _tag("ab")), wei)
    s.primitive = dnnl.matmul(pd)


def _scores(s, c):
    b, t, d = c["heads"], c["tokens"], c["d"]
    attr = dnnl.primitive_attr()
    attr.set_scales_mask(dnnl.DNNL_ARG_SRC, 0)
    attr.set_scales_mask(dnnl.DNNL_ARG_WEIGHTS, 0)
    mask_md = memory.desc([1, t, t], dt.f32, _tag("abc"))
    po = dnnl.post_ops()
    po.append_binary(dnnl.algorithm.binary_add, mask_md)
    attr.set_post_ops(po)
    pd = dnnl.matmul.primitive_desc(s.eng, memory.desc([b, t, d], dt.s8, _tag("abc")), memory.desc([b, d, t], dt.s8, tag.any),
                                    memory.desc([b, t, t], dt.f32, _tag("abc")), attr=attr)
    s.out = torch.empty((b, t, t), device="cuda")
    s.bind(dnnl.DNNL_ARG_SRC, pd.src_desc(), s.codes((b, t, d), 40))
    s.bind(dnnl.DNNL_ARG_DST, pd.dst_desc(), s.out)
    s.packed(pd, memory.desc([b, d, t], dt.s8, _tag("abc")), s.codes((b, d, t), 40))
    s.vector(SCALE_SRC, dt.f32, torch.full((1,), 0.01, device="cuda"))
    s.vector(SCALE_WEI, dt.f32, torch.full((1,), 0.012, device="cuda"))
    s.bind(dnnl.DNNL_ARG_ATTR_MULTIPLE_POST_OP(0) | dnnl.DNNL_ARG_SRC_1, mask_md,
           torch.triu(torch.full((t, t), -1e4, device="cuda"), 1))
    s.primitive = dnnl.matmul(pd)


def _sdpa(s, c):
    h, kv, q, keys, d = c["heads"], c["kv_heads"], c["queries"], c["keys"], c["d"]
    code, kind = DTYPE[c["src"]], TORCH[c["src"]]
    cache = dt.s8 if c["cache"] == "s8" else code
    q_md = memory.desc([1, h, q, d], code, _tag("abcd"))
    kt_md = memory.desc([1, kv, d, keys], cache, _tag("abdc"))  # the [keys, d] cache, seen as K^T
    v_md = memory.desc([1, kv, keys, d], cache, _tag("abcd"))
    s.bind(dnnl.DNNL_ARG_QUERIES, q_md, s.normal((h, q, d)).to(kind))
    s.vector(dnnl.DNNL_ARG_SCALE, code, torch.full((1,), d ** -0.5, device="cuda").to(kind))
    attrs = []
    for arg, md, groups in ((dnnl.DNNL_ARG_KEYS, kt_md, [d, 1]), (dnnl.DNNL_ARG_VALUES, v_md, [1, d])):
        attr = None
        if c["cache"] == "s8":
            attr = dnnl.primitive_attr()
            attr.set_scales(dnnl.DNNL_ARG_WEIGHTS, 0b1110, groups, dt.f16)
            attr.set_zero_points(dnnl.DNNL_ARG_WEIGHTS, 0b1110, groups, dt.s8)
            s.bind(arg, md, s.codes((kv, keys, d), 40))
            s.vector(dnnl.DNNL_ARG_ATTR_SCALES | arg, dt.f16, s.uniform(0.02, 0.04, (kv, keys), torch.float16))
            s.vector(dnnl.DNNL_ARG_ATTR_ZERO_POINTS | arg, dt.s8, s.integers(-6, 7, (kv, keys), torch.int8))
        else:
            s.bind(arg, md, s.normal((kv, keys, d)).to(kind))
        attrs.append(attr)
    s.out = torch.empty((1, h, q, d), dtype=kind, device="cuda")
    s.bind(dnnl.DNNL_ARG_DST, q_md, s.out)
    pd = dnnl.sdpa.primitive_desc(s.eng, q_md, kt_md, v_md, None, code, q_md, False, kv, c["causal"], None, attrs[0], attrs[1])
    s.primitive = dnnl.sdpa(pd)


def _fill(s, case):
    {"scores": _scores, "sdpa": _sdpa}.get(case["kind"], _linear)(s, case)
    return s


def prepare(case, seed):
    return _fill(_State(seed), case)


def run(state):
    state.primitive.execute(state.stream, state.args)
    return state.out


def work(case):
    c, kind = case, case["kind"]
    if kind == "scores":
        b, t, d = c["heads"], c["tokens"], c["d"]
        return {"bytes": 2 * b * t * d + 4 * t * t + 4 * b * t * t, "flops": 2.0 * b * t * t * d}
    if kind == "sdpa":
        h, kv, q, keys, d = c["heads"], c["kv_heads"], c["queries"], c["keys"], c["d"]
        seen = q * (q + 1) / 2.0 if c["causal"] else q * keys  # (query, key) pairs that are not masked
        cache = 2 * kv * keys * (d + 3) if c["cache"] == "s8" else 4 * kv * keys * d
        return {"bytes": 4 * h * q * d + cache, "flops": 4.0 * h * seen * d}
    m, k, n = c["m"], c["k"], c["n"]
    groups = k // GROUP
    nbytes = {"w8a8": lambda: m * k + k * n + m * n * ELEM[c["dst"]] + 4 * (m + n),
              "fp8": lambda: m * k + k * n + 4 * m * n,
              "w4": lambda: 2 * m * k + k * n // 2 + groups * n * 5 // 2 + 2 * m * n,
              "w8": lambda: 2 * m * k + k * n + 3 * n + m * n * ELEM[c["dst"]],
              "w4a8": lambda: m * k + k * n // 2 + 2 * groups * (m + n) + 2 * m * n}[kind]()
    return {"bytes": nbytes, "flops": 2.0 * m * k * n}


def tolerance(case):
    # About four times the distance of the results from a float64 evaluation of the same operands. It is the rounding of
    # the stored result wherever that is a 16-bit type.
    kind = case["kind"]
    if kind == "scores":
        return {"rel": 1e-6, "max": 1e-5}
    if kind == "sdpa":
        return {"rel": 6e-3, "max": 0.06} if case["src"] == "bf16" else {"rel": 1e-3, "max": 0.01}
    dst = {"fp8": "bf16", "w4": case.get("src"), "w4a8": "f16"}.get(kind, case.get("dst"))
    if dst == "f32":
        # (few rows of 8-bit weights: the offset of the byte -> float trick leaves through the sum of the activations)
        return {"rel": 1e-6, "max": 1e-5} if kind == "w8a8" else {"rel": 1e-4, "max": 6e-4}
    return {"rel": 6e-3, "max": 0.02} if dst == "bf16" else {"rel": 1e-3, "max": 3e-3}


def _nibbles(x, n, signed=False):
    """[rows, n] doubles out of bytes that hold two values each, the first in the low half."""
    v = torch.stack((x & 15, x >> 4), -1).reshape(-1, n).double()
    return torch.where(v > 7, v - 16, v) if signed else v


def exact(case, seed):
    """The outputs of run() for these inputs in float64, from the plain operands."""
    s = _State(seed)
    s.plain = {}
    _fill(s, case)
    c, kind, x = case, case["kind"], s.plain
    if kind == "scores":
        q, k = x[dnnl.DNNL_ARG_SRC].double(), x[dnnl.DNNL_ARG_WEIGHTS].double()
        scale = x[SCALE_SRC].double() * x[SCALE_WEI].double()
        mask = x[dnnl.DNNL_ARG_ATTR_MULTIPLE_POST_OP(0) | dnnl.DNNL_ARG_SRC_1].double()
        return torch.stack([q[b] @ k[b] * scale + mask for b in range(c["heads"])])
    if kind == "sdpa":
        q, scale = x[dnnl.DNNL_ARG_QUERIES].double(), x[dnnl.DNNL_ARG_SCALE].double()
        kv = []
        for arg in (dnnl.DNNL_ARG_KEYS, dnnl.DNNL_ARG_VALUES):
            t = x[arg].double()
            if c["cache"] == "s8":
                t = (t - x[dnnl.DNNL_ARG_ATTR_ZERO_POINTS | arg].double()[:, :, None]) * x[dnnl.DNNL_ARG_ATTR_SCALES | arg].double()[:, :, None]
            kv.append(t)
        hidden = torch.ones((c["queries"], c["keys"]), dtype=torch.bool, device="cuda").triu(1) if c["causal"] else None
        out = []
        for h in range(c["heads"]):
            g = h // (c["heads"] // c["kv_heads"])
            w = q[h] @ kv[0][g].t().contiguous() * scale
            if hidden is not None:
                w.masked_fill_(hidden, -math.inf)
            out.append(torch.softmax(w, -1) @ kv[1][g])
        return torch.stack(out)[None]
    k, n = c["k"], c["n"]
    src, wei = x[dnnl.DNNL_ARG_SRC].double(), x[dnnl.DNNL_ARG_WEIGHTS]
    if kind == "w8a8":
        if c["src"] == "u8":
            src = (src - x[ZERO_SRC].double()) * x[SCALE_SRC].double()
        else:
            src = src * x[SCALE_SRC].double()[:, None]
        wei = wei.double() * x[SCALE_WEI].double()
    elif kind == "fp8":
        wei = wei.double() * (x[SCALE_SRC].double() * x[SCALE_WEI].double())
    elif kind == "w8":
        wei = (wei.double() - x[ZERO_WEI].double()) * x[SCALE_WEI].double()
    else:
        wei = _nibbles(wei, n, signed=kind == "w4a8").view(-1, GROUP, n)
        if kind == "w4":
            wei = wei - _nibbles(x[ZERO_WEI], n)[:, None]
        else:
            src = (src.view(-1, k // GROUP, GROUP) * x[SCALE_SRC].double()[:, :, None]).view(-1, k)
        wei = (wei * x[SCALE_WEI].double()[:, None]).view(k, n)
    r = src @ wei
    if kind == "fp8":
        r += x[dnnl.DNNL_ARG_DST].double()  # this run() has not been called: still the residual
    return r * torch.sigmoid(r) if c.get("swish") else r
