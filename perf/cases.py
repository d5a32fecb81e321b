"""The work whose speed is measured: the operators and whole calls that a program makes through
this package, over the sizes, formats and options it uses them with.

The model shape is the package's own (QWEN25_05B: 24 layers, hidden 896, intermediate 4864, 14 query
and 2 kv heads of 64, vocabulary 151,936, context 2048); the wider matrices are generic. Weights are
N(0, 0.02) quantized to the two formats the kernels read: "sym" (two's-complement int4 with an f32
scale per 32, int8 per row for the table) and "ref" (unsigned codes with zero-points, blocks of 64).

Each case is a dict of plain values with an "op":
  gemv    one decode projection (matmul_q4_decode)
  plan    the decode projections of several layers that share K, batched (GemvPlan)
  head    the tied LM head: logits, the greedy token, or a sampled token
  gemm    one prefill projection (matmul_q4_prefill)
  swiglu  the prefill gate|up pair (eg_matmul_q4_prefill_swiglu)
  attn    the attention of one prompt chunk over an f16 or f32 cache (eg_attention_prefill[_f32])
  prompt  a whole prompt through the decoder (eg_decoder_prefill), logits and cache rows
  steps   decode steps through the decoder, a token read back per step as Session.generate does
"""

import ctypes
import math
from dataclasses import replace

import torch

from enargeia_amd import _lib
from enargeia_amd import kernels as K
from enargeia_amd.model import QWEN25_05B, Decoder, LayerDesc, ModelDesc, QuantMatrix, projection_shapes

DEV = "cuda"
VOCAB = QWEN25_05B.vocab


# ---- the cases ------------------------------------------------------------------------------


def listed():
    return [
        # the smallest call: one attention projection of a decode step, launch latency and host path
        dict(name="gemv 896x896 int4", op="gemv", n=896, k=896, bits=4, fmt="sym", bias=True),
        # a long-row down projection of a wider model, in the reference's shipped weight format
        dict(name="gemv 4096x11008 int4 ref", op="gemv", n=4096, k=11008, bits=4, fmt="ref", bias=False),
        # every K=896 projection of a decode step in one launch: the batched form of the headline
        dict(name="plan 24 layers K=896", op="plan", layers=24, hidden=896, fmt="sym"),
        # a sampled token from the tied table: head, penalty, top-p, draw (chat with sampling on)
        dict(name="head sample q8", op="head", rows=VOCAB, k=896, table="q8", fmt="sym", mode="sample", history=512),
        # a short ragged prompt through int8 down projections
        dict(name="gemm 37x896x4864 int8 ref", op="gemm", m=37, n=896, k=4864, bits=8, fmt="ref", bias=True),
        # the reference's prompt chunk (256 rows) through a gate projection
        dict(name="gemm 256x4864x896 int4", op="gemm", m=256, n=4864, k=896, bits=4, fmt="sym", bias=False),
        # a long prompt through a wider model's projection, reference format
        dict(name="gemm 2048x11008x4096 int4 ref", op="gemm", m=2048, n=11008, k=4096, bits=4, fmt="ref", bias=False),
        # the prompt MLP's first half over a long chunk
        dict(name="swiglu 1024x4864x896", op="swiglu", m=1024, n=4864, k=896, fmt="sym"),
        # a late chunk of a long prompt, on the default cache and on the exact one
        dict(name="attn f16 256 at 1792", op="attn", queries=256, begin=1792, heads=14, kv_heads=2, cache="f16"),
        dict(name="attn f32 256 at 1792", op="attn", queries=256, begin=1792, heads=14, kv_heads=2, cache="f32"),
        # a full-context prompt as one chunk: time to the first token
        dict(name="prompt 2048", op="prompt", layers=24, count=2048, begin=0, chunk=2048, cache="f16", fmt="sym"),
        # greedy generation at the end of the context, the captured step replayed
        dict(name="steps 8 at 2032", op="steps", layers=24, begin=2032, steps=8, cache="f16", fmt="sym", sampled=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["gemv", "gemv", "plan", "head", "head", "gemm", "gemm", "gemm", "swiglu", "attn", "attn", "prompt", "steps"])
    fmt = rng.choice(["sym", "ref"])
    block = 32 if fmt == "sym" else 64
    if op == "gemv":  # K from a small hidden size to a wide model's intermediate size
        bits = rng.choice([4, 4, 8])
        return dict(op=op, n=_log(rng, 64, 16384), k=block * _log(rng, 256 // block, 14336 // block), bits=bits, fmt=fmt,
                    bias=rng.random() < 0.4)
    if op == "plan":
        return dict(op=op, layers=rng.randint(1, 24), hidden=rng.choice([512, 896, 1024, 1536]), fmt=fmt)
    if op == "head":
        table = rng.choice(["q8", "q8", "f16", "f32"])
        mode = rng.choice(["sample", "argmax", "logits"]) if table == "q8" else rng.choice(["argmax", "logits"])
        return dict(op=op, rows=rng.choice([VOCAB, _log(rng, 4096, VOCAB)]), k=64 * rng.choice([8, 14, 16, 24]), table=table,
                    fmt=fmt, mode=mode, history=rng.randint(1, 2048))
    if op == "gemm":  # from one row to a whole prompt, odd row counts among them
        while True:
            c = dict(op=op, m=_log(rng, 1, 2048), n=_log(rng, 64, 11008), k=block * _log(rng, 256 // block, 8192 // block),
                     bits=rng.choice([4, 4, 4, 8]), fmt=fmt, bias=rng.random() < 0.4)
            if c["m"] * c["n"] * c["k"] <= 2048 * 11008 * 4096:
                return c
    if op == "swiglu":
        return dict(op=op, m=_log(rng, 1, 2048), n=4 * _log(rng, 64, 1216), k=block * _log(rng, 256 // block, 1920 // block), fmt=fmt)
    if op == "attn":
        heads, kv = rng.choice([(14, 2), (14, 2), (12, 2), (16, 2), (16, 8), (8, 8), (12, 12)])
        q = _log(rng, 1, 2048)
        return dict(op=op, queries=q, begin=rng.choice([0, rng.randint(0, 4096 - q)]), heads=heads, kv_heads=kv,
                    cache=rng.choice(["f16", "f16", "f32"]))
    if op == "prompt":
        cache = rng.choice(["f16", "f16", "f32"])
        count = _log(rng, 4, 2048)
        return dict(op=op, layers=rng.randint(2, 6 if cache == "f32" else 20), count=count,
                    begin=rng.choice([0, rng.randint(0, 2048 - count)]), chunk=rng.choice([256, 2048]), cache=cache, fmt=fmt)
    return dict(op=op, layers=rng.choice([4, 12, 24]), begin=rng.randint(1, 2032), steps=rng.randint(1, 12),
                cache=rng.choice(["f16", "f16", "f32"]), fmt=fmt, sampled=rng.random() < 0.4)


# ---- inputs ---------------------------------------------------------------------------------

_device = None


def device():
    """The program's one library device (its own stream), made on first use."""
    global _device
    if _device is None:
        _device = K.Device(0)
    return _device


class Quant:
    """One quantized matrix on the GPU: the three weight streams, and its values for exact()."""

    def __init__(self, gen, rows, cols, bits, fmt, block=None, sigma=0.02):
        self.bits = bits
        self.block = block or (32 if fmt == "sym" else 64)
        self.shape = (rows, cols)
        v = (torch.randn(rows * cols // self.block, self.block, device=DEV, generator=gen) * sigma)
        if fmt == "sym":
            self.encoding, top = K.ENC_SIGNED, 2 ** (bits - 1) - 1
            scale = v.abs().amax(1, keepdim=True) / top
            q = torch.round(v / scale).clamp_(-top - 1, top).to(torch.int16)
            self.zero, self.zeros = None, None
        else:
            self.encoding, levels = K.ENC_OFFSET_ZEROS, 2 ** bits - 1
            lo, hi = v.amin(1, keepdim=True), v.amax(1, keepdim=True)
            scale = (hi - lo) / levels
            zero = torch.round(-lo / scale).clamp_(0, levels)
            q = torch.round(v / scale + zero).clamp_(0, levels).to(torch.int16)
            self.zero = zero.to(torch.int16)
            self.zeros = self._pack(self.zero.reshape(-1))
        self.codes = q
        self.scale = scale
        self.scales = scale.reshape(-1).contiguous()
        self.packed = self._pack(q.reshape(-1))

    def _pack(self, c):
        per_word = 32 // self.bits
        if c.numel() % per_word:
            c = torch.cat([c, c.new_zeros(per_word - c.numel() % per_word)])
        c = c.to(torch.uint8) if c.min() >= 0 else (c & 0xFF).to(torch.uint8)
        if self.bits == 4:
            c = (c[0::2] & 15) | ((c[1::2] & 15) << 4)
        return c.contiguous().view(torch.int32)

    def values(self):
        """The dequantized matrix in float64."""
        c = self.codes.double()
        if self.zero is not None:
            c = c - self.zero.double()
        return (c * self.scale.double()).reshape(self.shape)

    def forget(self):
        """Leaves only what a program keeps: the streams."""
        self.codes = self.zero = self.scale = None
        return self

    def matrix(self):
        return QuantMatrix(self.packed.data_ptr(), self.scales.data_ptr(), None if self.zeros is None else self.zeros.data_ptr())


class Table:
    """A tied table stored as it is (f16 or f32)."""

    def __init__(self, gen, rows, cols, dtype):
        self.bits = 16 if dtype == "f16" else 32
        self.encoding, self.block, self.zeros, self.scales = K.ENC_SIGNED, cols, None, None
        v = torch.randn(rows, cols, device=DEV, generator=gen) * 0.02
        self.packed = v.half() if dtype == "f16" else v

    def values(self):
        return self.packed.double()

    def forget(self):
        return self


class Dims(ctypes.Structure):
    """eg_attention_prefill_dims"""

    _fields_ = [(f, ctypes.c_uint32) for f in
                ("queries", "keys", "query_begin", "heads", "kv_heads", "head_dim", "max_context")] + [("theta", ctypes.c_float)]


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(gen, *shape):
    return torch.randn(*shape, device=DEV, generator=gen)


def _p(t):
    return ctypes.c_void_p(None if t is None else t.data_ptr())


def _gemm_inputs(c, seed):
    g = _gen(seed)
    w = Quant(g, c["n"], c["k"], c["bits"], c["fmt"])
    x = _randn(g, c.get("m", 1), c["k"])
    return w, x, _randn(g, c["n"]) * 0.02 if c["bias"] else None


def _plan_shapes(c):
    """The projections of one layer that take the hidden vector's K, rows a multiple of 8."""
    h = c["hidden"]
    inter = 4864 if h == 896 else 4 * h
    return [h, 128, 128, h, inter, inter]


def _plan_inputs(c, seed):
    g = _gen(seed)
    mats = [Quant(g, n, c["hidden"], 4, c["fmt"]) for _ in range(c["layers"]) for n in _plan_shapes(c)]
    return mats, _randn(g, c["hidden"])


SAMPLING = K.SamplingParams(0.7, 0.9, 1.1)


def _head_inputs(c, seed):
    g = _gen(seed)
    # int8 tables: a scale per row ("sym") or blocks of 64 with zero-points, as shipped ("ref")
    t = Quant(g, c["rows"], c["k"], 8, c["fmt"], c["k"] if c["fmt"] == "sym" else 64) if c["table"] == "q8" else \
        Table(g, c["rows"], c["k"], c["table"])
    x = _randn(g, c["k"])
    hist = torch.randint(0, c["rows"], (c["history"],), device=DEV, generator=g, dtype=torch.int32)
    return t, x, hist, float(torch.rand(1, device=DEV, generator=g))


def _attn_inputs(c, seed):
    g = _gen(seed)
    q, b, h, kv = c["queries"], c["begin"], c["heads"], c["kv_heads"]
    ctx = max(2048, -(-(q + b) // 128) * 128)
    dt = torch.float16 if c["cache"] == "f16" else torch.float32
    caches = [_randn(g, ctx, kv, 64).to(dt) for _ in range(2)]
    return _randn(g, q, h, 64), _randn(g, q, kv, 64), _randn(g, q, kv, 64), caches


class Model:
    """The decoder's weights on the GPU, with the C description a program hands eg_decoder_create."""

    def __init__(self, c, seed, keep=False):
        g = _gen(seed)
        self.device = device()
        self.cfg = cfg = replace(QWEN25_05B, layers=c["layers"], group=32 if c["fmt"] == "sym" else 64)
        self.layers, self.layer_descs = [], (LayerDesc * cfg.layers)()
        for i in range(cfg.layers):
            L = {n: Quant(g, r, k, 4, c["fmt"]) for n, r, k in projection_shapes(cfg)}
            for n, r, _ in projection_shapes(cfg)[:3]:
                L[n + "_bias"] = _randn(g, r) * 0.02
            for n in ("input_norm", "post_attention_norm"):
                L[n] = 1.0 + 0.1 * _randn(g, cfg.hidden)
            d = self.layer_descs[i]
            for n, t in L.items():
                if isinstance(t, Quant):
                    setattr(d, n, t.matrix())
                    if not keep:
                        t.forget()
                else:
                    setattr(d, n, t.data_ptr())
            self.layers.append(L)
        self.table = Quant(g, cfg.vocab, cfg.hidden, 8, c["fmt"], cfg.hidden if c["fmt"] == "sym" else 64)
        if not keep:
            self.table.forget()
        self.final_norm = 1.0 + 0.1 * _randn(g, cfg.hidden)
        L0 = self.layers[0]["q"]
        self.desc = ModelDesc(cfg.layers, cfg.hidden, cfg.heads, cfg.kv_heads, cfg.head_dim, cfg.intermediate, cfg.vocab,
                              cfg.max_context, cfg.rms_eps, cfg.rope_theta, L0.encoding, 4, cfg.group, self.table.matrix(),
                              self.table.encoding, 8, self.table.block, self.final_norm.data_ptr(),
                              ctypes.cast(self.layer_descs, ctypes.POINTER(LayerDesc)))


def _decoder_inputs(c, seed):
    """Token ids and the cache rows that are there before the call ([layers][rows][kv][64])."""
    g = _gen(seed + (1 << 20))
    cfg = QWEN25_05B
    count = c["count"] if c["op"] == "prompt" else 1
    ids = torch.randint(0, cfg.vocab, (count,), device=DEV, generator=g)
    rows = [_randn(g, c["layers"], c["begin"], cfg.kv_heads, cfg.head_dim).to(_cache_type(c)) for _ in range(2)]
    return ids, rows


def _cache_type(c):
    return torch.float16 if c["cache"] == "f16" else torch.float32


class _Handle:
    """A decoder, closed when nothing refers to it or to its buffers any more."""

    def __init__(self, dec):
        self.dec = dec

    def __del__(self):
        self.dec.close()


class _Raw:
    """A buffer of a decoder as torch sees it; keeps the decoder."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "strides": None, "version": 2}


class Calls:
    """A decoder and what the calls on it take and give."""

    def __init__(self, c, seed):
        self.c = c
        self.model = Model(c, seed)
        ids, rows = _decoder_inputs(c, seed)
        torch.cuda.synchronize()  # the weights are there before the decoder reads them
        self.dec = Decoder(self.model, c["cache"])
        owner = _Handle(self.dec)
        cfg, b = self.model.cfg, self.dec.buffers
        shape = (cfg.layers, cfg.max_context, cfg.kv_heads, cfg.head_dim)
        kind = "<f2" if c["cache"] == "f16" else "<f4"
        self.k = torch.as_tensor(_Raw(owner, b.k_cache, shape, kind), device=DEV)
        self.v = torch.as_tensor(_Raw(owner, b.v_cache, shape, kind), device=DEV)
        self.logits = torch.as_tensor(_Raw(owner, b.logits, (cfg.vocab,), "<f4"), device=DEV)
        self.k.zero_()
        self.v.zero_()
        self.k[:, :c["begin"]].copy_(rows[0])
        self.v[:, :c["begin"]].copy_(rows[1])
        self.ids = [int(t) for t in ids.cpu()]
        torch.cuda.synchronize()
        end = c["begin"] + (c["count"] if c["op"] == "prompt" else c["steps"])
        self.out = {"logits": self.logits, "k": self.k[:, c["begin"]:end], "v": self.v[:, c["begin"]:end]}
        if c["op"] == "prompt":
            self.dec.set_prefill_chunk(min(c["chunk"], cfg.max_context))
        else:
            if c["sampled"]:
                self.dec.set_sampling(SAMPLING.temperature, SAMPLING.top_p, SAMPLING.repetition_penalty)
            self.dec.capture()

    def run(self):
        c = self.c
        if c["op"] == "prompt":
            self.dec.prefill(c["begin"], self.ids, read_token=False)
            return self.out
        # a continued generation: its history, draw source and position, then the steps
        self.dec.seed(0x5EED)
        self.dec.set_history(self.ids)
        self.dec.reset(c["begin"], self.ids[0])
        tokens = [self.dec.step() for _ in range(c["steps"])]
        return {"tokens": tokens, **self.out}


class Plan:
    """The batched projections of a decode step, planned once."""

    def __init__(self, c, seed):
        self.mats, self.x = _plan_inputs(c, seed)
        rows = [m.shape[0] for m in self.mats]
        self.out = torch.empty(sum(rows), device=DEV)
        at, segs = 0, []
        for m, n in zip(self.mats, rows):
            segs.append((m.packed, m.scales, m.zeros, None, self.out, n, at))
            at += n
            m.forget()
        torch.cuda.synchronize()
        self.plan = K.GemvPlan(device(), c["hidden"], self.mats[0].block, segs, 4, self.mats[0].encoding)

    def run(self):
        self.plan.launch(self.x)
        return self.out

    def __del__(self):
        plan = getattr(self, "plan", None)
        if plan is not None:
            plan.destroy()


def prepare(case, seed):
    c, dev = case, device()
    op = c["op"]
    if op in ("prompt", "steps"):
        return Calls(c, seed)
    if op == "plan":
        return Plan(c, seed)
    if op in ("gemv", "gemm"):
        w, x, bias = _gemm_inputs(c, seed)
        w.forget()
        m = c.get("m", 1)
        out = torch.empty(m, c["n"], device=DEV)
        base = K.MATMUL_Q4_DECODE if op == "gemv" else K.MATMUL_Q4_PREFILL
        kern = K.ComputeKernel(dev, K.with_format(base, c["bits"], w.encoding))
        u = kern.uniform()
        u.write(K.matmul_q4_dims(m, c["n"], c["k"], bias is not None, w.block))
        group = kern.bind_group([x, w.packed, w.scales, w.zeros, bias, out, u])
        grid = K.matmul_q4_decode_workgroups(c["n"]) if op == "gemv" else K.matmul_q4_prefill_workgroups(m, c["n"])
        return lambda: (kern.encode(group, grid), out)[1]
    if op == "head":
        t, x, hist, rnd = _head_inputs(c, seed)
        t.forget()
        out = torch.empty(c["rows"], device=DEV)
        token = torch.zeros(2, device=DEV, dtype=torch.int32)
        dims = K.embedding_dims(1, c["k"], 0, c["rows"], t.block)
        if c["mode"] == "logits":
            kern = K.ComputeKernel(dev, K.embedding_head_spec(c["table"], t.encoding))
            u = kern.uniform()
            u.write(dims)
            group = kern.bind_group([x, t.packed, t.scales, t.zeros, out, u])
            grid = K.embedding_head_workgroups(c["rows"])
            return lambda: (kern.encode(group, grid), out)[1]
        if c["mode"] == "argmax":
            return lambda: (K.lm_head_argmax(dev, x, t.packed, t.scales, t.zeros, out, token, dims, t.bits, t.encoding),
                            {"logits": out, "token": token[:1]})[1]
        sample = K.sample_dims(c["rows"], c["history"], SAMPLING, rnd)
        return lambda: (K.lm_head_sample(dev, x, t.packed, t.scales, t.zeros, out, hist, token, dims, sample, t.bits, t.encoding),
                        {"logits": out, "token": token[:1]})[1]
    lib = _lib.load()
    if op == "swiglu":
        g = _gen(seed)
        gate, up = (Quant(g, c["n"], c["k"], 4, c["fmt"]).forget() for _ in range(2))
        x = _randn(g, c["m"], c["k"])
        out, scratch = torch.empty(c["m"], c["n"], device=DEV), torch.empty(c["m"], 2 * c["n"], device=DEV)
        d = K.MatmulDims.from_buffer_copy(K.matmul_q4_dims(c["m"], c["n"], c["k"], False, gate.block))

        def swiglu():
            _lib.check(lib.eg_matmul_q4_prefill_swiglu(
                dev.ctx, _p(x), _p(gate.packed), _p(gate.scales), _p(gate.zeros), _p(up.packed), _p(up.scales), _p(up.zeros),
                _p(out), _p(scratch), ctypes.byref(d), gate.encoding, 4), dev.ctx)
            return out
        return swiglu
    q, k, v, (kc, vc) = _attn_inputs(c, seed)
    n, b = c["queries"], c["begin"]
    q_rope, out = torch.empty_like(q), torch.empty_like(q)
    d = Dims(n, b + n, b, c["heads"], c["kv_heads"], 64, kc.shape[0], QWEN25_05B.rope_theta)
    fn = lib.eg_attention_prefill if c["cache"] == "f16" else lib.eg_attention_prefill_f32

    def attention():
        _lib.check(fn(dev.ctx, _p(q), _p(k), _p(v), _p(kc), _p(vc), _p(q_rope), _p(out), ctypes.byref(d)), dev.ctx)
        return {"out": out, "q": q_rope, "k": kc[b:b + n], "v": vc[b:b + n]}
    return attention


def run(state):
    return state() if callable(state) else state.run()


# ---- what a pass cannot do without ------------------------------------------------------------


def _weight_bytes(n, k, bits, fmt, block=None):
    block = block or (32 if fmt == "sym" else 64)
    blocks = n * k // block
    return n * k * bits // 8 + 4 * blocks + (blocks * bits // 8 if fmt == "ref" else 0)


def _layer_weights():
    return [(n, k) for _, n, k in projection_shapes(QWEN25_05B)]


def work(case):
    c = case
    op = c["op"]
    if op in ("gemv", "gemm"):
        m, n, k = c.get("m", 1), c["n"], c["k"]
        return {"bytes": _weight_bytes(n, k, c["bits"], c["fmt"]) + 4 * (m * k + m * n + (n if c["bias"] else 0)), "flops": 2 * m * n * k}
    if op == "plan":
        rows, k = _plan_shapes(c) * c["layers"], c["hidden"]
        return {"bytes": sum(_weight_bytes(n, k, 4, c["fmt"]) + 4 * n for n in rows) + 4 * k, "flops": 2 * k * sum(rows)}
    if op == "head":
        n, k = c["rows"], c["k"]
        w = _weight_bytes(n, k, 8, c["fmt"], k if c["fmt"] == "sym" else 64) if c["table"] == "q8" else n * k * (2 if c["table"] == "f16" else 4)
        return {"bytes": w + 4 * (n + k) + (4 * c["history"] if c["mode"] == "sample" else 0), "flops": 2 * n * k}
    if op == "swiglu":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 2 * _weight_bytes(n, k, 4, c["fmt"]) + 4 * (m * k + m * n), "flops": 4 * m * n * k}
    seen = lambda n, b: n * b + n * (n + 1) // 2  # noqa: E731  (query, key) pairs of a causal chunk
    if op == "attn":
        n, b, h, kv, e = c["queries"], c["begin"], c["heads"], c["kv_heads"], 2 if c["cache"] == "f16" else 4
        return {"bytes": 64 * (4 * 3 * n * h + 4 * 2 * n * kv + 2 * e * (b + 2 * n) * kv), "flops": 4 * 64 * h * seen(n, b)}
    cfg, n = QWEN25_05B, c["count"] if op == "prompt" else c["steps"]
    kv, e, b = cfg.kv_heads * cfg.head_dim, 2 if c["cache"] == "f16" else 4, c["begin"]
    per_layer = sum(r * k for r, k in _layer_weights())
    weights = c["layers"] * sum(_weight_bytes(r, k, 4, c["fmt"]) for r, k in _layer_weights())
    head = _weight_bytes(cfg.vocab, cfg.hidden, 8, c["fmt"], cfg.hidden if c["fmt"] == "sym" else 64) + 4 * cfg.vocab
    attention = c["layers"] * 4 * cfg.hidden * seen(n, b)
    if op == "prompt":
        return {"bytes": weights + head + n * cfg.hidden + c["layers"] * 2 * e * kv * (b + n),
                "flops": 2 * c["layers"] * per_layer * n + attention + 2 * cfg.vocab * cfg.hidden}
    return {"bytes": n * (weights + head) + c["layers"] * 2 * e * kv * (seen(n, b) + n),
            "flops": n * 2 * (c["layers"] * per_layer + cfg.vocab * cfg.hidden) + attention}


def tolerance(case):
    """About four times what the path differs from exact() by (measured: f32 sums 4e-7, bf16 operands
    2.3e-3 to 3.4e-3, f16 operands 2.8e-4, a whole prompt 1.4e-2)."""
    op = case["op"]
    if op in ("gemv", "plan", "head"):  # f32 products and sums
        return {"rel": 4e-6}
    if op in ("gemm", "swiglu"):  # bf16 operands, f32 sums
        return {"rel": 1e-2}
    if op == "attn":  # f16 operands (q and the softmax weights), or f32 throughout
        return {"rel": 1.2e-3 if case["cache"] == "f16" else 4e-6}
    if op == "prompt":  # bf16 roundings that travel through the layers
        return {"rel": 0.03, "max": 0.5}
    return {"rel": 1e-3}  # f32 steps; the new rows are rounded to the cache's type


# ---- the same in 64 bits ----------------------------------------------------------------------


def _rope(x, begin, theta):
    """x [rows][heads][64]: pairs (e, e + 32) rotated by (begin + row) * theta^(-e / 32)."""
    n, half = x.shape[0], x.shape[2] // 2
    angle = (begin + torch.arange(n, device=DEV, dtype=torch.float64))[:, None] * \
        theta ** (-torch.arange(half, device=DEV, dtype=torch.float64) / half)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)


def _attend(q, k, v, begin):
    """q [n][heads][64] at positions begin.., k and v [begin + n][kv][64]."""
    n, heads, _ = q.shape
    group = heads // k.shape[1]
    out = torch.empty_like(q)
    mask = torch.arange(begin + n, device=DEV)[None] > begin + torch.arange(n, device=DEV)[:, None]
    for h in range(heads):
        s = (q[:, h] @ k[:, h // group].t().contiguous()) * 0.125
        out[:, h] = torch.softmax(s.masked_fill_(mask, -math.inf), 1) @ v[:, h // group].contiguous()
    return out


def _norm(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _forward(model, ids, begin, ks, vs, cache):
    """The rows `ids` at begin.. through the layers; ks and vs hold the earlier rows per layer and
    receive the new ones, rounded to the cache's type where they are read. Returns the last logits
    and the new rows as computed."""
    cfg = model.cfg
    h = _rows_of(model.table, ids)
    new_k, new_v = [], []
    for i, L in enumerate(model.layers):
        x = _norm(h, L["input_norm"], cfg.rms_eps)
        q, k, v = ((x @ L[n].values().t() + L[n + "_bias"].double()).reshape(len(ids), -1, 64) for n in ("q", "k", "v"))
        q, k = _rope(q, begin, cfg.rope_theta), _rope(k, begin, cfg.rope_theta)
        new_k.append(k)
        new_v.append(v)
        ks[i] = torch.cat([ks[i], k.to(cache).double()])
        vs[i] = torch.cat([vs[i], v.to(cache).double()])
        h = h + _attend(q, ks[i], vs[i], begin).reshape(len(ids), -1) @ L["o"].values().t()
        x = _norm(h, L["post_attention_norm"], cfg.rms_eps)
        g, u = x @ L["gate"].values().t(), x @ L["up"].values().t()
        h = h + (g / (1 + torch.exp(-g)) * u) @ L["down"].values().t()
    x = _norm(h[-1:], model.final_norm, cfg.rms_eps)
    return _times_table(model.table, x[0]), new_k, new_v


def _rows_of(t, ids):
    per = t.shape[1] // t.block
    at = (torch.as_tensor(ids, device=DEV)[:, None] * per + torch.arange(per, device=DEV)).reshape(-1)
    c = t.codes[at].double() - (0 if t.zero is None else t.zero[at].double())
    return (c * t.scale[at].double()).reshape(len(ids), -1)


def _times_table(t, x):
    """The table times x, a part at a time (the whole in 64 bits takes a gigabyte)."""
    step, n = 16384, t.shape[0]
    return torch.cat([_rows_of(t, torch.arange(a, min(a + step, n), device=DEV)) @ x for a in range(0, n, step)])


def _penalized(logits, history, penalty):
    ids = torch.unique(history.long())
    v = logits[ids]
    logits[ids] = torch.where(v > 0, v / penalty, v * penalty)
    return logits


def exact(case, seed):
    c = case
    op = c["op"]
    if op in ("gemv", "gemm"):
        w, x, bias = _gemm_inputs(c, seed)
        y = x.double() @ w.values().t()
        return y if bias is None else y + bias.double()
    if op == "plan":
        mats, x = _plan_inputs(c, seed)
        return torch.cat([m.values() @ x.double() for m in mats])
    if op == "head":
        t, x, hist, _ = _head_inputs(c, seed)
        y = (t.values() @ x.double()) if c["table"] != "q8" else _times_table(t, x.double())
        if c["mode"] == "logits":
            return y
        if c["mode"] == "sample":
            y = _penalized(y, hist, float(torch.tensor(SAMPLING.repetition_penalty, dtype=torch.float32)))
        return {"logits": y, "token": None}
    if op == "swiglu":
        g = _gen(seed)
        gate, up = (Quant(g, c["n"], c["k"], 4, c["fmt"]) for _ in range(2))
        x = _randn(g, c["m"], c["k"]).double()
        a, b = x @ gate.values().t(), x @ up.values().t()
        return a / (1 + torch.exp(-a)) * b
    if op == "attn":
        q, k, v, (kc, vc) = _attn_inputs(c, seed)
        b, theta = c["begin"], QWEN25_05B.rope_theta
        qr, kr = _rope(q.double(), b, theta), _rope(k.double(), b, theta)
        keys = torch.cat([kc[:b].double(), kr.to(kc.dtype).double()])
        vals = torch.cat([vc[:b].double(), v.to(vc.dtype).double()])
        return {"out": _attend(qr, keys, vals, b), "q": qr * 0.125, "k": kr, "v": v.double()}
    model = Model(c, seed, keep=True)
    ids, rows = _decoder_inputs(c, seed)
    ks, vs = (list(r.double()) for r in rows)
    if op == "prompt":
        # chunks attend to the rows before them: the same sums as one chunk, so one chunk here
        logits, k, v = _forward(model, ids, c["begin"], ks, vs, _cache_type(c))
        return {"logits": logits, "k": torch.stack(k), "v": torch.stack(v)}
    if c["sampled"]:
        return None  # the draw decides the tokens
    got_k, got_v, ids = [], [], ids.tolist()
    for s in range(c["steps"]):
        logits, k, v = _forward(model, ids, c["begin"] + s, ks, vs, _cache_type(c))
        got_k.append(torch.stack(k))
        got_v.append(torch.stack(v))
        ids = [int(logits.argmax())]
    return {"tokens": [None] * c["steps"], "logits": logits, "k": torch.cat(got_k, 1), "v": torch.cat(got_v, 1)}
