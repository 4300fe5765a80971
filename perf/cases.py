"""Performance cases of the dense-contraction path, through its public entry points.

Each case is what a program that serves a model with this library does between two points where it
looks at results: one Gemm, one feed-forward block, one attention step, the projections of one decoder
layer, a quantised convolution. Sizes are those of bench.py and of the tests where they name some,
else generic ones; `draw` spreads the same kinds over the sizes, data types and options they are
called with.

Inputs are torch tensors on the GPU made from the seed; the library reads them in place and writes
into torch buffers the case keeps (or, for graph sessions and operators, into its own pooled storage,
which is returned to the pool when the next pass begins, as a program does after reading a result).
"""
import math

import torch

from ingot_amd import DeviceTensor, Graph, Session, Weight
from ingot_amd import _lib as L

DT = {torch.float32: L.DT_F32, torch.bfloat16: L.DT_BF16, torch.int8: L.DT_I8, torch.uint8: L.DT_U8,
      torch.int32: L.DT_I32}
ACT = {"none": L.ACT_NONE, "relu": L.ACT_RELU, "gelu": L.ACT_GELU_ERF, "silu": L.ACT_SILU}


def _decoder(case):
    """(K, N) of a decoder layer's projections: QKV, attention output, gate+up, down (bench.py's decode workload at
    hidden 2048, inner 5632)."""
    h, f = case["hidden"], case["inner"]
    return (h, 3 * h), (h, h), (h, 2 * f), (f, h)


def listed():
    return [
        # The smallest call a user makes: one Gemm + bias + ReLU of a small classifier (latency and launch).
        dict(name="gemm_relu", kind="gemm", m=128, k=256, n=512, weight="f32", math="auto", act="relu", trans_a=False),
        # An encoder's feed-forward block as a compiled graph session, f32 throughout.
        dict(name="encoder_ffn", kind="ffn", m=1024, hidden=768, inner=3072, half=False),
        # The two batched products of an encoder's self-attention: 8 sequences of 128 tokens, 12 heads of 64.
        dict(name="attention", kind="attention", items=96, sq=128, sk=128, d=64, dtype="f32"),
        # The quantised feed-forward product, dequantised in the store.
        dict(name="int8_ffn_up", kind="int8", m=1024, k=768, n=3072, a="u8", out="f32"),
        # A quantised convolution of a residual stage (the test suite's large shape).
        dict(name="qconv_3x3", kind="qconv", n=1, c=256, h=56, w=56, m=256, ks=3, group=1, stride=1),
        # A quantised depthwise convolution of a mobile network, a small batch of images.
        dict(name="qconv_depthwise", kind="qconv", n=8, c=96, h=56, w=56, m=96, ks=3, group=96, stride=1),
        # One token through a decoder layer's projections, bf16 weights (HBM-bound).
        dict(name="decode_1", kind="decoder", m=1, hidden=2048, inner=5632, weight="bf16", math="auto"),
        # Sixteen sequences decoded together.
        dict(name="decode_16", kind="decoder", m=16, hidden=2048, inner=5632, weight="bf16", math="auto"),
        # One token, weights quantised to int8 in groups of 64.
        dict(name="decode_1_int8", kind="decoder", m=1, hidden=2048, inner=5632, weight="int8", math="auto"),
        # A prompt of odd length through the same layer, f32 activations at f32-class accuracy.
        dict(name="prefill_517", kind="decoder", m=517, hidden=2048, inner=5632, weight="bf16", math="auto"),
        # A diffusion transformer block's large products in bf16, hidden activations kept in bf16.
        dict(name="dit_block", kind="dit", m=4096, hidden=3072, qkv=9216, inner=12288),
        # What follows an unfused integer product: DequantizeLinear per column, then Gelu, as operators.
        dict(name="dequant_gelu", kind="nodes", rows=1024, cols=3072, x="i32", axis=1),
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("gemm", "gemm", "ffn", "attention", "attention", "int8", "qconv", "qconv", "decoder", "decoder",
                       "decoder", "dit", "nodes"))
    if kind == "gemm":
        weight = rng.choice(("f32", "f32", "bf16"))
        return dict(kind=kind, m=_size(rng, 1, 2048), k=_size(rng, 16, 4096), n=_size(rng, 16, 4096), weight=weight,
                    math=rng.choice(("auto", "bf16")) if weight == "bf16" else "auto",
                    act=rng.choice(("none", "relu", "gelu", "silu")), trans_a=rng.random() < 0.15)
    if kind == "ffn":
        hidden = 64 * rng.randint(4, 16)
        return dict(kind=kind, m=_size(rng, 16, 2048), hidden=hidden, inner=4 * hidden, half=rng.random() < 0.5)
    if kind == "attention":
        sk = _size(rng, 16, 512)
        return dict(kind=kind, items=_size(rng, 8, 128), sq=sk, sk=sk, d=rng.choice((32, 64, 80, 128)),
                    dtype=rng.choice(("f32", "f32", "bf16")))
    if kind == "int8":
        return dict(kind=kind, m=_size(rng, 1, 2048), k=_size(rng, 64, 4096), n=_size(rng, 64, 4096),
                    a=rng.choice(("u8", "i8")), out=rng.choice(("f32", "i32", "u8")))
    if kind == "qconv":
        ks, stride = rng.choice((1, 3, 3, 5)), rng.choice((1, 1, 2))
        depthwise = ks > 1 and rng.random() < 0.4
        c = 8 * _size(rng, 2, 48) if depthwise else _size(rng, 3, 256)
        side = _size(rng, 7, 64)
        return dict(kind=kind, n=rng.choice((1, 1, 4, 8)), c=c, h=side, w=max(7, side - rng.randint(0, 3)),
                    m=c if depthwise else 8 * _size(rng, 2, 32), ks=ks, group=c if depthwise else 1, stride=stride)
    if kind == "decoder":
        weight = rng.choice(("bf16", "bf16", "int8"))
        m = _size(rng, 1, 16) if weight == "int8" or rng.random() < 0.5 else _size(rng, 17, 1024)
        hidden = 256 * rng.randint(4, 14)
        return dict(kind=kind, m=m, hidden=hidden, inner=256 * round(2.75 * hidden / 256), weight=weight,
                    math=rng.choice(("auto", "auto", "bf16")) if weight == "bf16" else "auto")
    if kind == "dit":
        hidden = 256 * rng.randint(4, 12)
        return dict(kind=kind, m=_size(rng, 256, 4096), hidden=hidden, qkv=3 * hidden, inner=4 * hidden)
    return dict(kind=kind, rows=_size(rng, 16, 4096), cols=_size(rng, 64, 4096), x=rng.choice(("i32", "u8", "i8")),
                axis=rng.choice((0, 1, -1)))


# ---- inputs ----

def _inputs(case, seed):
    """The case's tensors, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))

    def normal(*shape, scale=1.0):
        return torch.randn(shape, generator=g, device="cuda") * scale

    def whole(lo, hi, dtype, *shape):
        return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=dtype)

    def uniform(lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(shape, generator=g, device="cuda")

    def octets(which, *shape):
        return whole(0, 256, torch.uint8, *shape) if which == "u8" else whole(-128, 128, torch.int8, *shape)

    kind, t = case["kind"], {}
    if kind == "gemm":
        m, k, n = case["m"], case["k"], case["n"]
        t["a"] = uniform(-1, 1, *((k, m) if case["trans_a"] else (m, k)))
        t["w"] = uniform(-1, 1, n, k).to(torch.float32 if case["weight"] == "f32" else torch.bfloat16)
        t["bias"] = normal(n, scale=0.1)
    elif kind == "ffn":
        h, i = case["hidden"], case["inner"]
        t["x"] = normal(case["m"], h)
        t["W1"], t["b1"] = normal(h, i, scale=0.02), normal(i, scale=0.02)
        t["W2"], t["b2"] = normal(i, h, scale=0.02), normal(h, scale=0.02)
    elif kind == "attention":
        z, sq, sk, d = case["items"], case["sq"], case["sk"], case["d"]
        dt = torch.float32 if case["dtype"] == "f32" else torch.bfloat16
        t["q"], t["k"], t["v"] = normal(z, sq, d).to(dt), normal(z, sk, d).to(dt), normal(z, sk, d).to(dt)
        t["p"] = torch.softmax(normal(z, sq, sk), dim=-1).to(dt)  # the probabilities the second product reads
    elif kind == "int8":
        m, k, n = case["m"], case["k"], case["n"]
        t["a"] = octets(case["a"], m, k)
        t["w"] = whole(-127, 128, torch.int8, k, n)
        t["scale"] = uniform(0.001, 0.01, n) * 0.02
    elif kind == "qconv":
        cg = case["c"] // case["group"]
        t["x"] = octets("u8", case["n"], case["c"], case["h"], case["w"])
        t["w"] = whole(-128, 128, torch.int8, case["m"], cg, case["ks"], case["ks"])
        t["bias"] = whole(-1024, 1024, torch.int32, case["m"])
        # multipliers that spread the outputs over the u8 range
        t["mult"] = uniform(0.5, 1.5, case["m"]) * (48.0 / (74.0 * 74.0 * math.sqrt(cg * case["ks"] ** 2)))
    elif kind == "decoder":
        for i, (k, n) in enumerate(_decoder(case)):
            t["x%d" % i] = normal(case["m"], k)
            t["w%d" % i] = normal(n, k, scale=0.02).to(torch.bfloat16)
    elif kind == "dit":
        h = case["hidden"]
        t["x0"], t["x1"] = normal(case["m"], h), normal(case["m"], h)
        t["w0"] = normal(case["qkv"], h, scale=0.02).to(torch.bfloat16)
        t["w1"] = normal(case["inner"], h, scale=0.02).to(torch.bfloat16)
        t["w2"] = normal(h, case["inner"], scale=0.02).to(torch.bfloat16)
    else:
        r, c, axis = case["rows"], case["cols"], case["axis"]
        if case["x"] == "i32":
            t["x"] = whole(-20000, 20000, torch.int32, r, c)
        else:
            t["x"] = octets(case["x"], r, c)
        ns = 1 if axis < 0 else (r, c)[axis]
        t["scale"] = uniform(0.5, 1.5, ns) * (2.0 / (10000.0 if case["x"] == "i32" else 100.0))
        if case["x"] != "i32":
            t["zp"] = whole(120, 136, torch.uint8, ns) if case["x"] == "u8" else whole(-8, 8, torch.int8, ns)
    return t


# ---- the program's side ----

_session = None


def _sess():
    global _session
    if _session is None:
        _session = Session(0)
    return _session


class _Pooled:
    """A pooled result of the library as torch sees it."""

    KINDS = {L.DT_F32: "<f4", L.DT_I32: "<i4", L.DT_U8: "|u1", L.DT_I8: "|i1"}

    def __init__(self, t):
        self.__cuda_array_interface__ = {"shape": t.shape, "typestr": self.KINDS[t.dtype], "data": (t.ptr, False),
                                         "version": 2}


class _State:
    """What the program keeps between passes: inputs, packed weights, output buffers, prepared calls."""

    def __init__(self):
        self.t, self.weights, self.closers, self.results, self.out, self.calls = {}, [], [], [], [], []

    def release(self):
        for r in self.results:
            r.free()
        self.results = []

    def __del__(self):
        self.release()
        for o in self.closers:
            o.free()
        for w in self.weights:
            w.free()


def _dev(t):
    return DeviceTensor(_sess(), DT[t.dtype], t.shape, t.data_ptr(), False)


def _pack(st, w, trans, pack_dtype):
    """A constant weight packed once from device memory."""
    import ctypes

    s, h = _sess(), ctypes.c_void_p()
    L.check(s.lib.ingot_rocm_weight_pack_device(s.h, DT[w.dtype], pack_dtype, w.shape[0], w.shape[1], w.shape[1],
                                                1 if trans else 0, w.data_ptr(), ctypes.byref(h)))
    st.weights.append(Weight(s, h.value))
    return st.weights[-1]


def _buffer(st, shape, dtype=torch.float32):
    st.out.append(torch.empty(shape, dtype=dtype, device="cuda"))
    return _dev(st.out[-1])


def _out_side(size, ks, stride):
    return (size + 2 * (ks // 2) - ks) // stride + 1


def prepare(case, seed):
    s, st = _sess(), _State()
    t = st.t = _inputs(case, seed)
    torch.cuda.synchronize()  # the library's stream is its own
    kind = case["kind"]
    if kind == "gemm":
        w = _pack(st, t["w"], True, DT[t["w"].dtype])
        y = _buffer(st, (case["m"], case["n"]))
        st.calls.append(s.prepare_gemm(_dev(t["a"]), w, y, case["m"], trans_a=case["trans_a"], beta=1.0,
                                       c=_dev(t["bias"]), c_mode=L.C_ROW, act=ACT[case["act"]],
                                       math=L.MATH_BF16 if case["math"] == "bf16" else L.MATH_AUTO))
    elif kind == "ffn":
        g = Graph(s, "\n".join((
            "input x f32 %d,%d" % (case["m"], case["hidden"]),
            "const W1 f32 %d,%d" % (case["hidden"], case["inner"]), "const b1 f32 %d" % case["inner"],
            "const W2 f32 %d,%d" % (case["inner"], case["hidden"]), "const b2 f32 %d" % case["hidden"],
            "node MatMul x,W1 -> h1", "node Add h1,b1 -> h2", "node ingot.Gelu h2 -> h3", "node MatMul h3,W2 -> h4",
            "node Add h4,b2 -> y", "output y")) + "\n")
        for name in ("W1", "b1", "W2", "b2"):
            g.bind(name, _dev(t[name]))
        g.compile(L.GRAPH_FUSE_BIAS | L.GRAPH_FUSE_ACT | (L.GRAPH_HALF if case["half"] else 0))
        st.closers.append(g)
        x = _dev(t["x"])
        st.calls.append(lambda: g.run({"x": x}))
    elif kind == "attention":
        z, sq, sk, d = case["items"], case["sq"], case["sk"], case["d"]
        q, k, p, v = (_dev(t[n]) for n in "qkpv")
        scores, mixed = _buffer(st, (z, sq, sk)), _buffer(st, (z, sq, d))
        st.calls.append(lambda: s.gemm_dynamic_b(q, k, scores, sq, sk, d, True, d, sk * d, alpha=1.0 / math.sqrt(d),
                                                 batch=z, stride_a=sq * d, stride_y=sq * sk))
        st.calls.append(lambda: s.gemm_dynamic_b(p, v, mixed, sq, d, sk, False, d, sk * d, batch=z, stride_a=sq * sk,
                                                 stride_y=sq * d))
    elif kind == "int8":
        w = _pack(st, t["w"], False, L.DT_I8)
        m, n = case["m"], case["n"]
        a, za = _dev(t["a"]), (128 if case["a"] == "u8" else 3)
        if case["out"] == "u8":
            y = _buffer(st, (m, n), torch.uint8)
            mult = _requant_mult(case)
            st.calls.append(lambda: s.qlinear_matmul(a, w, m, za, mult, 120, y))
        elif case["out"] == "i32":
            st.calls.append(s.prepare_matmul_integer(a, w, m, za, y_i32=_buffer(st, (m, n), torch.int32)))
        else:
            st.calls.append(s.prepare_matmul_integer(a, w, m, za, scale=_dev(t["scale"]), y_f32=_buffer(st, (m, n))))
    elif kind == "qconv":
        ks, stride, pad = case["ks"], case["stride"], case["ks"] // 2
        w = _pack(st, t["w"].view(case["m"], -1), True, L.DT_I8)
        y = _buffer(st, (case["n"], case["m"], _out_side(case["h"], ks, stride), _out_side(case["w"], ks, stride)),
                    torch.uint8)
        x, mult, bias = _dev(t["x"]), _dev(t["mult"]), _dev(t["bias"])
        wshape = tuple(t["w"].shape)
        st.calls.append(lambda: s.qlinear_conv(x, 120, w, wshape, mult, 128, y, bias=bias, group=case["group"],
                                               strides=(stride, stride), pads=(pad, pad, pad, pad)))
    elif kind == "decoder":
        for i, (k, n) in enumerate(_decoder(case)):
            w = _pack(st, t["w%d" % i], True, L.PACK_I8G if case["weight"] == "int8" else L.DT_BF16)
            st.calls.append(s.prepare_gemm(_dev(t["x%d" % i]), w, _buffer(st, (case["m"], n)), case["m"],
                                           math=L.MATH_BF16 if case["math"] == "bf16" else L.MATH_AUTO))
    elif kind == "dit":
        m = case["m"]
        w = [_pack(st, t["w%d" % i], True, L.DT_BF16) for i in range(3)]
        qkv = _buffer(st, (m, case["qkv"]))
        hid = _buffer(st, (m, case["inner"]), torch.bfloat16)
        y = _buffer(st, (m, case["hidden"]))
        st.calls.append(s.prepare_gemm(_dev(t["x0"]), w[0], qkv, m, math=L.MATH_BF16))
        st.calls.append(s.prepare_gemm(_dev(t["x1"]), w[1], hid, m, math=L.MATH_BF16, act=L.ACT_GELU_ERF))
        st.calls.append(s.prepare_gemm(hid, w[2], y, m))
    else:
        dq = s.op("DequantizeLinear", 10, {"axis": max(0, case["axis"])})
        gelu = s.op("Gelu", 20)
        st.closers += [dq, gelu]
        x, scale = _dev(t["x"]), _dev(t["scale"])
        zp = _dev(t["zp"]) if "zp" in t else None

        def both():
            (f,) = dq.run(x, scale, zp) if zp is not None else dq.run(x, scale)
            (y,) = gelu.run(f)
            return [f, y]

        st.calls.append(both)
    s.sync()
    return st


def run(st):
    if st.out:
        for call in st.calls:
            call()
        return st.out
    st.release()
    for call in st.calls:
        st.results += call()
    return [torch.as_tensor(_Pooled(r), device="cuda") for r in st.results]


# ---- what a pass cannot do without, and how close results have to be ----

def _requant_mult(case):
    return 48.0 / (74.0 * 74.0 * math.sqrt(case["k"]))


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 4 * m * k + (4 if case["weight"] == "f32" else 2) * n * k + 4 * n + 4 * m * n, "flops": 2.0 * m * k * n}
    if kind == "ffn":
        m, h, i = case["m"], case["hidden"], case["inner"]
        wb, hb = (2, 2) if case["half"] else (4, 4)
        return {"bytes": 8 * m * h + 2 * wb * h * i + 2 * hb * m * i + 4 * (h + i), "flops": 4.0 * m * h * i}
    if kind == "attention":
        z, sq, sk, d = case["items"], case["sq"], case["sk"], case["d"]
        e = 4 if case["dtype"] == "f32" else 2
        return {"bytes": z * (e * (sq * d + 2 * sk * d + sq * sk) + 4 * (sq * sk + sq * d)), "flops": 4.0 * z * sq * sk * d}
    if kind == "int8":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": m * k + k * n + (1 if case["out"] == "u8" else 4) * m * n + 4 * n, "flops": 2.0 * m * k * n}
    if kind == "qconv":
        oh, ow = (_out_side(case[a], case["ks"], case["stride"]) for a in "hw")
        taps = case["c"] // case["group"] * case["ks"] ** 2
        y = case["n"] * case["m"] * oh * ow
        return {"bytes": case["n"] * case["c"] * case["h"] * case["w"] + case["m"] * (taps + 8) + y, "flops": 2.0 * y * taps}
    if kind == "decoder":
        per = 2.0 if case["weight"] == "bf16" else 1.0 + 4.0 / 64
        return {"bytes": sum(per * k * n + 4 * case["m"] * (k + n) for k, n in _decoder(case)),
                "flops": sum(2.0 * case["m"] * k * n for k, n in _decoder(case))}
    if kind == "dit":
        m, h, q, i = case["m"], case["hidden"], case["qkv"], case["inner"]
        return {"bytes": 8 * m * h + 2 * (h * q + 2 * h * i) + 4 * m * q + 4 * m * i + 4 * m * h, "flops": 2.0 * m * h * (q + 2 * i)}
    n = case["rows"] * case["cols"]
    return {"bytes": n * (4 if case["x"] == "i32" else 1) + 12 * n, "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind in ("int8", "qconv"):
        return "exact"  # integer sums; one rounded multiply per result
    if kind == "nodes":
        return {"rel": 5e-7}
    if kind == "dit" or kind == "ffn" and case["half"]:
        return {"rel": 1e-2}  # a bf16 hidden activation, rounded once more
    if kind == "attention" and case["dtype"] == "bf16" or case.get("math") == "bf16":
        return {"rel": 1e-5}  # bf16 operands, f32 sums and results
    if kind == "decoder" or case.get("weight") == "bf16":
        return {"rel": 1e-5}  # f32 activations as two bf16 terms: 2.5e-6 from the 64-bit result
    return {"rel": 5e-6}  # f32 sums of up to 4096 products: up to 1.2e-6 from the 64-bit result


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    act = {"none": lambda v: v, "relu": torch.relu, "gelu": torch.nn.functional.gelu, "silu": torch.nn.functional.silu}
    if kind == "gemm":
        a = t["a"].double()
        return [act[case["act"]]((a.t() if case["trans_a"] else a) @ t["w"].double().t() + t["bias"].double())]
    if kind == "ffn":
        h = act["gelu"](t["x"].double() @ t["W1"].double() + t["b1"].double())
        return [h @ t["W2"].double() + t["b2"].double()]
    if kind == "attention":
        return [torch.bmm(t["q"].double(), t["k"].double().transpose(1, 2).contiguous()) / math.sqrt(case["d"]),
                torch.bmm(t["p"].double(), t["v"].double())]
    if kind == "int8":
        y = (t["a"].double() - (128 if case["a"] == "u8" else 3)) @ t["w"].double()
        if case["out"] == "f32":
            return [y * t["scale"].double()]
        return None  # whole numbers: compared as they are
    if kind == "qconv":
        return None
    if kind == "decoder":
        out = []
        for i in range(4):
            w = t["w%d" % i].double()
            if case["weight"] == "int8":  # the weights as packed: one scale per 64 of a row, whole steps
                g = t["w%d" % i].float().view(w.shape[0], -1, 64)
                scale = g.abs().amax(dim=2, keepdim=True)
                scale = scale / torch.full_like(scale, 127)  # a true quotient (torch multiplies by 1 / number)
                q = torch.clamp(torch.round(g / torch.where(scale == 0, torch.ones_like(scale), scale)), -127, 127)
                w = (q.double() * scale.double()).view(w.shape)
            out.append(t["x%d" % i].double() @ w.t())
        return out
    if kind == "dit":
        hid = act["gelu"](t["x1"].double() @ t["w1"].double().t())
        return [t["x0"].double() @ t["w0"].double().t(), hid, hid @ t["w2"].double().t()]
    x, axis = t["x"].double(), case["axis"]
    if "zp" in t:
        x = x - (t["zp"].double().view(-1, 1) if axis == 0 else t["zp"].double())
    f = x * (t["scale"].double().view(-1, 1) if axis == 0 else t["scale"].double())
    return [f, act["gelu"](f)]
