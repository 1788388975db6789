"""The work that is timed: the calls a converted model, a calibration run or a
quantization-aware training step makes through ``torch.ops.quantized_ops`` and
the FakeQuantize modules, at the sizes of LLaMA-7B / BERT / ViT layers and over
the ranges around them.

Kinds of case (``case["kind"]``):

* ``linear``     one ``linear_mx``: the projection of a converted model, from a
                 decode step's single token to a prefill's 2048;
* ``attention``  one ``matmul_mx`` of prefill attention (Q K^T or P V), any
                 sequence length;
* ``decode``     the two ``matmul_mx`` of one decode step against the cache;
* ``quantize``   one ``quantize_mx``: an activation on its way into a product;
* ``outlier``    ``quantize_mx_outlier`` and the ``linear_mx`` that takes its
                 inliers and its CSR outliers;
* ``train``      forward and backward of a ``FusedAmaxObsFakeQuantize``;
* ``pack``       a weight to packed codes and back.
"""

import math

import torch

import __graft_entry__

vqx = __graft_entry__.load_package()
Q = torch.ops.quantized_ops
DEV = "cuda"

# The 16 levels of NormalFloat-4 (QLoRA), and the integer grid nf4_6 puts them on.
NF4 = [-1.0, -0.6961928, -0.52507305, -0.39491749, -0.28444138, -0.18477343, -0.09105004, 0.0, 0.0795803, 0.1609302,
       0.2461123, 0.33791524, 0.44070983, 0.562617, 0.72295684, 1.0]
NF4_6 = [-31., -22., -16., -12., -9., -6., -3., 0., 2., 5., 8., 10., 14., 17., 22., 31.]

# (in features, out features) of the linears: LLaMA-7B's projections and MLP,
# BERT-base / ViT-base, and a 1000-class head.
LINEARS = [(4096, 4096), (4096, 11008), (11008, 4096), (768, 768), (768, 3072), (3072, 768), (2048, 1000)]


def listed():
    return [
        # one token through the MLP's up projection, weights NF4, activations bf16
        dict(name="linear nf4 m1", kind="linear", fmt="nf4", m=1, k=4096, n=11008, bias=False),
        # the same layer in a 2048-token prefill
        dict(name="linear nf4 m2048", kind="linear", fmt="nf4", m=2048, k=4096, n=11008, bias=False),
        # a short prompt through the down projection, both operands NF4 codes
        dict(name="linear mxnf4 m333", kind="linear", fmt="mxnf4", m=333, k=11008, n=4096, bias=True),
        # an attention projection, both operands MXINT8
        dict(name="linear mxint8 m1000", kind="linear", fmt="mxint8", m=1000, k=4096, n=4096, bias=False),
        # prefill attention scores, full context
        dict(name="attention qk 2048", kind="attention", which="qk", coded=False, h=32, s=2048, d=128),
        # prefill attention output, a prompt of no particular length
        dict(name="attention pv 1333", kind="attention", which="pv", coded=True, h=32, s=1333, d=128),
        # one decode step of attention against a cache of 1999 tokens
        dict(name="decode 1999", kind="decode", coded=False, b=1, h=32, s=1999, d=128),
        # the activation of the down projection on its way into the product
        dict(name="quantize 2048x11008", kind="quantize", fmt="nf4_6", dtype="bf16", rows=2048, cols=11008, axis=-1,
             bs=64),
        # a projection whose activation has outliers, split off as CSR
        dict(name="outlier linear m512", kind="outlier", m=512, k=4096, n=4096),
        # calibration / training of an activation quantizer that keeps the top 1%
        dict(name="train outlier 2048x4096", kind="train", spec="nf4_6,qs=microscaling,bs=64,ax=-1,scale=fp8_e5m3,opct=0.01",
             dtype="bf16", rows=2048, cols=4096),
        # int8 quantization-aware training of a ViT layer's input, fp32
        dict(name="train int8 3152x768", kind="train", spec="int8,qs=per_tensor_symmetric", dtype="f32", rows=3152,
             cols=768),
        # a weight into packed NF4 for storage and back
        dict(name="pack nf4 4096x11008", kind="pack", fmt="nf4", rows=4096, cols=11008, bs=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "attention", "attention", "decode", "quantize", "quantize", "outlier",
                       "train", "train", "pack"])
    if kind == "linear":
        k, n = rng.choice(LINEARS)
        fmt = rng.choice(["nf4", "mxnf4", "mxint8"])
        return dict(kind=kind, fmt=fmt, m=_log(rng, 1, 2048), k=k, n=n, bias=rng.random() < 0.5)
    if kind == "attention":
        return dict(kind=kind, which=rng.choice(["qk", "pv"]), coded=rng.random() < 0.5, h=rng.choice([12, 16, 32]),
                    s=_log(rng, 64, 2048), d=rng.choice([64, 128]))
    if kind == "decode":
        return dict(kind=kind, coded=rng.random() < 0.5, b=rng.choice([1, 1, 2, 4]), h=rng.choice([12, 32]),
                    s=_log(rng, 64, 4096), d=rng.choice([64, 128]))
    if kind == "quantize":
        return dict(kind=kind, fmt=rng.choice(["nf4_6", "int6", "int8", "fp8_e4m3"]), dtype=rng.choice(["bf16", "bf16", "f32"]),
                    rows=_log(rng, 1, 2048), cols=rng.choice([768, 1000, 3072, 4096, 11008]), axis=rng.choice([-1, -1, -2]),
                    bs=rng.choice([16, 32, 64]))
    if kind == "outlier":
        return dict(kind=kind, m=_log(rng, 16, 2048), k=rng.choice([768, 4096]), n=rng.choice([768, 4096]))
    if kind == "train":
        spec = rng.choice(["nf4_6,qs=microscaling,bs=64,ax=-1,scale=fp8_e5m3,opct=0.01",
                           "int8,qs=microscaling,bs=32,ax=-1", "int8,qs=per_tensor_symmetric",
                           "fp8_e4m3,qs=per_tensor_symmetric", "int8,qs=per_channel_symmetric,ax=0"])
        return dict(kind=kind, spec=spec, dtype=rng.choice(["bf16", "f32"]), rows=_log(rng, 16, 4096),
                    cols=rng.choice([768, 1000, 3072, 4096]))
    return dict(kind=kind, fmt=rng.choice(["nf4", "int8", "fp8_e4m3", "fp6_e3m2"]), rows=_log(rng, 64, 4096),
                cols=rng.choice([768, 3072, 4096, 11008]), bs=rng.choice([32, 64]))


# -- inputs, plain torch ------------------------------------------------------
_TYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _ints(g, lo, hi, shape):
    return torch.randint(lo, hi, shape, generator=g, device=DEV).to(torch.bfloat16)


def _int8(g, shape):
    return (torch.randn(shape, generator=g, device=DEV) * 40).round_().clamp_(-127, 127).to(torch.bfloat16)


def _e5m3(g, shape, lo=-10, hi=1):
    """bf16 scales on the fp8_e5m3 grid."""
    e = torch.randint(lo, hi, shape, generator=g, device=DEV).float()
    return (torch.exp2(e) * (1 + torch.randint(0, 8, shape, generator=g, device=DEV).float() / 8)).to(torch.bfloat16)


def _pow2(g, shape, lo=-12, hi=-4):
    return torch.exp2(torch.randint(lo, hi, shape, generator=g, device=DEV).float()).to(torch.bfloat16)


def _code(levels):
    return torch.tensor(levels, dtype=torch.bfloat16, device=DEV)


def _activation(g, shape, dtype=torch.bfloat16, share=0.005, factor=32):
    x = torch.randn(shape, generator=g, device=DEV)
    return torch.where(torch.rand(shape, generator=g, device=DEV) < share, x * factor, x).to(dtype)


def _linear_inputs(c, seed):
    g, m, k, n = _gen(seed), c["m"], c["k"], c["n"]
    bias = torch.randn(n, generator=g, device=DEV).to(torch.bfloat16) if c["bias"] else None
    if c["fmt"] == "mxint8":
        bs = 16
        return dict(x=_int8(g, (m, k)), w=_int8(g, (n, k)), bias=bias, xs=_pow2(g, (m, k // bs)), ws=_pow2(g, (n, k // bs)),
                    bs=bs, xc=None, wc=None)
    w = _ints(g, 0, 16, (n, k))
    ws = _e5m3(g, (n, k // 64), -9, -4)
    if c["fmt"] == "nf4":
        return dict(x=torch.randn(m, k, generator=g, device=DEV).to(torch.bfloat16), w=w, bias=bias, xs=None, ws=ws, bs=64,
                    xc=None, wc=_code(NF4))
    return dict(x=_ints(g, 0, 16, (m, k)), w=w, bias=bias, xs=_e5m3(g, (m, k // 64), -6, -2), ws=ws, bs=64, xc=_code(NF4_6),
                wc=_code(NF4_6))


def _operand(g, shape, coded, kdim, lo=-32, hi=32):
    scale = list(shape)
    scale[kdim] = -(-scale[kdim] // 64)
    return _ints(g, 0 if coded else lo, 16 if coded else hi, shape), _e5m3(g, scale)


def _attention_inputs(c, seed):
    g, h, s, d = _gen(seed), c["h"], c["s"], c["d"]
    m, n, k = (s, s, d) if c["which"] == "qk" else (s, d, s)
    low = -32 if c["which"] == "qk" else 0  # probabilities are not negative
    a, sa = _operand(g, (1, h, m, k), c["coded"], -1, low)
    b, sb = _operand(g, (1, h, k, n), c["coded"], -2)
    return dict(a=a, sa=sa, b=b, sb=sb, code=_code(NF4_6) if c["coded"] else None)


def _decode_inputs(c, seed):
    g, b, h, s, d = _gen(seed), c["b"], c["h"], c["s"], c["d"]
    q, sq = _operand(g, (b, h, 1, d), c["coded"], -1)
    k, sk = _operand(g, (b, h, d, s), c["coded"], -2)
    p, sp = _operand(g, (b, h, 1, s), c["coded"], -1, 0)
    v, sv = _operand(g, (b, h, s, d), c["coded"], -2)
    return dict(q=q, sq=sq, k=k, sk=sk, p=p, sp=sp, v=v, sv=sv, code=_code(NF4_6) if c["coded"] else None)


def _outlier_inputs(c, seed):
    g, m, k, n = _gen(seed), c["m"], c["k"], c["n"]
    return dict(x=_activation(g, (m, k)), w=_int8(g, (n, k)), ws=_pow2(g, (n, k // 32)))


OUTLIER_THRESHOLD = 6.0


# -- the program --------------------------------------------------------------
def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear":
        return dict(_linear_inputs(c, seed), kind=kind)
    if kind == "attention":
        return dict(_attention_inputs(c, seed), kind=kind)
    if kind == "decode":
        return dict(_decode_inputs(c, seed), kind=kind)
    if kind == "outlier":
        return dict(_outlier_inputs(c, seed), kind=kind, qmap=vqx.get_quantization_map("int8", DEV))
    if kind == "quantize":
        qmap = vqx.get_quantization_map(c["fmt"], DEV)
        code, nf = None, c["fmt"].startswith("nf")
        if nf:  # a converted graph keeps the indices as the table and the levels as the code
            qmap, code = qmap[0].to(torch.bfloat16), qmap[1]
        return dict(kind=kind, x=_activation(_gen(seed), (c["rows"], c["cols"]), _TYPES[c["dtype"]]), qmap=qmap, code=code,
                    qmax={"nf4_6": 31.0, "int6": 31.0, "int8": 127.0, "fp8_e4m3": 448.0}[c["fmt"]], axis=c["axis"],
                    bs=c["bs"], pow2=c["fmt"] in ("int8", "fp8_e4m3"),
                    smap=vqx.get_quantization_map("fp8_e5m3", DEV) if c["fmt"] in ("nf4_6", "int6") else None)
    if kind == "train":
        g, dt = _gen(seed), _TYPES[c["dtype"]]
        x = _activation(g, (c["rows"], c["cols"]), dt, 0.01, 20).requires_grad_()
        fq = vqx.quantization.QuantizationSpec.from_str(c["spec"]).make_fake_quantize(DEV).to(DEV)
        return dict(kind=kind, x=x, g=torch.randn(c["rows"], c["cols"], generator=g, device=DEV).to(dt), fq=fq)
    g = _gen(seed)
    return dict(kind=kind, x=(0.02 * torch.randn(c["rows"], c["cols"], generator=g, device=DEV)).to(torch.bfloat16),
                fmt=c["fmt"], bs=c["bs"], pow2=c["fmt"] != "nf4")


def run(s):
    kind = s["kind"]
    if kind == "linear":
        return Q.linear_mx(s["x"], s["w"], s["bias"], input_scale=s["xs"], weight_scale=s["ws"], block_size=s["bs"],
                           input_code=s["xc"], weight_code=s["wc"])
    if kind == "attention":
        return Q.matmul_mx(s["a"], s["b"], input_scale=s["sa"], weight_scale=s["sb"], block_size=64, input_code=s["code"],
                           weight_code=s["code"])
    if kind == "decode":
        qk = Q.matmul_mx(s["q"], s["k"], input_scale=s["sq"], weight_scale=s["sk"], block_size=64, input_code=s["code"],
                         weight_code=s["code"])
        pv = Q.matmul_mx(s["p"], s["v"], input_scale=s["sp"], weight_scale=s["sv"], block_size=64, input_code=s["code"],
                         weight_code=s["code"])
        return qk, pv
    if kind == "quantize":
        return Q.quantize_mx(s["x"], s["qmap"], [s["axis"]], s["bs"], s["qmax"], s["pow2"], s["smap"], s["code"])
    if kind == "outlier":
        data, indices, indptr, scale, inliers = Q.quantize_mx_outlier(s["x"], s["qmap"], [-1], 32, 127.0, True, None, None,
                                                                      OUTLIER_THRESHOLD, 0.01)
        y = Q.linear_mx(inliers, s["w"], None, input_scale=scale, weight_scale=s["ws"], block_size=32, A_data=data,
                        A_indices=indices, A_indptr=indptr)
        return y, data, indices, indptr, scale, inliers
    if kind == "train":
        fq, x = s["fq"], s["x"]
        y = fq(x)
        grad, = torch.autograd.grad(y, x, s["g"])
        state = [fq.scale] if "microscaling" in str(fq.qscheme).lower() else [fq.scale, fq.amax_history]
        return [y, grad] + state + ([fq.outlier_threshold] if fq.outlier_pct is not None else [])
    scale, codes = Q.quantize_mx_packed(s["x"], s["fmt"], -1, s["bs"], s["pow2"], None, "e8m0" if s["pow2"] else "float32")
    return scale, codes, Q.dequantize_mx_packed(codes, scale, s["fmt"], s["bs"], list(s["x"].shape))


# -- what a pass cannot do without --------------------------------------------
def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        m, k, n = c["m"], c["k"], c["n"]
        weight = n * k + 2 * n * (k // 16) if c["fmt"] == "mxint8" else n * k // 2 + 2 * n * (k // 64)
        scales = {"nf4": 0, "mxnf4": 2 * m * (k // 64), "mxint8": 2 * m * (k // 16)}[c["fmt"]]
        return dict(bytes=2 * m * k + weight + scales + 2 * m * n, flops=2 * m * n * k)
    if kind == "attention":
        s, h, d = c["s"], c["h"], c["d"]
        m, n, k = (s, s, d) if c["which"] == "qk" else (s, d, s)
        nb = -(-k // 64)
        return dict(bytes=2 * h * (m * k + k * n + m * nb + nb * n + m * n), flops=2 * h * m * n * k)
    if kind == "decode":
        s, h, d = c["s"], c["b"] * c["h"], c["d"]
        one = s * d + s * d // 64 + 2 * s + 2 * d
        return dict(bytes=2 * 2 * h * one, flops=2 * 2 * h * s * d)
    if kind == "quantize":
        n, e = c["rows"] * c["cols"], 2 if c["dtype"] == "bf16" else 4
        return dict(bytes=2 * e * n + e * n // c["bs"], flops=3 * n)
    if kind == "outlier":
        m, k, n = c["m"], c["k"], c["n"]
        return dict(bytes=4 * m * k + m * k // 16 + m * k * 6 // 100 + n * k + n * k // 16 + 2 * m * n,
                    flops=2 * m * n * k + 2 * m * n * k // 200)
    n = c["rows"] * c["cols"]
    if kind == "train":
        e = 2 if c["dtype"] == "bf16" else 4
        return dict(bytes=2 * e * n + (e * n if "opct" in c["spec"] else 0), flops=4 * n)
    bits = {"nf4": 4, "int8": 8, "fp8_e4m3": 8, "fp6_e3m2": 6}[c["fmt"]]
    scale = n // c["bs"] * (4 if c["fmt"] == "nf4" else 1)
    return dict(bytes=2 * (2 * n + n * bits // 8 + scale), flops=4 * n)


def tolerance(case):
    # The products: the result's own rounding to bf16 is most of it (2^-9 /
    # sqrt(3) is 1.1e-3; measured 1.7e-3 against float64); an outlier linear
    # adds two bf16 results.  Everything else is table values, integers and
    # scales of a stated arithmetic, the same bits whatever the order.
    if case["kind"] in ("linear", "attention", "decode"):
        return {"rel": 7e-3}
    if case["kind"] == "outlier":
        return {"rel": 1e-2}
    return "exact"


# -- the products in float64 --------------------------------------------------
def _decoded(x, code, scale, bs, kdim):
    """bf16(code[x] * scale of the block), the operand the product is defined on, as float64."""
    v = x if code is None else code[x.to(torch.int64)]
    if scale is not None:
        e = scale.repeat_interleave(bs, kdim).narrow(kdim, 0, x.shape[kdim])
        v = (v.float() * e.float()).to(torch.bfloat16)
    return v.double()


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear":
        i = _linear_inputs(c, seed)
        y = _decoded(i["x"], i["xc"], i["xs"], i["bs"], -1) @ _decoded(i["w"], i["wc"], i["ws"], i["bs"], -1).t()
        return y if i["bias"] is None else y + i["bias"].double()
    if kind == "attention":
        i = _attention_inputs(c, seed)
        a, b = _decoded(i["a"], i["code"], i["sa"], 64, -1), _decoded(i["b"], i["code"], i["sb"], 64, -2)
        return torch.stack([a[0, h] @ b[0, h] for h in range(c["h"])])[None]
    if kind == "decode":
        i = _decode_inputs(c, seed)
        q, k = _decoded(i["q"], i["code"], i["sq"], 64, -1), _decoded(i["k"], i["code"], i["sk"], 64, -2)
        p, v = _decoded(i["p"], i["code"], i["sp"], 64, -1), _decoded(i["v"], i["code"], i["sv"], 64, -2)
        return (q.transpose(-2, -1) * k).sum(-2, keepdim=True), (p.transpose(-2, -1) * v).sum(-2, keepdim=True)
    if kind == "outlier":
        i = _outlier_inputs(c, seed)
        x = i["x"]
        out = x.abs() > OUTLIER_THRESHOLD
        inl = torch.where(out, torch.zeros_like(x), x)
        amax = inl.abs().reshape(c["m"], -1, 32).amax(-1)
        e = torch.floor(torch.log2(amax.double()).to(torch.bfloat16).double()) - 6
        scale = torch.where(amax > 0, torch.exp2(e), torch.ones_like(e))
        sx = scale.repeat_interleave(32, -1)
        inl = (inl.double() / sx).to(torch.bfloat16).double().round().clamp(-128, 127) * sx
        # the CSR holds the first entries in row-major order, up to its capacity
        keep = out.reshape(-1).cumsum(0).reshape(out.shape) <= int(c["m"] * c["k"] * 0.01)
        w = _decoded(i["w"], None, i["ws"], 32, -1)
        y = inl @ w.t() + torch.where(out & keep, x, torch.zeros_like(x)).double() @ w.t()
        return y, None, None, None, scale, None
    return None
