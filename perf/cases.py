"""The work whose speed counts: what a program built on this package has it do.

Kinds of cases (``case["kind"]``):

* ``linear``     -- one quantized linear layer, or several that read the same
                    x, on M rows of x (``QuantizedLinear``, ``qlinear_grouped``):
                    a token of a small model, a batch, a prompt.
* ``decode``     -- decoder layers of one decode step for a batch of
                    sequences, recorded in a HIP graph and replayed, as
                    ``GraphDecoder`` does for every token: norms, projections,
                    attention over the key/value cache, MLP, residuals.
* ``quantize``   -- ``quantize_tensor`` of one weight, ``quantize_tensors`` of
                    a layer's: loading a model.
* ``dequantize`` -- ``dequantize_tensor``: a weight back in fp16 (shapes the
                    fused kernels do not take, gradients, export).

Weights are N(0, 0.02) with 0.1 % outliers of 8 to 20 sigma, or Student-t(3)
with 1 %; activations N(0, 1) with four channels x30.  Shapes are those of the
OPT-1.3b, Llama-3-8B, Mistral-7B and Gemma-2B layers, and generic ones.
"""
import ctypes
import math

import torch

from atlasinfer_amd import _lib
from atlasinfer_amd.integration import atlas_wrappers as AW
from atlasinfer_amd.quant import adaptive_quantizer as AQ

# ---------------------------------------------------------------- the cases

# (N, K) lists separated by "+": the weights of one case, out x in
LLAMA_LAYER = "4096x4096+1024x4096+1024x4096+4096x4096+14336x4096+14336x4096+4096x14336"
SHAPES = [(2048, 2048), (8192, 2048), (2048, 8192),                   # OPT-1.3b
          (4096, 4096), (1024, 4096), (14336, 4096), (4096, 14336),   # Llama-3-8B, Mistral-7B
          (16384, 2048), (2048, 16384)]                               # Gemma-2B
MAX_LINEAR_FLOPS = 2 * 2048 * 28672 * 4096  # the largest listed linear case
MAX_QUANT_ELEMS = 218103808                 # the largest listed quantize case
PLANTED, TAIL = 0.001, 0.0022               # planted outliers; share of elements past the threshold in all


def listed():
    return [
        # one attention projection of a small model for one token, called by
        # itself: the smallest call, where the launch and the host count
        dict(name="linear-m1-opt", kind="linear", shapes="2048x2048", m=1, g=128, fmt="e4m3", bias=True, dist="normal"),
        # batch-1 decode of a 7-8 B model early in a conversation
        dict(name="decode-b1", kind="decode", arch="llama", layers=2, b=1, ctx=700, g=-1),
        # a serving batch with long histories, in the default block size
        dict(name="decode-b8-long", kind="decode", arch="llama", layers=2, b=8, ctx=4000, g=128),
        # a full serving batch
        dict(name="decode-b64", kind="decode", arch="llama", layers=2, b=64, ctx=500, g=-1),
        # a short prompt through an MLP layer in the original's int8 format
        dict(name="linear-m128-fc1-int8", kind="linear", shapes="8192x2048", m=128, g=128, fmt="int8", bias=True,
             dist="normal"),
        # a prompt of odd length through the longest rows
        dict(name="linear-m509-down", kind="linear", shapes="4096x14336", m=509, g=-1, fmt="e4m3", bias=False,
             dist="normal"),
        # a long prompt (or a batch of prompts) through gate and up together
        dict(name="linear-m2048-gateup", kind="linear", shapes="14336x4096+14336x4096", m=2048, g=-1, fmt="e4m3",
             bias=False, dist="normal"),
        # loading a model: a whole layer per output channel
        dict(name="quantize-layer", kind="quantize", shapes=LLAMA_LAYER, g=-1, fmt="e4m3", dist="normal"),
        # one weight in the default block size, heavy tails
        dict(name="quantize-gate-g128", kind="quantize", shapes="14336x4096", g=128, fmt="e4m3", dist="t3"),
        # a small model's weight in the original's int8 format
        dict(name="quantize-fc2-int8", kind="quantize", shapes="2048x8192", g=128, fmt="int8", dist="normal"),
        # a large weight back in fp16
        dict(name="dequantize-gate", kind="dequantize", shapes="14336x4096", g=128, fmt="e4m3", dist="normal"),
        # a small weight of the original's format back in fp16
        dict(name="dequantize-fc1-int8", kind="dequantize", shapes="8192x2048", g=128, fmt="int8", dist="normal"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _shapes(s):
    return [tuple(int(v) for v in p.split("x")) for p in s.split("+")]


def _block(rng, k, choices):
    """A block size for rows of k.  Per output channel, rows of 2049 to 4095
    are left out: the tiled codes of such weights were once written past
    their rows, so versions from before that was mended cannot be run there."""
    g = rng.choice(choices)
    return 128 if g == -1 and 2048 < k < 4096 else g


def _draw_linear(rng):
    count = rng.choice([1, 1, 1, 2, 3])
    if rng.random() < 0.5:
        n, k = rng.choice(SHAPES)
        ns = [n] * count
    else:
        k = 128 * _log_int(rng, 2, 128)
        ns = [16 * _log_int(rng, 16, 1024) for _ in range(count)]
    g = _block(rng, k, [-1, -1, 128, 128, 64, 256])
    if g > 0 and k % g:
        g = 128
    m = _log_int(rng, 1, 4096)
    m = max(1, min(m, MAX_LINEAR_FLOPS // (2 * k * sum(ns))))
    return dict(kind="linear", shapes="+".join(f"{n}x{k}" for n in ns), m=m, g=g,
                fmt=rng.choice(["e4m3", "e4m3", "e4m3", "int8"]), bias=rng.random() < 0.3,
                dist=rng.choice(["normal", "normal", "t3"]))


def _draw_decode(rng):
    b = 1 if rng.random() < 0.35 else _log_int(rng, 2, 64)
    ctx = _log_int(rng, 16, 8192)
    ctx = max(16, min(ctx, 32768 // b))
    return dict(kind="decode", arch=rng.choice(["llama", "llama", "opt"]), layers=rng.choice([1, 2]), b=b, ctx=ctx,
                g=rng.choice([-1, 128]))


def _draw_weights(rng, kind):
    while True:
        if rng.random() < 0.6:
            shapes = [rng.choice(SHAPES)]
            if kind == "quantize" and rng.random() < 0.3:
                shapes = shapes * rng.choice([2, 3])
        elif rng.random() < 0.6:
            shapes = [(16 * _log_int(rng, 2, 1024), 128 * _log_int(rng, 1, 128))]
        else:  # any size: rows that do not tile, blocks that cross rows
            shapes = [(_log_int(rng, 7, 8000), _log_int(rng, 31, 8000))]
        if sum(n * k for n, k in shapes) <= MAX_QUANT_ELEMS // 2:
            break
    return dict(kind=kind, shapes="+".join(f"{n}x{k}" for n, k in shapes),
                g=_block(rng, shapes[0][1], [-1, -1, 128, 128, 128, 32, 64, 256, 512, 1024]), fmt=rng.choice(["e4m3", "e4m3", "int8"]),
                dist=rng.choice(["normal", "normal", "t3"]))


def draw(rng):
    kind = rng.choice(["linear", "linear", "decode", "quantize", "dequantize"])
    if kind == "linear":
        return _draw_linear(rng)
    if kind == "decode":
        return _draw_decode(rng)
    return _draw_weights(rng, kind)


# ---------------------------------------------------------------- the inputs


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _weight(n, k, dist, gen):
    numel = n * k
    w = torch.randn(numel, generator=gen, device="cuda")
    frac = PLANTED
    if dist == "t3":
        chi = torch.randn(3, numel, generator=gen, device="cuda").square_().sum(0).div_(3.0).sqrt_()
        w.div_(chi)
        frac = 0.01
    w.mul_(0.02)
    c = max(1, round(frac * numel))
    pos = torch.randint(0, numel, (c,), generator=gen, device="cuda")
    # a position drawn twice keeps the larger magnitude, whatever order the
    # two are written in; its sign goes by the position
    val = (torch.rand(c, generator=gen, device="cuda") * 12 + 8) * 0.02
    hit = torch.zeros(numel, device="cuda").scatter_reduce_(0, pos, val, "amax")
    flip = torch.zeros(numel, device="cuda").scatter_(0, pos, (pos & 1).to(torch.float32))
    w = torch.where(hit > 0, hit * (1.0 - 2.0 * flip), w)
    return w.view(n, k).to(torch.float16)


def _stored_weights(case, seed):
    """Weights of a quantize or dequantize case: the seed deals out the
    blocks of the case's own weight and the places inside a block, so that
    every seed has the same number of outliers and its outputs the same
    shapes."""
    ws = []
    for i, (n, k) in enumerate(_shapes(case["shapes"])):
        w = _weight(n, k, case["dist"], _gen(7919 * (i + 1) + n + k)).view(-1)
        gen = _gen(seed + 31 * i)
        g = min(k if case["g"] == -1 else case["g"], w.numel())
        whole = w.numel() // g * g  # a last, partial block stays as it is
        order = torch.randperm(whole // g, generator=gen, device="cuda")
        inner = torch.randperm(g, generator=gen, device="cuda")
        ws.append(torch.cat([w[:whole].view(-1, g)[order][:, inner].reshape(-1), w[whole:]]).view(n, k))
    return ws


def _acts(m, k, gen):
    x = torch.randn(m, k, generator=gen, device="cuda")
    ch = torch.randperm(k, generator=gen, device="cuda")[:4]
    x[:, ch] *= 30
    return x.to(torch.float16)


def _bias(n, gen):
    return (torch.randn(n, generator=gen, device="cuda") * 0.1).to(torch.float16)


def _linear_inputs(case, seed):
    gen = _gen(seed)
    shapes = _shapes(case["shapes"])
    ws = [_weight(n, k, case["dist"], gen) for n, k in shapes]
    bs = [_bias(n, gen) if case["bias"] else None for n, _ in shapes]
    return ws, bs, _acts(case["m"], shapes[0][1], gen)


ARCH = {
    # hidden, heads, key/value heads, head size, MLP width
    "llama": dict(hidden=4096, h=32, hkv=8, d=128, ffn=14336),
    "opt": dict(hidden=2048, h=32, hkv=32, d=64, ffn=8192),
}
EPS = 1e-5


def _decode_names(arch):
    if arch == "opt":
        return ["q", "k", "v", "o", "fc1", "fc2"]
    return ["q", "k", "v", "o", "gate", "up", "down"]


def _decode_shape(arch, name):
    a = ARCH[arch]
    hid, kv, ffn = a["hidden"], a["hkv"] * a["d"], a["ffn"]
    return {"q": (hid, hid), "k": (kv, hid), "v": (kv, hid), "o": (hid, hid), "gate": (ffn, hid), "up": (ffn, hid),
            "down": (hid, ffn), "fc1": (ffn, hid), "fc2": (hid, ffn)}[name]


def _cache_len(case):
    return (case["ctx"] + 128 + 63) // 64 * 64  # room for the tokens to come


def _decode_inputs(case, seed):
    """Residual stream, weights, norms, biases and a cache filled up to ctx."""
    gen = _gen(seed)
    arch, a = case["arch"], ARCH[case["arch"]]
    b, ctx, length = case["b"], case["ctx"], _cache_len(case)

    def rnd(*shape, scale=1.0, at=0.0):
        return (torch.randn(*shape, generator=gen, device="cuda") * scale + at).to(torch.float16)

    x = rnd(b, a["hidden"], scale=0.5)
    layers = []
    for _ in range(case["layers"]):
        lay = {"w": {n: _weight(*_decode_shape(arch, n), "normal", gen) for n in _decode_names(arch)}}
        lay["norm1"], lay["norm2"] = rnd(a["hidden"], scale=0.1, at=1.0), rnd(a["hidden"], scale=0.1, at=1.0)
        if arch == "opt":
            lay["nb1"], lay["nb2"] = rnd(a["hidden"], scale=0.1), rnd(a["hidden"], scale=0.1)
            lay["bias"] = {n: rnd(_decode_shape(arch, n)[0], scale=0.1) for n in _decode_names(arch)}
        lay["kc"] = torch.zeros(b, a["hkv"], length, a["d"], dtype=torch.float16, device="cuda")
        lay["vc"] = torch.zeros_like(lay["kc"])
        lay["kc"][:, :, :ctx] = rnd(b, a["hkv"], ctx, a["d"])
        lay["vc"][:, :, :ctx] = rnd(b, a["hkv"], ctx, a["d"])
        layers.append(lay)
    inv = 1.0 / (1e6 ** (torch.arange(0, a["d"], 2, device="cuda", dtype=torch.float64) / a["d"]))
    ang = torch.arange(length, device="cuda", dtype=torch.float64)[:, None] * inv[None]
    ang = torch.cat([ang, ang], 1)
    return x, layers, ang.cos().to(torch.float16), ang.sin().to(torch.float16)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        ws, bs, x = _linear_inputs(case, seed)
        qts = AQ.quantize_tensors(ws, case["g"], code_format=case["fmt"])
        if len(qts) == 1:
            return dict(kind=kind, x=x, layer=AW.QuantizedLinear(qts[0], bs[0]))
        return dict(kind=kind, x=x, layer=None, qts=qts, biases=bs, codes=[AQ.kernel_codes(q, x.device) for q in qts],
                    tiles=[AQ.outlier_tiles(q, x.device) for q in qts])
    if kind == "decode":
        return _prepare_decode(case, seed)
    ws = _stored_weights(case, seed)
    if kind == "quantize":
        return dict(kind=kind, ws=ws, g=case["g"], fmt=case["fmt"])
    qts = [AQ.quantize_tensor(w, case["g"], code_format=case["fmt"]) for w in ws]
    return dict(kind=kind, qts=qts, device=ws[0].device)


# -------------------------------------------------- a decode step of layers


def _norm(x, w, b, n):
    y = torch.empty_like(x)
    L = _lib.load()
    _lib.check(L.aq_decode_norm(x.data_ptr(), None, w.data_ptr(), None if b is None else b.data_ptr(),
                                ctypes.c_float(EPS), x.shape[0], n, 0 if b is None else 1, y.data_ptr(),
                                _lib.stream_of(x.device)), "aq_decode_norm")
    return y


def _silu_mul(g, u):
    out = torch.empty_like(g)
    _lib.check(_lib.load().aq_silu_mul(g.data_ptr(), u.data_ptr(), out.data_ptr(), g.numel(),
                                       _lib.stream_of(g.device)), "aq_silu_mul")
    return out


def _attend(st, lay, q, k, v):
    a, b = st["arch_dims"], st["b"]
    o = torch.empty_like(q)
    opt = st["arch"] == "opt"
    scale = a["d"] ** -0.5
    _lib.check(_lib.load().aq_decode_attention(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), lay["kc"].data_ptr(), lay["vc"].data_ptr(), st["pos"].data_ptr(), b,
        a["h"], a["hkv"], a["d"], lay["kc"].shape[2], ctypes.c_float(1.0 if opt else scale),
        ctypes.c_float(scale if opt else 1.0), None if opt else st["cos"].data_ptr(),
        None if opt else st["sin"].data_ptr(), st["ws"].data_ptr(), st["ws"].numel(), o.data_ptr(),
        _lib.stream_of(q.device)), "aq_decode_attention")
    return o


def _step(st):
    """One decode step over the layers, in the launches GraphDecoder makes:
    at batch 1 the norms, activation and residuals inside the linears, at
    6..64 the activation and residuals, otherwise launches of their own."""
    b, hid, opt = st["b"], st["arch_dims"]["hidden"], st["arch"] == "opt"
    folded = b == 1 or b >= AW.LISTS_MIN_M
    x = st["x"]
    for lay in st["layers"]:

        def dec(names, inp, **kw):
            return AW.qlinear_decode(inp, [lay["q"][n] for n in names], [lay["bias"].get(n) for n in names],
                                     [lay["codes"][n] for n in names],
                                     tiles=[lay["tiles"][n] for n in names] if b > 1 else None, **kw)

        def grouped(names, inp):
            return AW.qlinear_grouped(inp, [lay["q"][n] for n in names], [lay["bias"].get(n) for n in names],
                                      [lay["codes"][n] for n in names])

        def normed(names, inp, w, nb, **kw):
            if b == 1:
                pro = AW.PRO_RMS if nb is None else AW.PRO_LAYERNORM
                return dec(names, inp, prologue=pro, norm_weight=w, norm_bias=nb, eps=EPS, **kw)
            h = _norm(inp, w, nb, hid)
            return dec(names, h, **kw) if folded else grouped(names, h)

        q, k, v = normed(["q", "k", "v"], x, lay["norm1"], lay.get("nb1"))
        o = _attend(st, lay, q, k, v)
        x1 = dec(["o"], o, residuals=[x])[0] if folded else x + grouped(["o"], o)[0]
        if opt:
            if folded:
                f = normed(["fc1"], x1, lay["norm2"], lay["nb2"], relu=[1])[0]
                x = dec(["fc2"], f, residuals=[x1])[0]
            else:
                f = torch.relu(normed(["fc1"], x1, lay["norm2"], lay["nb2"])[0])
                x = x1 + grouped(["fc2"], f)[0]
        elif b == 1:
            g, u = normed(["gate", "up"], x1, lay["norm2"], None)
            x = dec(["down"], g, prologue=AW.PRO_SWIGLU, x2=u, residuals=[x1])[0]
        elif folded:
            h = _norm(x1, lay["norm2"], None, hid)
            act = dec(["gate", "up"], h, swiglu_pair=True)[0]
            x = dec(["down"], act, residuals=[x1])[0]
        else:
            g, u = normed(["gate", "up"], x1, lay["norm2"], None)
            x = x1 + grouped(["down"], _silu_mul(g, u))[0]
    return x


def _prepare_decode(case, seed):
    x, layers, cos, sin = _decode_inputs(case, seed)
    arch, a, b = case["arch"], ARCH[case["arch"]], case["b"]
    dev = x.device
    out = []
    for lay in layers:
        names = _decode_names(arch)
        qts = dict(zip(names, AQ.quantize_tensors([lay["w"][n] for n in names], case["g"])))
        out.append(dict(q=qts, codes={n: AQ.kernel_codes(qts[n], dev) for n in names},
                        tiles={n: AQ.outlier_tiles(qts[n], dev) for n in names}, bias=lay.get("bias", {}),
                        **{n: lay[n] for n in ("norm1", "norm2", "nb1", "nb2", "kc", "vc") if n in lay}))
    nb = _lib.load().aq_decode_attention_workspace(b, a["h"], a["hkv"], a["d"], _cache_len(case))
    st = dict(kind="decode", arch=arch, arch_dims=a, b=b, x=x, layers=out, cos=cos, sin=sin,
              pos=torch.full((1,), case["ctx"], dtype=torch.long, device=dev),
              ws=torch.empty(max(nb, 16), dtype=torch.uint8, device=dev))
    side = torch.cuda.Stream(device=dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        _step(st)
    torch.cuda.current_stream(dev).wait_stream(side)
    st["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(st["graph"]):
        st["y"] = _step(st)
    return st


# ------------------------------------------------------------------ one pass


def _quantized(qt):
    return [qt.fp8_data.view(torch.uint8), qt.scale_factors, qt.fp16_outliers, qt.outlier_indices, qt.outlier_row_ptr,
            qt.outlier_cols, qt.outlier_tile_ptr, qt.outlier_tile_ent]


def run(state):
    kind = state["kind"]
    if kind == "linear":
        if state["layer"] is not None:
            return state["layer"](state["x"])
        return AW.qlinear_grouped(state["x"], state["qts"], state["biases"], state["codes"], state["tiles"])
    if kind == "decode":
        state["graph"].replay()
        return [state["y"]] + [t for lay in state["layers"] for t in (lay["kc"], lay["vc"])]
    if kind == "quantize":
        if len(state["ws"]) == 1:
            return [_quantized(AQ.quantize_tensor(state["ws"][0], state["g"], code_format=state["fmt"]))]
        return [_quantized(q) for q in AQ.quantize_tensors(state["ws"], state["g"], code_format=state["fmt"])]
    out = []
    for q in state["qts"]:
        out.append(AQ.dequantize_tensor(q, state["device"]))
        AQ.discard_dequantized(id(q))  # the caller keeps the tensor, not the package's cache
    return out


# -------------------------------------------------------- what it cannot avoid


def _code_bytes(n, k, g):
    g = k if g == -1 else g
    return n * k + 2 * n * k / g + 6 * TAIL * n * k + 4 * (n + 1)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m = case["m"]
        shapes = _shapes(case["shapes"])
        k = shapes[0][1]
        by = 2 * m * k + sum(_code_bytes(n, k, case["g"]) + 2 * m * n + (2 * n if case["bias"] else 0)
                             for n, _ in shapes)
        return {"bytes": by, "flops": 2.0 * m * sum(n * k for n, k in shapes)}
    if kind == "decode":
        arch, a, b, ctx = case["arch"], ARCH[case["arch"]], case["b"], case["ctx"]
        shapes = [_decode_shape(arch, n) for n in _decode_names(arch)]
        by = sum(_code_bytes(n, k, case["g"]) for n, k in shapes) + 4 * b * a["hkv"] * (ctx + 1) * a["d"]
        by += 4 * a["hidden"] + 4 * b * a["hidden"]
        fl = 2.0 * b * sum(n * k for n, k in shapes) + 4.0 * b * a["h"] * (ctx + 1) * a["d"]
        return {"bytes": case["layers"] * by, "flops": case["layers"] * fl}
    shapes = _shapes(case["shapes"])
    t3 = case["dist"] == "t3"
    by = 0.0
    for n, k in shapes:
        g = k if case["g"] == -1 else case["g"]
        # fp16 on one side; codes, scales and the outlier lists on the other
        by += 2 * n * k + n * k + 2 * n * k / g + (0.02 if t3 else TAIL) * n * k * 10
        if kind == "quantize":
            by += 4 * (n + 1)
    return {"bytes": by, "flops": 0.0}


def tolerance(case):
    kind = case["kind"]
    if kind == "linear":
        # fp16 outputs of f32 sums: about 2e-4 from rounding each output once,
        # at most an fp16 unit (2^-10 of the value) at one output
        return {"rel": 8e-4, "max": 4e-3}
    if kind == "decode":
        # fp16 activations rounded between the operations of up to two layers
        return {"rel": 6e-3, "max": 6e-2}
    return "exact"


# ------------------------------------------------------------ in 64 bits


def _plain_quantize(w, g, fmt, thr=3.0):
    """(codes' values, scales in fp16 and before rounding, outlier mask) per
    block of the zero-padded flat tensor, op by op: statistics in 64 bits
    rounded to fp16, the test and the quotients in fp16."""
    f = w.reshape(-1)
    g = w.shape[-1] if g == -1 else g
    nb = -(-f.numel() // g)
    x = torch.zeros(nb * g, dtype=torch.float16, device=f.device)
    x[:f.numel()] = f
    x = x.view(nb, g)
    xd = x.double()
    mean = xd.mean(1, keepdim=True)
    std = (xd - mean).square_().sum(1, keepdim=True).div_(max(g - 1, 1)).sqrt_()
    del xd
    m16, s16 = mean.float().half(), std.float().half()
    den = (s16.float() + 1e-6).half()
    out = ((x - m16) / den).abs() > thr
    amax = x.abs().masked_fill(out, 0.0).amax(1, keepdim=True)
    qmax = 127.0 if fmt == "int8" else 448.0
    exact_scale = amax.double() / qmax
    sc = (amax.float() / qmax).half()
    sc = torch.where(sc.float() < 1e-6, torch.full_like(sc, 1e-6), sc)
    none = out.all(1, keepdim=True)
    sc = torch.where(none, torch.ones_like(sc), sc)
    exact_scale = torch.where(none, torch.ones_like(exact_scale), exact_scale.clamp_min(1e-6))
    q = x / sc
    if fmt == "int8":
        c = q.float().round().clamp_(-127, 127)
    else:
        c = q.float().clamp_(-448, 448).to(torch.float8_e4m3fn).float()
    return x, c, sc, exact_scale, out


def _plain_dequantized(w, g, fmt):
    """The weight a quantized layer stands for, in 64 bits, in w's shape."""
    x, c, sc, _, out = _plain_quantize(w, g, fmt)
    d = torch.where(out, x, (c.half() * sc))
    return d.reshape(-1)[:w.numel()].view(w.shape).double()


def _exact_decode(case, seed):
    x16, layers, cos, sin = _decode_inputs(case, seed)
    arch, a = case["arch"], ARCH[case["arch"]]
    b, ctx, h, hkv, d = case["b"], case["ctx"], a["h"], a["hkv"], a["d"]
    x = x16.double()
    outs = []

    def rms(t, w):
        return t / (t.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()

    def ln(t, w, nb):
        return torch.nn.functional.layer_norm(t, (t.shape[-1],), w.double(), nb.double(), EPS)

    def rope(t):  # [b, heads, d] at position ctx
        c, s = cos[ctx].double(), sin[ctx].double()
        return t * c + torch.cat([-t[..., d // 2:], t[..., :d // 2]], -1) * s

    for lay in layers:
        def lin(name, t):
            y = t @ _plain_dequantized(lay["w"][name], case["g"], "e4m3").t()
            return y + lay["bias"][name].double() if "bias" in lay else y

        hcur = ln(x, lay["norm1"], lay["nb1"]) if arch == "opt" else rms(x, lay["norm1"])
        q, k, v = lin("q", hcur).view(b, h, d), lin("k", hcur).view(b, hkv, d), lin("v", hcur).view(b, hkv, d)
        if arch != "opt":
            q, k = rope(q), rope(k)
        kc, vc = lay["kc"].double(), lay["vc"].double()
        kc[:, :, ctx], vc[:, :, ctx] = k, v
        kk = kc[:, :, :ctx + 1].repeat_interleave(h // hkv, 1)
        s = (kk * (q * d ** -0.5).unsqueeze(2)).sum(-1)
        p = torch.softmax(s, -1)
        del kk
        vv = vc[:, :, :ctx + 1].repeat_interleave(h // hkv, 1)
        o = (vv * p.unsqueeze(-1)).sum(2).reshape(b, h * d)
        del vv
        x = x + lin("o", o)
        if arch == "opt":
            x = x + lin("fc2", torch.relu(lin("fc1", ln(x, lay["norm2"], lay["nb2"]))))
        else:
            hcur = rms(x, lay["norm2"])
            x = x + lin("down", torch.nn.functional.silu(lin("gate", hcur)) * lin("up", hcur))
        outs += [kc, vc]
    return [x] + outs


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        ws, bs, x = _linear_inputs(case, seed)
        ys = []
        for w, b in zip(ws, bs):
            y = x.double() @ _plain_dequantized(w, case["g"], case["fmt"]).t()
            ys.append(y + b.double() if b is not None else y)
        return ys[0] if len(ys) == 1 else ys
    if kind == "decode":
        return _exact_decode(case, seed)
    ws = _stored_weights(case, seed)
    if kind == "quantize":
        res = []
        for w in ws:
            x, _, _, scale, out = _plain_quantize(w, case["g"], case["fmt"])
            res.append([None, scale.reshape(-1), x[out].double(), None, None, None, None, None])
        return res
    return [_plain_dequantized(w, case["g"], case["fmt"]) for w in ws]
