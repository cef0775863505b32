"""Performance cases: the calls that users of this provider make, over the range of sizes they make them at.

Every case goes through a public entry point (oxionnx_amd.ep.HipContext for single operators,
oxionnx_amd.session for whole graphs) with packed weights and output buffers held between calls, as a
serving loop holds them.  `listed` names twelve of them, `draw` gives more from the same ranges.
"""
import functools
import math

import numpy as np
import torch

from oxionnx_amd import _lib as L
from oxionnx_amd import workloads
from oxionnx_amd.ep import HipContext
from oxionnx_amd.session import Session

DTYPES = {"f32": (L.F32, torch.float32, 4), "f16": (L.F16, torch.float16, 2), "bf16": (L.BF16, torch.bfloat16, 2)}


def listed():
    return [
        # The smallest call: one AdaIN style projection of a face-swap generator (latent 512 -> 1024), f32.
        {"name": "gemm_style_f32", "kind": "gemm", "dtype": "f32", "m": 1, "k": 512, "n": 1024},
        # The embedding head of a face recogniser (25088 -> 512) on the few faces of one picture, f16.
        {"name": "gemm_head_f16", "kind": "gemm", "dtype": "f16", "m": 5, "k": 25088, "n": 512},
        # A classifier layer with sizes that are multiples of nothing, bf16.
        {"name": "gemm_ragged_bf16", "kind": "gemm", "dtype": "bf16", "m": 300, "k": 777, "n": 1001},
        # The largest projection: a 4096-token prefill through a 4096 -> 11008 MLP layer, f16.
        {"name": "gemm_mlp_f16", "kind": "gemm", "dtype": "f16", "m": 4096, "k": 4096, "n": 11008},
        # Attention scores of eight images through twelve heads of 64, 197 tokens each: both operands are
        # activations, so nothing is packed ahead.
        {"name": "matmul_scores_f16", "kind": "matmul", "dtype": "f16", "batch": 96, "m": 197, "k": 64, "n": 197},
        # One f32 convolution with a fused Relu at a detector's resolution, NCHW in and out.
        {"name": "conv_f32", "kind": "conv", "dtype": "f32", "b": 1, "c": 64, "h": 128, "w": 128, "cout": 64,
         "k": 3, "s": 1},
        # A residual stage's 3x3 convolution on a batch of eight, f16, NCHW as the ONNX node has it.
        {"name": "conv_batch_f16", "kind": "conv", "dtype": "f16", "b": 8, "c": 128, "h": 56, "w": 56, "cout": 128,
         "k": 3, "s": 1},
        # The depthwise 3x3 of a mobile network's block on a batch of four, f16, fused Relu6.
        {"name": "depthwise_f16", "kind": "depthwise", "dtype": "f16", "b": 4, "c": 256, "h": 56, "w": 56, "s": 1},
        # A decoder's learned 2x upsampling, ConvTranspose 4x4 stride 2, f16.
        {"name": "upconv_f16", "kind": "convt", "dtype": "f16", "b": 1, "c": 512, "h": 32, "w": 32, "cout": 256},
        # The INT8 feed-forward pair of a BERT-base layer on 4096 tokens, requantised between the two.
        {"name": "ffn_int8", "kind": "qffn", "m": 4096, "k": 768, "n": 3072},
        # The whole face-swap generator in f16: a captured forward replayed on a new frame, host to host.
        {"name": "face_swap_f16", "kind": "face_swap", "dtype": "f16", "blocks": 6},
        # The whole int8 detector backbone at 640 x 640: a captured forward replayed on a new frame.
        {"name": "yolo_int8", "kind": "yolo", "size": 640},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "matmul", "conv", "conv", "depthwise", "convt", "qffn", "qffn",
                       "face_swap", "yolo"])
    dtype = rng.choice(["f32", "f16", "bf16"])
    if kind == "gemm":
        # Rows from one latent to a long prefill; half of the feature counts round, half odd.
        most = 1.5e9 if dtype == "f32" else 4e10
        while True:
            m, k, n = _log_int(rng, 1, 4096), _log_int(rng, 64, 25088), _log_int(rng, 32, 11008)
            if rng.random() < 0.5:
                k, n = (k + 63) // 64 * 64, (n + 63) // 64 * 64
            if m * k * n <= most and k * n <= 5e7:
                return {"kind": kind, "dtype": dtype, "m": m, "k": k, "n": n}
    if kind == "matmul":
        while True:
            b, m, k, n = _log_int(rng, 1, 192), _log_int(rng, 16, 1024), _log_int(rng, 16, 512), _log_int(rng, 16, 1024)
            if b * m * k * n <= 4e9:
                return {"kind": kind, "dtype": dtype, "batch": b, "m": m, "k": k, "n": n}
    if kind == "conv":
        most = 1.5e9 if dtype == "f32" else 1e10
        while True:
            b, c, cout, h = _log_int(rng, 1, 8), _log_int(rng, 16, 512), _log_int(rng, 16, 512), _log_int(rng, 7, 160)
            if rng.random() < 0.5:
                c, cout = (c + 15) // 16 * 16, (cout + 15) // 16 * 16
            k, s = rng.choice([1, 3, 3, 5]), rng.choice([1, 1, 2])
            w = max(7, int(h * rng.uniform(0.75, 1.34)))
            if rng.random() < 0.5:
                h = w = max(8, h // 8 * 8)
            if b * c * cout * h * w * k * k / (s * s) <= most and b * max(c, cout) * h * w <= 3e7:
                return {"kind": kind, "dtype": dtype, "b": b, "c": c, "h": h, "w": w, "cout": cout, "k": k, "s": s}
    if kind == "depthwise":
        while True:
            b, c, h = _log_int(rng, 1, 16), _log_int(rng, 16, 1024), _log_int(rng, 7, 224)
            w = h if rng.random() < 0.5 else max(7, int(h * rng.uniform(0.75, 1.34)))
            if b * c * h * w <= 2e7:
                return {"kind": kind, "dtype": dtype, "b": b, "c": c, "h": h, "w": w, "s": rng.choice([1, 1, 2])}
    if kind == "convt":
        most = 1e9 if dtype == "f32" else 8e9
        while True:
            b, c, cout = _log_int(rng, 1, 4), _log_int(rng, 16, 512), _log_int(rng, 16, 256)
            h = _log_int(rng, 7, 96)
            w = h if rng.random() < 0.5 else max(7, int(h * rng.uniform(0.75, 1.34)))
            if b * c * cout * h * w * 16 <= most:
                return {"kind": kind, "dtype": dtype, "b": b, "c": c, "h": h, "w": w, "cout": cout}
    if kind == "qffn":
        k = 64 * rng.randint(2, 16)
        return {"kind": kind, "m": _log_int(rng, 1, 4096), "k": k, "n": rng.choice([2, 4]) * k}
    if kind == "face_swap":
        dtype = rng.choice(["f16", "f16", "f32"])
        return {"kind": kind, "dtype": dtype, "blocks": rng.randint(1, 6 if dtype == "f16" else 2)}
    return {"kind": kind, "size": 32 * rng.randint(4, 20)}


# ------------------------------------------------------------------ state
# One context per process and graph, as a program has: it holds the stream and the weight cache.
@functools.lru_cache(None)
def _ctx():
    return HipContext(0)


@functools.lru_cache(None)
def _model(kind, dtype, blocks):
    if kind == "face_swap":
        graph, _ = workloads.face_swap_generator(dtype=dtype, n_blocks=blocks)
    else:
        graph, _ = workloads.yolo_backbone_int8(size=64)   # the weights do not depend on the frame's size
    ctx = HipContext(0)
    return ctx, graph, Session(graph, ctx)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _uniform(g, shape, dtype):
    return (torch.rand(shape, generator=g, device="cuda") * 2 - 1).to(dtype)


def _normal(g, shape, std, dtype):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(dtype)


def _tensors(case, seed):
    """The operands of a case in its own data type, on the device."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "qffn":
        m, k, n = case["m"], case["k"], case["n"]
        t = {"a": torch.randint(0, 256, (m, k), generator=g, device="cuda", dtype=torch.int32).to(torch.uint8)}
        for i, (rows, cols) in enumerate(((k, n), (n, k)), 1):
            t["b%d" % i] = torch.randint(-127, 128, (rows, cols), generator=g, device="cuda",
                                         dtype=torch.int32).to(torch.int8)
            t["s%d" % i] = torch.rand(cols, generator=g, device="cuda") * 0.009 + 0.001
        return t
    dt = DTYPES[case["dtype"]][1]
    if kind == "gemm":
        m, k, n = case["m"], case["k"], case["n"]
        return {"a": _uniform(g, (m, k), dt), "b": _normal(g, (k, n), k ** -0.5, dt), "c": _normal(g, (n,), 0.1, dt)}
    if kind == "matmul":
        b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
        return {"a": _normal(g, (b, m, k), 1.0, dt), "b": _normal(g, (b, k, n), k ** -0.5, dt)}
    x = _uniform(g, (case["b"], case["c"], case["h"], case["w"]), dt)
    if kind == "conv":
        shape = (case["cout"], case["c"], case["k"], case["k"])
        std = (case["c"] * case["k"] ** 2) ** -0.5
    elif kind == "depthwise":
        shape, std = (case["c"], 1, 3, 3), 1 / 3
    else:
        shape, std = (case["c"], case["cout"], 4, 4), (case["c"] * 4) ** -0.5
    bias = case["c"] if kind == "depthwise" else case["cout"]
    return {"x": x, "w": _normal(g, shape, std, dt), "bias": _normal(g, (bias,), 0.1, dt)}


def _host(w):
    return w.float().cpu().numpy()


def _feeds(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] == "yolo":
        return {"x": rng.integers(0, 256, (1, 3, case["size"], case["size"])).astype(np.uint8)}
    dt = np.float16 if case["dtype"] == "f16" else np.float32
    return {"x": rng.uniform(0, 1, (1, 3, 128, 128)).astype(dt), "latent": rng.normal(0, 1, (1, 512)).astype(dt)}


def _out_hw(case):
    k = case.get("k", 3)
    return tuple((v + 2 * (k // 2) - k) // case["s"] + 1 for v in (case["h"], case["w"]))


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("face_swap", "yolo"):
        _, _, session = _model(kind, case.get("dtype"), case.get("blocks"))
        feeds = _feeds(case, seed)
        return {"kind": kind, "feeds": feeds, "forward": session.capture(feeds)}
    ctx, t = _ctx(), _tensors(case, seed)
    s = {"kind": kind, "ctx": ctx}
    if kind == "qffn":
        m, k, n = case["m"], case["k"], case["n"]
        for i in (1, 2):
            s["w%d" % i] = ctx.weight_qgemm(t["b%d" % i].cpu().numpy(), zp=0, scale=t["s%d" % i].cpu().numpy())
        s.update(a=t["a"], h=torch.empty((m, n), dtype=torch.uint8, device="cuda"),
                 y=torch.empty((m, k), dtype=torch.uint8, device="cuda"))
        return s
    ldt, dt, _ = DTYPES[case["dtype"]]
    if kind == "gemm":
        s.update(a=t["a"], w=ctx.weight_gemm(_host(t["b"]), dtype=ldt), c=t["c"],
                 y=torch.empty((case["m"], case["n"]), dtype=dt, device="cuda"))
    elif kind == "matmul":
        s.update(a=t["a"], b=t["b"], y=torch.empty((case["batch"], case["m"], case["n"]), dtype=dt, device="cuda"))
    else:
        if kind == "convt":
            s["w"] = ctx.weight_conv_transpose(_host(t["w"]), dtype=ldt, strides=(2, 2), pads=(1, 1, 1, 1))
            shape = (case["b"], case["cout"], 2 * case["h"], 2 * case["w"])
        else:
            s["w"] = ctx.weight_conv(_host(t["w"]), dtype=ldt)
            shape = (case["b"], case.get("cout", case["c"])) + _out_hw(case)
            p = case.get("k", 3) // 2
            s.update(stride=(case["s"],) * 2, pads=(p,) * 4)
        s.update(x=t["x"], bias=t["bias"], y=torch.empty(shape, dtype=dt, device="cuda"))
    return s


def run(s):
    kind = s["kind"]
    if kind in ("face_swap", "yolo"):
        return s["forward"].replay(s["feeds"])
    ctx = s["ctx"]
    if kind == "gemm":
        return ctx.gemm(s["a"], s["w"], s["c"], out=s["y"])
    if kind == "matmul":
        return ctx.matmul(s["a"], s["b"], out=s["y"])
    if kind == "conv":
        return ctx.conv2d(s["x"], s["w"], s["bias"], strides=s["stride"], pads=s["pads"], act=L.ACT_RELU, out=s["y"])
    if kind == "depthwise":
        return ctx.conv2d(s["x"], s["w"], s["bias"], strides=s["stride"], pads=s["pads"], act=L.ACT_CLIP, act_lo=0.0,
                          act_hi=6.0, group=s["x"].shape[1], out=s["y"])
    if kind == "convt":
        return ctx.conv_transpose2d(s["x"], s["w"], s["bias"], strides=(2, 2), pads=(1, 1, 1, 1), out=s["y"])
    h = ctx.qgemm(s["a"], s["w1"], a_zp=128, a_scale=0.02, y_scale=0.5, y_zp=128, out=s["h"])
    y = ctx.qgemm(h, s["w2"], a_zp=128, a_scale=0.5, y_scale=20.0, y_zp=128, out=s["y"])
    return {"h": h, "y": y}


# ------------------------------------------------------------------ work
def _face_swap_convs(blocks):
    """(cin, cout, kernel, output pixels) of every convolution of the generator."""
    return ([(3, 128, 7, 128 ** 2), (128, 256, 3, 64 ** 2), (256, 512, 3, 32 ** 2)] + [(512, 512, 3, 32 ** 2)] * 2 * blocks
            + [(512, 256, 3, 64 ** 2), (256, 128, 3, 128 ** 2), (128, 3, 7, 128 ** 2)])


def _yolo_convs(size):
    out = []

    def conv(cin, cout, k, px):
        out.append((cin, cout, k, px * px))

    def c2f(cin, cout, n, px):
        c = cout // 2
        conv(cin, 2 * c, 1, px)
        for _ in range(2 * n):
            conv(c, c, 3, px)
        conv((2 + n) * c, cout, 1, px)

    px = (size + 1) // 2
    conv(3, 16, 3, px)
    for cin, cout, n in ((16, 32, 1), (32, 64, 2), (64, 128, 2), (128, 256, 1)):
        px = (px + 1) // 2
        conv(cin, cout, 3, px)
        c2f(cout, cout, n, px)
    conv(256, 128, 1, px)
    conv(512, 256, 1, px)
    return out, px


def work(case):
    kind = case["kind"]
    if kind == "qffn":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": m * k * 2 + m * n + 2 * k * n + 4 * (k + n), "flops": 4.0 * m * k * n}
    if kind == "yolo":
        convs, px = _yolo_convs(case["size"])
        weights = sum(ci * co * k * k for ci, co, k, _ in convs)
        outs = 256 * px ** 2 + 128 * (2 * px) ** 2 + 64 * (4 * px) ** 2
        return {"bytes": 3 * case["size"] ** 2 + weights + outs,
                "flops": sum(2.0 * ci * co * k * k * p for ci, co, k, p in convs)}
    eb = DTYPES[case["dtype"]][2]
    if kind == "face_swap":
        convs, styles = _face_swap_convs(case["blocks"]), 2 * case["blocks"] * 512 * 1024
        weights = sum(ci * co * k * k for ci, co, k, _ in convs) + styles
        return {"bytes": eb * (weights + 9 * 128 ** 2 + 512),
                "flops": 2.0 * styles + sum(2.0 * ci * co * k * k * p for ci, co, k, p in convs)}
    if kind == "gemm":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": eb * (m * k + k * n + m * n + n), "flops": 2.0 * m * k * n}
    if kind == "matmul":
        b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
        return {"bytes": eb * b * (m * k + k * n + m * n), "flops": 2.0 * b * m * k * n}
    b, c, hw = case["b"], case["c"], case["h"] * case["w"]
    if kind == "convt":
        co = case["cout"]
        return {"bytes": eb * (b * c * hw + 16 * c * co + co + b * co * 4 * hw), "flops": 2.0 * b * c * co * 16 * hw}
    oh, ow = _out_hw(case)
    if kind == "depthwise":
        return {"bytes": eb * (b * c * (hw + oh * ow) + 10 * c), "flops": 18.0 * b * c * oh * ow}
    co, kk = case["cout"], case["k"] ** 2
    return {"bytes": eb * (b * c * hw + c * co * kk + co + b * co * oh * ow), "flops": 2.0 * b * c * co * kk * oh * ow}


def tolerance(case):
    kind = case["kind"]
    if kind in ("qffn", "yolo"):
        return "exact"   # int32 sums and one defined requantisation: the bytes have one right value
    # One sum in f32 and one rounding to the data type.
    one = {"f32": {"rel": 4e-6, "max": 4e-5}, "f16": {"rel": 8e-4, "max": 2e-3}, "bf16": {"rel": 7e-3, "max": 1.6e-2}}
    if kind == "face_swap":
        # Twelve instance norms renormalise each plane, so a change of the order of sums travels.
        return {"rel": 1.2e-2, "max": 0.12} if case["dtype"] == "f16" else {"rel": 1.6e-5, "max": 2e-4}
    return one[case["dtype"]]


# ------------------------------------------------------------------ exact
def _conv64(x, w, bias, stride, pad, mode="constant"):
    """Convolution in 64 bits, one product per tap."""
    x, w = x.double(), w.double()
    b, c, _, _ = x.shape
    co, _, kh, kw = w.shape
    x = torch.nn.functional.pad(x, (pad,) * 4, mode=mode)
    oh, ow = (x.shape[2] - kh) // stride + 1, (x.shape[3] - kw) // stride + 1
    y = bias.double().reshape(1, co, 1).expand(b, co, oh * ow).contiguous()
    for ky in range(kh):
        for kx in range(kw):
            v = x[:, :, ky:ky + stride * (oh - 1) + 1:stride, kx:kx + stride * (ow - 1) + 1:stride]
            y += w[:, :, ky, kx].contiguous() @ v.reshape(b, c, oh * ow)
    return y.reshape(b, co, oh, ow)


def _depthwise64(x, w, bias, stride):
    x, w = torch.nn.functional.pad(x.double(), (1,) * 4), w.double()
    oh, ow = (x.shape[2] - 3) // stride + 1, (x.shape[3] - 3) // stride + 1
    y = bias.double().reshape(1, -1, 1, 1)
    for ky in range(3):
        for kx in range(3):
            v = x[:, :, ky:ky + stride * (oh - 1) + 1:stride, kx:kx + stride * (ow - 1) + 1:stride]
            y = y + v * w[:, 0, ky, kx].reshape(1, -1, 1, 1)
    return y


def _upconv64(x, w, bias):
    b, c, h, wd = x.shape
    co = w.shape[1]
    x, w = x.double().reshape(b, c, h * wd), w.double()
    y = torch.zeros((b, co, 2 * h + 2, 2 * wd + 2), dtype=torch.float64, device=x.device)
    for ky in range(4):
        for kx in range(4):
            v = (w[:, :, ky, kx].t().contiguous() @ x).reshape(b, co, h, wd)
            y[:, :, ky:ky + 2 * h:2, kx:kx + 2 * wd:2] += v
    return y[:, :, 1:-1, 1:-1] + bias.double().reshape(1, co, 1, 1)


def _qgemm64(a, b, a_scale, b_scale, y_scale):
    combined = (torch.tensor(a_scale, dtype=torch.float32) * b_scale.cpu()) / torch.tensor(y_scale, dtype=torch.float32)
    acc = (a.double() - 128) @ b.double()
    return torch.clamp(torch.round(acc * combined.to(a.device).double() + 128), 0, 255)


def _face_swap64(case, seed):
    _, graph, _ = _model("face_swap", case["dtype"], case["blocks"])
    feeds = {k: torch.from_numpy(v).cuda().double() for k, v in _feeds(case, seed).items()}
    operands = {op: iter([[torch.from_numpy(np.asarray(graph.initializers[t])).cuda().double() for t in n.inputs[1:3]]
                          for n in graph.nodes if n.op == op]) for op in ("Conv", "Gemm")}

    def conv(x, stride=1, pad=1, mode="constant"):
        return _conv64(x, *next(operands["Conv"]), stride, pad, mode)

    def adain(x):
        w, b = next(operands["Gemm"])
        gamma, beta = (feeds["latent"] @ w + b).reshape(2, 1, -1, 1, 1)
        mean, var = x.mean((2, 3), keepdim=True), x.var((2, 3), unbiased=False, keepdim=True)
        return (x - mean) / torch.sqrt(var + 1e-5) * gamma + beta

    def up(x):
        return x.repeat_interleave(2, 2).repeat_interleave(2, 3)

    leaky = functools.partial(torch.nn.functional.leaky_relu, negative_slope=0.2)
    h = leaky(conv(feeds["x"], 1, 3, "reflect"))
    h = leaky(conv(h, 2))
    h = leaky(conv(h, 2))
    for _ in range(case["blocks"]):
        r = torch.relu(adain(conv(h, 1, 1, "reflect")))
        h = h + adain(conv(r, 1, 1, "reflect"))
    h = leaky(conv(up(h)))
    h = leaky(conv(up(h)))
    logits = conv(h, 1, 3, "reflect")
    return {"y": torch.tanh(logits), "logits": logits}


def exact(case, seed):
    kind = case["kind"]
    if kind == "yolo":
        return None   # fifty layers of bytes that 32-bit steps define
    if kind == "face_swap":
        return _face_swap64(case, seed)
    t = _tensors(case, seed)
    if kind == "qffn":
        h = _qgemm64(t["a"], t["b1"], 0.02, t["s1"], 0.5)
        return {"h": h, "y": _qgemm64(h, t["b2"], 0.5, t["s2"], 20.0)}
    if kind == "gemm":
        return t["a"].double() @ t["b"].double() + t["c"].double()
    if kind == "matmul":
        return t["a"].double() @ t["b"].double()
    if kind == "conv":
        return torch.relu(_conv64(t["x"], t["w"], t["bias"], case["s"], case["k"] // 2))
    if kind == "depthwise":
        return torch.clamp(_depthwise64(t["x"], t["w"], t["bias"], case["s"]), 0, 6)
    return _upconv64(t["x"], t["w"], t["bias"])
