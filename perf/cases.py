"""The work a user of this framework has it do, as a list of measurable cases.

Every case is one call through the public entry points of `maxim_amd.hip`: a
whole MAXIM pass, one block of it, or one convolution, each as a plan handed
to an executor. `listed()` names fixed cases, `draw()` more of the same
ranges; `prepare` / `run` make and time one, `exact` is the same computation
in 64 bits as plain torch gives it, op by op.

Kinds of case:
  pass    a whole MAXIM forward pass over an [3][h][w] image (h and w multiples
          of 64, as the padding pipeline makes them), device image to device
          image (`Gpu.run_noalloc`) or, with host set, host array to host
          array (`Gpu.run`, the enhancement command's call)
  gmlp    one split-head multi-axis gMLP layer of the network (LayerNorm,
          Dense, GELU, block and grid gating, Dense, residual) at `c` channels
  rcab    one residual channel-attention block (LayerNorm, two 3x3
          convolutions, channel attention, residual) at `c` channels
  conv    one convolution: 3x3, 4x4 stride 2 or transposed 2x2 stride 2, of
          any height and width
All data is fp32, the only type the framework has. There is no backward.
"""

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "maxim-rs_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from maxim_amd import hip as H  # noqa: E402
from maxim_amd import plan as P  # noqa: E402

# MACs per pixel of the padded image, in millions, for choosing drawn sizes
_PASS_COST = {"S-1": 0.63, "S-2": 1.48, "S-3": 2.33, "M-1": 2.3, "M-2": 5.6}
_LARGEST = 2.33 * 1536 * 2048


def listed():
    return [
        # the smallest image the padding pipeline makes: every launch is tiny,
        # so launch count and latency are what a user waits for
        {"name": "pass_s1_64", "kind": "pass", "variant": "S-1", "h": 64, "w": 64, "host": False},
        # the two-stage model (the low-light enhancement checkpoint's) on a
        # 256x256 crop
        {"name": "pass_s2_256", "kind": "pass", "variant": "S-2", "h": 256, "w": 256, "host": False},
        # the three-stage model on a 600x400 photograph padded to 640x448: the
        # benchmark's configuration
        {"name": "pass_s3_640x448", "kind": "pass", "variant": "S-3", "h": 448, "w": 640, "host": False},
        # the wider model (64 to 512 channels) on a tall crop
        {"name": "pass_m1_256x320", "kind": "pass", "variant": "M-1", "h": 320, "w": 256, "host": False},
        # a three-megapixel photograph from host memory to host memory, the
        # enhancement command's call
        {"name": "pass_s3_2048x1536_host", "kind": "pass", "variant": "S-3", "h": 1536, "w": 2048, "host": True},
        # one gMLP layer at each resolution level: 16x16 blocks and grids over
        # 256x256, the ragged cells of 224x320, and the bottleneck's 8x8 over
        # 56x80 (64 windows of 70 pixels)
        {"name": "gmlp_c32_256", "kind": "gmlp", "c": 32, "h": 256, "w": 256},
        {"name": "gmlp_c64_224x320", "kind": "gmlp", "c": 64, "h": 224, "w": 320},
        {"name": "gmlp_c128_56x80", "kind": "gmlp", "c": 128, "h": 56, "w": 80},
        # the channel-attention block behind it, at full resolution
        {"name": "rcab_c32_448x640", "kind": "rcab", "c": 32, "h": 448, "w": 640},
        # single convolutions: an encoder 3x3, a ragged 3x3, the encoder's
        # downsampling
        {"name": "conv3_c64_256", "kind": "conv", "op": "3x3", "ci": 64, "co": 64, "h": 256, "w": 256},
        {"name": "conv3_c128_225x319", "kind": "conv", "op": "3x3", "ci": 128, "co": 128, "h": 225, "w": 319},
        {"name": "down_c32_64_512", "kind": "conv", "op": "4x4s2", "ci": 32, "co": 64, "h": 512, "w": 512},
    ]


def _log_size(rng, lo, hi, step=1):
    return max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step)


def draw(rng):
    kind = rng.choice(["pass", "pass", "gmlp", "gmlp", "rcab", "conv", "conv"])
    if kind == "pass":
        variant = rng.choice(["S-1", "S-2", "S-3", "M-1", "M-2"])
        host = rng.random() < 0.3
        # the device-to-device entry holds what the static scratch does (about
        # 640x448 in the S models, half of that in the wider ones)
        area = 448 * 640 if not host else _LARGEST / _PASS_COST[variant]
        if variant[0] == "M":
            area /= 3
        a = math.exp(rng.uniform(math.log(64 * 64), math.log(area)))
        shape = rng.uniform(0.6, 1.6)
        h = max(64, int(math.sqrt(a * shape) / 64) * 64)
        w = max(64, int(a / h / 64) * 64)
        if h == w == 64:  # listed; the next size up
            h = 128
        return {"kind": kind, "variant": variant, "h": h, "w": w, "host": host}
    if kind in ("gmlp", "rcab"):
        # the levels of one image: sides are multiples of 64 at c = 32, of 32
        # at c = 64, and at c = 128 of 16 (encoder) or 8 (bottleneck)
        c = rng.choice([32, 64, 128])
        step = {32: 64, 64: 32, 128: 8 if kind == "gmlp" else 16}[c]
        h = _log_size(rng, step, 14 * step, step)
        w = min(_log_size(rng, step, 14 * step, step), 70 * step * step // h // step * step)
        return {"kind": kind, "c": c, "h": h, "w": w}
    op = rng.choice(["3x3", "3x3", "4x4s2", "t2x2"])
    ci = rng.choice([3, 32, 64, 96, 128, 256])
    co = rng.choice([3, 32, 64, 128, 160])
    if op == "t2x2" and ci == 3:
        ci = 64
    return {"kind": kind, "op": op, "ci": ci, "co": co, "h": _log_size(rng, 17, 512), "w": _log_size(rng, 17, 512)}


# ------------------------------------------------------------------ plans

_weights = {}
_plans = {}


def _checkpoint(variant):
    """The model's parameters, the same for every image: seeded random-init
    (He-normal times 0.3, biases N(0, 0.02), LayerNorm scales N(1, 0.1), which
    keeps activations of order one through the network, as a trained
    checkpoint does)."""
    if variant not in _weights:
        _weights[variant] = P.Weights.synthetic(variant, seed=1, gain=0.3, bias_std=0.02, ln_std=0.1)
    return _weights[variant]


def _part(plan, x, y, first, last):
    """Ops [first, last) of a built plan as a plan of their own, from buffer x
    to buffer y, with the buffers and weights they touch."""
    ids, wids, views = {}, {}, {}

    def buf(b):
        if b < 0:
            return b
        if b not in ids:
            parent = plan.alias(b)
            if parent is not None:
                pid = buf(parent[0])
                ids[b] = len(ids)
                views[ids[b]] = (pid, parent[1])
            else:
                ids[b] = len(ids)
        return ids[b]

    def wt(i):
        return i if i < 0 else wids.setdefault(i, len(wids))

    ops = []
    buf(x)
    for i in range(first, last):
        o = P.Op.from_buffer_copy(plan.ops[i])
        o.dst, o.src, o.src2 = buf(o.dst), buf(o.src), buf(o.src2)
        o.w, o.wt, o.bias, o.scale = wt(o.w), -1, wt(o.bias), wt(o.scale)
        ops.append(o)
    bufs = [plan.bufs[b] for b in sorted(ids, key=ids.get)]
    return P.CustomPlan(bufs, ops, [plan.weight(i).copy() for i in sorted(wids, key=wids.get)], input=ids[x], output=ids[y],
                        views=views)


def _block(case):
    """The case's block out of the one-stage model: the first gMLP layer (of
    encoder level 0 or 1, or the bottleneck, whose windows are 8x8) or the
    first channel-attention block (of encoder level 0, 1 or 2)."""
    c, h, w = case["c"], case["h"], case["w"]
    level = {32: 0, 64: 1, 128: 3 if case["kind"] == "gmlp" else 2}[c]
    plan = P.Plan(_checkpoint("S-1"), h << level, w << level, named=True, deep=True)
    dumps = dict(plan.dumps)
    writer = {}
    for i, o in enumerate(plan.ops):
        writer.setdefault(o.dst, i)
    if case["kind"] == "rcab":
        name = "stage_0_encoder_block_%d_mid_g0_" % level
        x, y = dumps[name + "gmlp"], dumps[name + "rcab"]
        return _part(plan, x, y, writer[x] + 1, writer[y] + 1)
    name = "stage_0_%s_block_%d" % (("global", 0) if level == 3 else ("encoder", level))
    # the layer: LayerNorm, Dense, GELU, then the grid branch's permutation
    grid = writer[dumps[name + "/SplitHeadMultiAxisGmlpLayer_0/GridGmlpLayer_blocked"]]
    first = max(i for i in range(grid) if plan.ops[i].kind == P.CHAN_LN)
    x = plan.ops[first].src
    # through the residual add of the layer's input
    last = next(i for i in range(grid, len(plan.ops)) if plan.ops[i].kind == P.ADD and x in (plan.ops[i].src, plan.ops[i].src2))
    return _part(plan, x, plan.ops[last].dst, first, last + 1)


def _conv(case):
    ci, co, h, w = case["ci"], case["co"], case["h"], case["w"]
    g = np.random.default_rng(ci * 1000 + co)
    k = {"3x3": 3, "4x4s2": 4, "t2x2": 2}[case["op"]]
    shape = (ci, co, 2, 2) if case["op"] == "t2x2" else (co, ci, k, k)
    weight = (g.standard_normal(shape) * math.sqrt(2.0 / (k * k * ci))).astype(np.float32)
    bias = (0.1 * g.standard_normal(co)).astype(np.float32)
    kw = dict(dst=1, src=0, w=0, bias=1, c_in=ci, c_out=co, h=h, wd=w)
    if case["op"] == "3x3":
        oh, ow, op = h, w, P.make_op(P.CONV3X3, **kw)
    elif case["op"] == "4x4s2":
        oh, ow = (h + 1) // 2, (w + 1) // 2
        pads = [P.same_pad(h, 2, 4)[0], P.same_pad(w, 2, 4)[0]]
        op = P.make_op(P.CONV4X4S2, oh=oh, ow=ow, p=pads, **kw)
    else:
        oh, ow, op = 2 * h, 2 * w, P.make_op(P.CONVT2X2, **kw)
    return P.CustomPlan([(ci, h, w), (co, oh, ow)], [op], [weight, bias])


def _plan(case):
    key = tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "host")))
    if key not in _plans:
        if len(_plans) > 16:
            _plans.clear()
        if case["kind"] == "pass":
            _plans[key] = P.Plan(_checkpoint(case["variant"]), case["h"], case["w"])
        else:
            _plans[key] = _conv(case) if case["kind"] == "conv" else _block(case)
    return _plans[key]


def _input(case, seed):
    """An image for a pass (a smooth pattern plus noise, clipped to [0, 1], as
    photographs are), N(0, 1) activations for a block or a convolution."""
    c, h, w = _plan(case).shape
    g = np.random.default_rng(seed)
    if case["kind"] != "pass":
        return g.standard_normal((c, h, w), dtype=np.float32)
    y, x = np.arange(h)[:, None] / h, np.arange(w)[None, :] / w
    img = g.standard_normal((c, h, w), dtype=np.float32) * np.float32(0.1)
    for k in range(c):
        f, ph = g.uniform(0.5, 3.0, (3, 2)), g.uniform(0, 2 * np.pi, 3)
        img[k] += 0.5 + sum(0.1 * np.sin(2 * np.pi * (f[j, 0] * y + f[j, 1] * x) + ph[j]) for j in range(3))
    return np.clip(img, 0, 1)


# ------------------------------------------------------------------ a case

def prepare(case, seed):
    plan = _plan(case)
    image = _input(case, seed)
    state = {"plan": plan, "host": case.get("host", False)}
    if state["host"]:
        state["x"] = image
    else:
        state["x"] = torch.from_numpy(image).cuda()
        state["y"] = torch.zeros(plan.bufs[plan.output], dtype=torch.float32, device="cuda")
    state["gpu"] = H.Gpu(plan)
    try:
        # an optional kernel that the executor looked up and did not find may
        # have left the runtime's last error set; torch reports and clears it
        # at its next launch
        torch.zeros(1, device="cuda")
    except RuntimeError:
        pass
    return state


# The default stream's handle for a caller that has to name it (the entry takes
# 0 for "the executor's own stream", and passes of several executors, which
# share the entry's static scratch, must not overlap): hipStreamLegacy.
_DEFAULT_STREAM = 1


def run(state):
    if state["host"]:
        return state["gpu"].run(state["x"])
    stream = torch.cuda.current_stream().cuda_stream or _DEFAULT_STREAM
    state["gpu"].run_noalloc(state["x"].data_ptr(), state["y"].data_ptr(), stream)
    return state["y"]


def work(case):
    plan = _plan(case)
    flops = 0
    used = set()
    for o in plan.ops:
        if o.kind == P.CONV1X1:
            flops += 2 * o.c_in * o.c_out * o.h * o.wd
        elif o.kind == P.CONV3X3:
            flops += 18 * o.c_in * o.c_out * o.h * o.wd
        elif o.kind == P.CONV4X4S2:
            flops += 32 * o.c_in * o.c_out * o.oh * o.ow
        elif o.kind == P.CONVT2X2:
            flops += 8 * o.c_in * o.c_out * o.h * o.wd
        elif o.kind == P.GATE_MM:
            flops += 2 * o.c * o.p[0] * o.p[1] * (o.p[0] if o.mode == 0 else o.p[1])
        used.update(i for i in (o.w, o.bias, o.scale) if i >= 0)
    floats = plan.buf_len(plan.input) + plan.buf_len(plan.output) + sum(plan.weight(i).size for i in used)
    return {"bytes": 4 * floats, "flops": flops}


def tolerance(case):
    """About four times the error of fp32 sums against 64 bits, as measured:
    6e-8 to 9e-8 for a pass, 3e-8 to 4.3e-8 for a block (whose residual is
    most of its output), 1.8e-8 sqrt(K) for a convolution that sums K
    products (7e-9 to 1.1e-8 sqrt(K) where Winograd does)."""
    if case["kind"] == "pass":
        return {"rel": 4e-7}
    if case["kind"] != "conv":
        return {"rel": 2e-7}
    return {"rel": 8e-8 * math.sqrt(case["ci"] * {"3x3": 9, "4x4s2": 16, "t2x2": 1}[case["op"]])}


# ------------------------------------------------- the same in 64 bits

def _taps(n_in, n_out):
    """The antialiased bilinear resize of one axis as an [n_out][n_in] matrix."""
    scale = n_in / n_out
    k = max(scale, 1.0)
    at = (torch.arange(n_out, dtype=torch.float64) + 0.5) * scale - 0.5
    m = (1 - (at[:, None] - torch.arange(n_in, dtype=torch.float64)[None, :]).abs() / k).clamp(min=0)
    return (m / m.sum(1, keepdim=True)).cuda()


def _conv2d(x, w, stride, top, left, oh, ow):
    """Cross-correlation with zero padding, tap by tap."""
    co, ci, kh, kw = w.shape
    pad = torch.nn.functional.pad(x, (left, stride * ow + kw - x.shape[2] - left, top, stride * oh + kh - x.shape[1] - top))
    y = torch.zeros(co, oh * ow, dtype=torch.float64, device=x.device)
    for ky in range(kh):
        for kx in range(kw):
            t = pad[:, ky:ky + stride * oh:stride, kx:kx + stride * ow:stride]
            y += w[:, :, ky, kx].contiguous() @ t.reshape(ci, oh * ow)
    return y.view(co, oh, ow)


def _apply(o, x, x2, wt):
    """One op of the plan on float64 tensors; x is the flat source."""
    bias = wt(o.bias) if o.bias >= 0 else None
    if o.kind == P.COPY:
        return x
    if o.kind == P.ADD:
        return x + x2
    if o.kind == P.MUL:
        return x * x2
    if o.kind == P.GATE_APPLY:
        return x * (x2 + 1)
    if o.kind == P.GELU:
        return 0.5 * x * (1 + torch.erf(x / math.sqrt(2.0)))
    if o.kind == P.LRELU:
        return torch.where(x >= 0, x, o.slope * x)
    if o.kind == P.SIGMOID:
        return torch.sigmoid(x)
    if o.kind == P.CHAN_LN:
        v = x.view(o.c, o.hw)
        m = v.mean(0)
        var = ((v - m) ** 2).mean(0)
        return (v - m) / torch.sqrt(var + 1e-6) * wt(o.scale)[:, None] + bias[:, None]
    if o.kind == P.CHAN_MEAN:
        return x.view(o.c, o.hw).mean(1)
    if o.kind == P.CHAN_SCALE:
        return x.view(o.c, o.hw) * x2[:, None]
    if o.kind == P.GATE_MM:
        w, v = wt(o.w), x.view(o.c, o.p[0], o.p[1])
        if o.mode == 0:
            y = torch.stack([w.view(o.p[0], o.p[0]) @ v[c] for c in range(o.c)])
            return y if bias is None else y + bias[:, None]
        y = v.reshape(-1, o.p[1]) @ w.view(o.p[1], o.p[1]).t()
        return y if bias is None else y + bias
    if o.kind == P.BLOCK_PERM:
        gh, gw, fh, fw = o.p
        swap, forward = o.mode & P.PERM_SWAP, o.mode & P.PERM_FORWARD
        if forward:
            v = x.view(o.c, gh, fh, gw, fw)
            return v.permute(0, 2, 4, 1, 3) if swap else v.permute(0, 1, 3, 2, 4)
        if swap:
            return x.view(o.c, fh, fw, gh, gw).permute(0, 3, 1, 4, 2)
        return x.view(o.c, gh, gw, fh, fw).permute(0, 1, 3, 2, 4)
    if o.kind == P.RESIZE:
        v = x.view(o.c * o.h, o.wd) @ _taps(o.wd, o.ow).t()
        ty = _taps(o.h, o.oh)
        return torch.stack([ty @ p for p in v.view(o.c, o.h, o.ow)])
    if o.kind == P.DOWN_S:
        return x.view(o.c, o.h, o.wd)[:, o.p[1]::o.p[0], o.p[1]::o.p[0]][:, :o.oh, :o.ow]
    w = wt(o.w)
    if o.kind == P.CONV1X1:
        y = w.view(o.c_out, o.c_in) @ x.view(o.c_in, o.h * o.wd)
        return y if bias is None else y + bias[:, None]
    v = x.view(o.c_in, o.h, o.wd)
    if o.kind == P.CONV3X3:
        y = _conv2d(v, w.view(o.c_out, o.c_in, 3, 3), 1, 1, 1, o.h, o.wd)
    elif o.kind == P.CONV4X4S2:
        y = _conv2d(v, w.view(o.c_out, o.c_in, 4, 4), 2, o.p[0], o.p[1], o.oh, o.ow)
    else:  # transposed 2x2 stride 2
        t = w.view(o.c_in, o.c_out * 4).t().contiguous() @ v.reshape(o.c_in, -1)
        y = t.view(o.c_out, 2, 2, o.h, o.wd).permute(0, 3, 1, 4, 2).reshape(o.c_out, 2 * o.h, 2 * o.wd)
    return y if bias is None else y + bias[:, None, None]


def exact(case, seed):
    plan = _plan(case)
    image = torch.from_numpy(_input(case, seed)).double().cuda()

    def alias(b):
        if isinstance(plan, P.Plan):
            return plan.alias(b)
        d = plan.desc
        return (d.alias_parent[b], d.alias_delta[b]) if d.alias_parent and d.alias_parent[b] >= 0 else None

    def base(b):
        off = 0
        while alias(b) is not None:
            b, d = alias(b)
            off += d
        return b, off

    last = {}  # base buffer -> the last op that touches it
    for i, o in enumerate(plan.ops):
        for b in _operands(o):
            last[base(b)[0]] = i
    last[base(plan.output)[0]] = len(plan.ops)
    store = {}

    def flat(b):
        p, off = base(b)
        if p not in store:
            store[p] = torch.zeros(plan.buf_len(p), dtype=torch.float64, device="cuda")
        return store[p][off:off + plan.buf_len(b)]

    def wt(i):
        return torch.from_numpy(np.array(plan.weight(i))).double().cuda()

    flat(plan.input).copy_(image.reshape(-1))
    for i, o in enumerate(plan.ops):
        two = o.kind in (P.ADD, P.MUL, P.GATE_APPLY, P.CHAN_SCALE)
        y = _apply(o, flat(o.src), flat(o.src2) if two else None, wt)
        flat(o.dst).copy_(y.reshape(-1))
        for b in _operands(o):
            if last[base(b)[0]] == i:
                store.pop(base(b)[0], None)
    out = flat(plan.output).clone().view(plan.bufs[plan.output])
    return out.cpu().numpy() if case.get("host", False) else out


def _operands(o):
    """The buffers an op reads and writes (a resize's intermediate excluded)."""
    two = o.kind in (P.ADD, P.MUL, P.GATE_APPLY, P.CHAN_SCALE)
    return [o.dst, o.src, o.src2] if two else [o.dst, o.src]
