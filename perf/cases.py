"""What a program does with this framework, as cases that can be timed and checked: single layers
through the C ABI of the kernel library (include/vkhip.h, heuristic plans), and blocks and a whole
network through vknn sessions created from an ONNX model (default options: timed plans).

A layer case is a call a C or C++ host makes per layer: NC4HW4 fp16 activations that already sit
on the GPU, a weight blob packed once, one entry point on the program's own stream. A session case
binds an fp32 NCHW input that sits on the GPU, runs the forward pass and hands the fp32 outputs to
work on the program's stream.
"""
import ctypes
import math
import os
import struct
import tempfile

import numpy as np
import torch

import vknn_amd as V

# ------------------------------------------------------------------------------------ cases
ACT = {"none": 0, "relu": 1, "relu6": 2, "hardswish": 4, "silu": 5}


def _conv(name, n, cin, h, w, cout, k, s, act, res=False):
    return dict(name=name, kind="conv", n=n, cin=cin, h=h, w=w, cout=cout, k=k, s=s, act=act, res=res)


def listed():
    return [
        # The last 1x1 expansion of ResNet-50 for one image, with its shortcut: a call of a few
        # microseconds, where latency and the spread over the chip count.
        _conv("pw_b1", 1, 512, 7, 7, 2048, 1, 1, "relu", True),
        # The 1x1 expansion of ResNet-50's third stage at batch 64, the most frequent layer shape there.
        _conv("pw_b64", 64, 256, 14, 14, 1024, 1, 1, "relu", True),
        # The 3x3 conv of the same stage: the ordinary compute-bound layer.
        _conv("c3_b64", 64, 256, 14, 14, 256, 3, 1, "relu"),
        # A detector's 3x3 stride-2 conv on an input that is no multiple of its stride (600 x 600
        # images): odd rows and columns, channels that fill no tile.
        _conv("c3s2_odd_b8", 8, 48, 75, 75, 108, 3, 2, "silu"),
        # MobileNetV3-Large's 5x5 depthwise layer with 672 channels at batch 128.
        dict(name="dw5_b128", kind="dwconv", n=128, c=672, h=14, w=14, k=5, s=1, act="hardswish"),
        # The depthwise conv and linear projection of MobileNetV2's block, with the shortcut, batch 32.
        dict(name="dwpw_b32", kind="dwpw", n=32, c=144, h=56, w=56, cout=24, k=3, s=1, act="relu6", res=True),
        # A squeeze-excite called op by op: pool, the two FCs with their gate, the channel scale.
        dict(name="se_b128", kind="se", n=128, c=672, h=14, w=14, cr=168),
        # The way in and out of a detector: 16 fp32 images into the activation layout, and one of
        # its feature maps back to fp32.
        dict(name="boundary_b16", kind="boundary", n=16, hw=640, c=64),
        # A MobileNetV3-Large block as a model of its own: 1x1 expansion, 3x3 depthwise,
        # squeeze-excite, projection and shortcut, batch 128.
        dict(name="mnv3_block_b128", kind="mnv3_block", n=128, c=112, e=672, h=14, w=14, k=3),
        # A YOLOv8n C2f block with two bottlenecks at 80 x 80, batch 16.
        dict(name="c2f_b16", kind="c2f", n=16, c=64, h=80, w=80, reps=2),
        # ResNet-50 on one image (latency) and on 64 (throughput).
        dict(name="resnet50_b1", kind="resnet50", n=1, hw=224),
        dict(name="resnet50_b64", kind="resnet50", n=64, hw=224),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["conv", "conv", "conv", "conv", "dwconv", "dwconv", "dwpw", "se", "boundary", "mnv3_block", "c2f", "resnet50"])
    while True:
        if kind == "conv":
            # 1x1 and 3x3 layers of the networks above: batch 1 to 128, maps of 7 to 80 pixels
            k = rng.choice([1, 1, 3, 3])
            s = rng.choice([1, 1, 1, 2])
            c = dict(kind=kind, n=_log(rng, 1, 128), cin=_log(rng, 16, 2048 if k == 1 else 512), h=_log(rng, 7, 80), w=_log(rng, 7, 80),
                     cout=_log(rng, 16, 2048 if k == 1 else 512), k=k, s=s, act=rng.choice(["none", "relu", "relu6", "hardswish", "silu"]),
                     res=k == 1 and s == 1 and rng.random() < 0.4)
        elif kind == "dwconv":
            c = dict(kind=kind, n=_log(rng, 1, 128), c=_log(rng, 16, 960), h=_log(rng, 7, 112), w=_log(rng, 7, 112), k=rng.choice([3, 5]),
                     s=rng.choice([1, 1, 2]), act=rng.choice(["relu", "relu6", "hardswish"]))
        elif kind == "dwpw":
            c = dict(kind=kind, n=_log(rng, 1, 128), c=_log(rng, 32, 320), h=_log(rng, 14, 112), w=_log(rng, 14, 112), cout=_log(rng, 12, 64),
                     k=3, s=rng.choice([1, 1, 2]), act=rng.choice(["none", "relu", "relu6"]), res=False)
            c["res"] = c["s"] == 1 and rng.random() < 0.5
        elif kind == "se":
            c = dict(kind=kind, n=_log(rng, 1, 128), c=_log(rng, 24, 960), h=_log(rng, 7, 56), w=_log(rng, 7, 56))
            c["cr"] = max(8, (c["c"] // 4 + 7) // 8 * 8)
        elif kind == "boundary":
            c = dict(kind=kind, n=_log(rng, 1, 16), hw=rng.randint(160, 640), c=_log(rng, 16, 256))
        elif kind == "mnv3_block":
            ch = rng.choice([40, 80, 112, 160]) if rng.random() < 0.5 else rng.randint(24, 160)
            c = dict(kind=kind, n=_log(rng, 1, 128), c=ch, e=int(ch * rng.uniform(2.3, 6.0)), h=_log(rng, 7, 28), w=_log(rng, 7, 28), k=rng.choice([3, 5]))
        elif kind == "c2f":
            c = dict(kind=kind, n=_log(rng, 1, 16), c=rng.choice([32, 64, 128, 256]), h=rng.randint(20, 80), w=rng.randint(20, 80), reps=rng.choice([1, 2]))
        else:
            c = dict(kind=kind, n=_log(rng, 1, 64), hw=rng.randint(160, 224))
        wk = work(c)
        # no layer above the largest activations and products of the listed networks
        if kind == "resnet50" or (wk["bytes"] <= 400e6 and wk["flops"] <= 60e9):
            return c


# ------------------------------------------------------------------------------------ inputs
def _rng(seed, salt):
    return np.random.default_rng([seed & 0x7FFFFFFF, salt])


def _half(a):
    """Weights as an fp16 checkpoint holds them, in fp32."""
    return a.astype(np.float16).astype(np.float32)


def _normal(rng, shape, scale):
    a = rng.standard_normal(shape, dtype=np.float32)
    a *= np.float32(scale)
    return _half(a)


def _act_tensor(n, c, h, w, seed, salt, positive=False):
    """An activation tensor on the GPU, NCHW fp32 holding fp16 values: unit variance, or its positive part."""
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 131 + salt) & 0x7FFFFFFF)
    x = torch.randn((n, c, h, w), generator=g, device="cuda")
    return (x.clamp_(min=0) if positive else x).half().float()


def _nc4(x, dtype=torch.float16):
    """NCHW -> NC4HW4: [n, ceil(c/4), h, w, 4], missing channels zero."""
    n, c, h, w = x.shape
    cb = (c + 3) // 4
    y = torch.zeros((n, cb * 4, h, w), device=x.device, dtype=dtype)
    y[:, :c] = x
    return y.view(n, cb, 4, h, w).permute(0, 1, 3, 4, 2).contiguous()


_stream_of_program = []


def _stream():
    """The program's compute stream: every layer call goes to it and every session pass is ordered by it."""
    if not _stream_of_program:
        _stream_of_program.append(torch.cuda.Stream())
    return _stream_of_program[0]


def _check(rc, what):
    V.check(rc, what)


def _upload(host):
    return torch.from_numpy(host).cuda()


def _out_hw(c):
    p = c["k"] // 2
    return (c["h"] + 2 * p - c["k"]) // c["s"] + 1, (c["w"] + 2 * p - c["k"]) // c["s"] + 1


def _desc(c, cin, cout, group, act, res):
    oh, ow = _out_hw(c)
    p = c["k"] // 2
    return V.ConvDesc(N=c["n"], Cin=cin, H=c["h"], W=c["w"], Cout=cout, OH=oh, OW=ow, KH=c["k"], KW=c["k"], SH=c["s"], SW=c["s"], PT=p, PL=p,
                      DH=1, DW=1, group=group, act=ACT[act], act_lo=0.0, act_hi=6.0 if act == "relu6" else 0.0, has_res=int(res))


def _layer_inputs(c, seed):
    """Everything random of a layer case, as fp32 values that fp16 holds."""
    kind, n, h, w = c["kind"], c["n"], c["h"], c["w"]
    r = _rng(seed, 1)
    if kind == "conv":
        d = dict(x=_act_tensor(n, c["cin"], h, w, seed, 1, positive=True),
                 w=_normal(r, (c["cout"], c["cin"], c["k"], c["k"]), math.sqrt(2.0 / (c["cin"] * c["k"] ** 2))), b=_normal(r, (c["cout"],), 0.1))
        if c["res"]:
            d["res"] = _act_tensor(n, c["cout"], *_out_hw(c), seed, 2)
        return d
    if kind == "dwconv":
        return dict(x=_act_tensor(n, c["c"], h, w, seed, 1, positive=True), w=_normal(r, (c["c"], 1, c["k"], c["k"]), math.sqrt(2.0) / c["k"]),
                    b=_normal(r, (c["c"],), 0.1))
    if kind == "dwpw":
        d = dict(x=_act_tensor(n, c["c"], h, w, seed, 1, positive=True), w=_normal(r, (c["c"], 1, c["k"], c["k"]), math.sqrt(2.0) / c["k"]),
                 b=_normal(r, (c["c"],), 0.1), w2=_normal(r, (c["cout"], c["c"], 1, 1), math.sqrt(2.0 / c["c"])), b2=_normal(r, (c["cout"],), 0.1))
        if c["res"]:
            d["res"] = _act_tensor(n, c["cout"], *_out_hw(c), seed, 2)
        return d
    return dict(x=_act_tensor(n, c["c"], h, w, seed, 1, positive=True), w1=_normal(r, (c["cr"], c["c"]), math.sqrt(2.0 / c["c"])),
                b1=_normal(r, (c["cr"],), 0.1), w2=_normal(r, (c["c"], c["cr"]), math.sqrt(2.0 / c["cr"])), b2=_normal(r, (c["c"],), 0.1))


# ------------------------------------------------------------------------------------ models
class _Graph:
    """A network as a list of operators over named tensors: written as an ONNX model for a session
    and evaluated in float64 for reference values."""

    def __init__(self, shape, seed):
        self.ops, self.weights, self.shapes, self.outputs = [], {}, {"x": tuple(shape)}, []
        self.rng = _rng(seed, 7)

    def _emit(self, op, inputs, shape, outputs=1, **attrs):
        names = ["t%d_%d" % (len(self.ops), i) for i in range(outputs)]
        self.ops.append((op, list(inputs), names, attrs))
        for o in names:
            self.shapes[o] = tuple(shape)
        return names[0] if outputs == 1 else tuple(names)

    def weight(self, shape, scale):
        name = "w%d" % len(self.weights)
        self.weights[name] = _normal(self.rng, shape, scale)
        return name

    def conv(self, x, cout, k=1, s=1, group=1, gain=1.0):
        n, c, h, w = self.shapes[x]
        p = k // 2
        wt = self.weight((cout, c // group, k, k), gain * math.sqrt(2.0 / (c // group * k * k)))
        b = self.weight((cout,), 0.1)
        shape = (n, cout, (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1)
        return self._emit("Conv", [x, wt, b], shape, kernel_shape=[k, k], strides=[s, s], pads=[p] * 4, dilations=[1, 1], group=group)

    def unary(self, op, x, **attrs):
        return self._emit(op, [x], self.shapes[x], **attrs)

    def binary(self, op, a, b):
        return self._emit(op, [a, b], self.shapes[a])

    def silu(self, x):
        return self.binary("Mul", x, self.unary("Sigmoid", x))

    def hardswish(self, x):
        return self.binary("Mul", x, self.unary("HardSigmoid", x, alpha=1.0 / 6, beta=0.5))

    def maxpool(self, x, k, s, p):
        n, c, h, w = self.shapes[x]
        return self._emit("MaxPool", [x], (n, c, (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1), kernel_shape=[k, k], strides=[s, s], pads=[p] * 4)

    def pool(self, x):
        return self._emit("GlobalAveragePool", [x], self.shapes[x][:2] + (1, 1))

    def split2(self, x):
        n, c, h, w = self.shapes[x]
        return self._emit("Split", [x], (n, c // 2, h, w), outputs=2, axis=1, split=[c // 2, c // 2])

    def concat(self, xs):
        n, _, h, w = self.shapes[xs[0]]
        return self._emit("Concat", xs, (n, sum(self.shapes[t][1] for t in xs), h, w), axis=1)

    def head(self, x, classes):
        n, c = self.shapes[x][:2]
        flat = self._emit("Flatten", [x], (n, c), axis=1)
        return self._emit("Gemm", [flat, self.weight((classes, c), math.sqrt(1.0 / c)), self.weight((classes,), 0.1)], (n, classes), transB=1)

    # the ONNX file, field by field (protobuf wire format)
    def onnx(self):
        def varint(v):
            v &= (1 << 64) - 1
            out = bytearray()
            while v > 0x7F:
                out.append(v & 0x7F | 0x80)
                v >>= 7
            out.append(v)
            return bytes(out)

        def num(f, v):
            return varint(f << 3) + varint(v)

        def blob(f, b):
            b = b.encode() if isinstance(b, str) else b
            return varint(f << 3 | 2) + varint(len(b)) + b

        def attr(name, v):
            if isinstance(v, list):
                return blob(1, name) + blob(8, b"".join(varint(i) for i in v)) + num(20, 7)
            if isinstance(v, float):
                return blob(1, name) + varint(2 << 3 | 5) + struct.pack("<f", v) + num(20, 1)
            return blob(1, name) + num(3, v) + num(20, 2)

        def value(name):
            dims = b"".join(blob(1, num(1, d)) for d in self.shapes[name])
            return blob(1, name) + blob(2, blob(1, num(1, 1) + blob(2, dims)))

        g = [blob(1, b"".join(blob(1, i) for i in ins) + b"".join(blob(2, o) for o in outs) + blob(3, op + "_" + outs[0]) + blob(4, op) +
                  b"".join(blob(5, attr(k, a)) for k, a in sorted(attrs.items()))) for op, ins, outs, attrs in self.ops]
        g.append(blob(2, "g"))
        for name, a in self.weights.items():
            g.append(blob(5, blob(1, b"".join(varint(d) for d in a.shape)) + num(2, 1) + blob(8, name) + blob(9, a.tobytes())))
        g.append(blob(11, value("x")) + b"".join(blob(12, value(o)) for o in self.outputs))
        return num(1, 8) + blob(7, b"".join(g)) + blob(8, blob(1, "") + num(2, 11))

    def run64(self, x):
        """The outputs in float64."""
        t = {"x": x.double()}
        wt = {k: torch.from_numpy(v).cuda().double() for k, v in self.weights.items()}
        last = {}
        for i, (_, ins, _, _) in enumerate(self.ops):
            for name in ins:
                last[name] = i
        for i, (op, ins, outs, at) in enumerate(self.ops):
            a = t[ins[0]]
            if op == "Conv":
                y = _conv64(a, wt[ins[1]], wt[ins[2]], at["strides"][0], at["group"])
            elif op == "Relu":
                y = a.clamp(min=0)
            elif op == "Sigmoid":
                y = torch.sigmoid(a)
            elif op == "HardSigmoid":
                y = (a * at["alpha"] + at["beta"]).clamp(0, 1)
            elif op == "Mul":
                y = a * t[ins[1]]
            elif op == "Add":
                y = a + t[ins[1]]
            elif op == "MaxPool":
                y = _maxpool64(a, at["kernel_shape"][0], at["strides"][0], at["pads"][0])
            elif op == "GlobalAveragePool":
                y = a.mean((2, 3), keepdim=True)
            elif op == "Concat":
                y = torch.cat([t[k] for k in ins], 1)
            elif op == "Flatten":
                y = a.flatten(1)
            elif op == "Gemm":
                y = a @ wt[ins[1]].t() + wt[ins[2]]
            else:
                y = None
                t.update(zip(outs, a.chunk(2, 1)))  # Split
            if y is not None:
                t[outs[0]] = y
            for name in set(ins):
                if last.get(name) == i and name not in self.outputs:
                    t.pop(name, None)
        return [t[o] for o in self.outputs]


def _model(c, seed):
    if c["kind"] == "resnet50":
        g = _Graph((c["n"], 3, c["hw"], c["hw"]), seed)
        h = g.maxpool(g.unary("Relu", g.conv("x", 64, 7, 2)), 3, 2, 1)
        for stage, blocks in enumerate((3, 4, 6, 3)):
            mid = 64 << stage
            for i in range(blocks):
                s = 2 if i == 0 and stage else 1
                y = g.unary("Relu", g.conv(h, mid))
                y = g.unary("Relu", g.conv(y, mid, 3, s))
                y = g.conv(y, mid * 4, gain=0.2)
                h = g.unary("Relu", g.binary("Add", y, g.conv(h, mid * 4, 1, s) if i == 0 else h))
        g.outputs = [g.head(g.pool(h), 1000)]
    elif c["kind"] == "mnv3_block":
        g = _Graph((c["n"], c["c"], c["h"], c["w"]), seed)
        h = g.hardswish(g.conv("x", c["e"]))
        h = g.hardswish(g.conv(h, c["e"], c["k"], group=c["e"]))
        s = g.unary("Relu", g.conv(g.pool(h), max(8, (c["e"] // 4 + 7) // 8 * 8)))
        s = g.unary("HardSigmoid", g.conv(s, c["e"]), alpha=1.0 / 6, beta=0.5)
        g.outputs = [g.binary("Add", g.conv(g.binary("Mul", h, s), c["c"]), "x")]
    else:  # c2f
        g = _Graph((c["n"], c["c"], c["h"], c["w"]), seed)
        parts = list(g.split2(g.silu(g.conv("x", c["c"]))))
        for _ in range(c["reps"]):
            y = g.silu(g.conv(g.silu(g.conv(parts[-1], c["c"] // 2, 3)), c["c"] // 2, 3))
            parts.append(g.binary("Add", parts[-1], y))
        g.outputs = [g.silu(g.conv(g.concat(parts), c["c"]))]
    return g


def _model_input(c, seed):
    if c["kind"] == "resnet50":
        return _act_tensor(c["n"], 3, c["hw"], c["hw"], seed, 1)
    return _act_tensor(c["n"], c["c"], c["h"], c["w"], seed, 1)


class _DeviceView:
    """Device memory a session owns, as torch sees foreign arrays. A tensor made from it keeps this
    object, and so the session and its memory."""

    def __init__(self, session, ptr, shape):
        self.session = session
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<f4", data=(ptr, False), version=2, strides=None)


class _Model:
    def __init__(self, c, seed):
        g = _model(c, seed)
        shapes = [g.shapes[o] for o in g.outputs]
        with tempfile.TemporaryDirectory() as tmp:
            path = os.path.join(tmp, "model.onnx")
            with open(path, "wb") as f:
                f.write(g.onnx())
            self.session = V.Session.from_onnx(path, list(g.shapes["x"]), [int(np.prod(s)) for s in shapes])
        self.x = _model_input(c, seed)
        torch.cuda.synchronize()
        self.session.bind_device_input(self.x.data_ptr())
        self.session.run_device()  # the first pass records the launch sequence
        self.session.sync()
        self.stream = torch.cuda.ExternalStream(self.session.stream)
        self.outputs = [torch.as_tensor(_DeviceView(self.session, V.vknn().vknn_session_device_output(self.session.h, k), s), device="cuda")
                        for k, s in enumerate(shapes)]


# ------------------------------------------------------------------------------------ prepare, run
def prepare(case, seed):
    c, kind = case, case["kind"]
    stream = _stream()
    if kind in ("resnet50", "mnv3_block", "c2f"):
        return {"kind": kind, "model": _Model(c, seed), "stream": stream}
    lib = V.require_gpu()
    st = {"kind": kind, "case": c, "lib": lib, "stream": stream}
    if kind == "boundary":
        # images as a decoder leaves them: fp32 NCHW; and a feature map of the deepest usual stride-8 level
        st["image"] = _act_tensor(c["n"], 3, c["hw"], c["hw"], seed, 1)
        f = (c["n"], c["c"], c["hw"] // 8, c["hw"] // 8)
        st["features"] = _nc4(_act_tensor(*f, seed, 2))
        st["packed"] = torch.empty((c["n"], 1, c["hw"], c["hw"], 4), dtype=torch.float16, device="cuda")
        st["unpacked"] = torch.empty(f, device="cuda")
        torch.cuda.synchronize()
        return st
    d = _layer_inputs(c, seed)
    st["x"] = _nc4(d["x"])
    st["res"] = _nc4(d["res"]) if "res" in d else None
    oh, ow = (c["h"], c["w"]) if kind == "se" else _out_hw(c)
    cout = c["cout"] if kind in ("conv", "dwpw") else c["c"]
    st["y"] = torch.empty((c["n"], (cout + 3) // 4, oh, ow, 4), dtype=torch.float16, device="cuda")
    if kind == "conv" or kind == "dwconv":
        cd = _desc(c, c["cin"], c["cout"], 1, c["act"], c["res"]) if kind == "conv" else _desc(c, c["c"], c["c"], c["c"], c["act"], False)
        plan = V.ConvPlan()
        _check(lib.vkhip_conv_plan_make(ctypes.byref(cd), V.CONV_AUTO, -1, 0, ctypes.byref(plan)), "conv plan")
        blob = np.zeros(plan.weight_bytes, np.uint8)
        _check(lib.vkhip_conv_pack_weights(ctypes.byref(cd), ctypes.byref(plan), d["w"].ctypes.data, d["b"].ctypes.data, blob.ctypes.data), "conv weights")
        st.update(desc=cd, plan=plan, blob=_upload(blob), ws=torch.zeros(max(plan.workspace_bytes, 16), dtype=torch.uint8, device="cuda"))
    elif kind == "dwpw":
        pd = V.DwPwDesc(dw=_desc(c, c["c"], c["c"], c["c"], "relu6", False), Cout=c["cout"], act=ACT[c["act"]], act_lo=0.0,
                        act_hi=6.0 if c["act"] == "relu6" else 0.0, has_res=int(c["res"]))
        blob = np.zeros(lib.vkhip_dwpw_weight_bytes(ctypes.byref(pd)), np.uint8)
        _check(lib.vkhip_dwpw_pack_weights(ctypes.byref(pd), d["w"].ctypes.data, d["b"].ctypes.data, d["w2"].ctypes.data, d["b2"].ctypes.data,
                                           blob.ctypes.data), "dwpw weights")
        st.update(desc=pd, blob=_upload(blob))
    else:
        blob = np.zeros(lib.vkhip_se_weight_bytes(c["c"], c["cr"]), np.uint8)
        _check(lib.vkhip_se_pack_weights(c["c"], c["cr"], d["w1"].ctypes.data, d["b1"].ctypes.data, d["w2"].ctypes.data, d["b2"].ctypes.data,
                                         blob.ctypes.data), "se weights")
        rows = (c["n"], (c["c"] + 3) // 4 * 4)
        st.update(blob=_upload(blob), avg=torch.empty(rows, dtype=torch.float16, device="cuda"), gate=torch.empty(rows, dtype=torch.float16, device="cuda"),
                  ws=torch.zeros(lib.vkhip_se_workspace_bytes(c["n"], c["cr"]), dtype=torch.uint8, device="cuda"))
    torch.cuda.synchronize()
    return st


def run(state):
    kind, stream = state["kind"], state["stream"]
    if "model" in state:
        m = state["model"]
        m.stream.wait_stream(stream)  # the input the program wrote
        m.session.run_device()
        stream.wait_stream(m.stream)  # what the program does with the outputs
        return list(m.outputs)
    lib, c, s = state["lib"], state["case"], state["stream"].cuda_stream
    if kind == "conv" or kind == "dwconv":
        res = state["res"]
        _check(lib.vkhip_conv_forward(ctypes.byref(state["desc"]), ctypes.byref(state["plan"]), state["x"].data_ptr(), state["blob"].data_ptr(),
                                      res.data_ptr() if res is not None else None, state["y"].data_ptr(), state["ws"].data_ptr(), s), "conv")
        return [state["y"]]
    if kind == "dwpw":
        res = state["res"]
        _check(lib.vkhip_dwpw_forward(ctypes.byref(state["desc"]), state["x"].data_ptr(), state["blob"].data_ptr(),
                                      res.data_ptr() if res is not None else None, state["y"].data_ptr(), s), "dwpw")
        return [state["y"]]
    if kind == "se":
        n, ch, hw = c["n"], c["c"], c["h"] * c["w"]
        _check(lib.vkhip_global_avg_pool(state["x"].data_ptr(), state["avg"].data_ptr(), n, ch, c["h"], c["w"], s), "pool")
        _check(lib.vkhip_fused_se(state["avg"].data_ptr(), state["blob"].data_ptr(), state["gate"].data_ptr(), n, ch, c["cr"], 1.0 / 6, 0.5,
                                  state["ws"].data_ptr(), s), "se")
        _check(lib.vkhip_channel_scale(state["x"].data_ptr(), state["gate"].data_ptr(), state["y"].data_ptr(), n, ch, hw, s), "scale")
        return [state["gate"], state["y"]]
    n, hw = c["n"], c["hw"]
    f = state["unpacked"].shape
    _check(lib.vkhip_pack_nchw_f32(state["image"].data_ptr(), state["packed"].data_ptr(), n, 3, hw, hw, s), "pack")
    _check(lib.vkhip_unpack_nchw_f32(state["features"].data_ptr(), state["unpacked"].data_ptr(), f[0], f[1], f[2], f[3], s), "unpack")
    return [state["packed"], state["unpacked"]]


# ------------------------------------------------------------------------------------ float64 values
def _conv64(x, w, b, s, group):
    """Same-padded convolution tap by tap."""
    n, c, h, wd = x.shape
    co, _, k, _ = w.shape
    p = k // 2
    oh, ow = (h + 2 * p - k) // s + 1, (wd + 2 * p - k) // s + 1
    xp = torch.nn.functional.pad(x, (p, p, p, p)) if p else x
    y = torch.zeros((n, co, oh, ow), dtype=torch.float64, device=x.device)
    for ky in range(k):
        for kx in range(k):
            t = xp[:, :, ky:ky + (oh - 1) * s + 1:s, kx:kx + (ow - 1) * s + 1:s]
            if group > 1:
                y += t * w[:, 0, ky, kx].view(1, co, 1, 1)
            else:
                y += torch.matmul(w[:, :, ky, kx].contiguous(), t.reshape(n, c, oh * ow)).view(n, co, oh, ow)
    return y + b.view(1, co, 1, 1)


def _maxpool64(x, k, s, p):
    n, c, h, w = x.shape
    oh, ow = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1
    xp = torch.nn.functional.pad(x, (p, p, p, p), value=float("-inf"))
    y = None
    for ky in range(k):
        for kx in range(k):
            t = xp[:, :, ky:ky + (oh - 1) * s + 1:s, kx:kx + (ow - 1) * s + 1:s]
            y = t if y is None else torch.maximum(y, t)
    return y


def _act64(v, act):
    if act == "relu":
        return v.clamp(min=0)
    if act == "relu6":
        return v.clamp(0, 6)
    if act == "hardswish":
        return v * (v + 3).clamp(0, 6) / 6
    return v * torch.sigmoid(v) if act == "silu" else v


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("resnet50", "mnv3_block", "c2f"):
        return _model(c, seed).run64(_model_input(c, seed))
    if kind == "boundary":
        f = (c["n"], c["c"], c["hw"] // 8, c["hw"] // 8)
        return [_nc4(_act_tensor(c["n"], 3, c["hw"], c["hw"], seed, 1), torch.float64), _act_tensor(*f, seed, 2).double()]
    d = {k: (torch.from_numpy(v).cuda() if isinstance(v, np.ndarray) else v).double() for k, v in _layer_inputs(c, seed).items()}
    if kind == "se":
        avg = d["x"].mean((2, 3))
        gate = (((avg @ d["w1"].t() + d["b1"]).clamp(min=0) @ d["w2"].t() + d["b2"]) / 6 + 0.5).clamp(0, 1)
        row = torch.zeros((c["n"], (c["c"] + 3) // 4 * 4), dtype=torch.float64, device="cuda")
        row[:, :c["c"]] = gate
        return [row, _nc4(d["x"] * gate.view(c["n"], c["c"], 1, 1), torch.float64)]
    if kind == "dwpw":
        t = _conv64(d["x"], d["w"], d["b"], c["s"], c["c"]).clamp(0, 6)
        v, act = _conv64(t, d["w2"], d["b2"], 1, 1), c["act"]
    else:
        v, act = _conv64(d["x"], d["w"], d["b"], c["s"], c["c"] if kind == "dwconv" else 1), c["act"]
    if "res" in d:
        v = v + d["res"]
    return [_nc4(_act64(v, act), torch.float64)]


# ------------------------------------------------------------------------------------ work, tolerance
def _blocks(c):
    return (c + 3) // 4 * 4


def work(case):
    """fp16 NC4HW4 (sessions: fp32 NCHW) inputs read once, outputs written once, fp16 weights read once."""
    c, kind = case, case["kind"]
    if kind == "conv":
        oh, ow = _out_hw(c)
        x, y = c["n"] * _blocks(c["cin"]) * c["h"] * c["w"], c["n"] * _blocks(c["cout"]) * oh * ow
        wt = c["cout"] * c["cin"] * c["k"] ** 2
        return {"bytes": 2 * (x + y * (2 if c["res"] else 1) + wt) + 4 * c["cout"], "flops": 2 * c["n"] * oh * ow * wt}
    if kind == "dwconv":
        oh, ow = _out_hw(c)
        return {"bytes": 2 * c["n"] * _blocks(c["c"]) * (c["h"] * c["w"] + oh * ow) + 2 * c["c"] * (c["k"] ** 2 + 2),
                "flops": 2 * c["n"] * c["c"] * oh * ow * c["k"] ** 2}
    if kind == "dwpw":
        oh, ow = _out_hw(c)
        out = c["n"] * _blocks(c["cout"]) * oh * ow
        return {"bytes": 2 * (c["n"] * _blocks(c["c"]) * c["h"] * c["w"] + out * (2 if c["res"] else 1)) + 2 * c["c"] * (c["k"] ** 2 + c["cout"]),
                "flops": 2 * c["n"] * oh * ow * c["c"] * (c["k"] ** 2 + c["cout"])}
    if kind == "se":
        x = c["n"] * _blocks(c["c"]) * c["h"] * c["w"]
        return {"bytes": 2 * 2 * x + 4 * c["c"] * c["cr"], "flops": 2 * x + 4 * c["n"] * c["c"] * c["cr"]}
    if kind == "boundary":
        px, ft = c["n"] * c["hw"] ** 2, c["n"] * (c["hw"] // 8) ** 2
        return {"bytes": px * (3 * 4 + 4 * 2) + ft * (_blocks(c["c"]) * 2 + c["c"] * 4), "flops": 0}
    # sessions: the products of every conv and FC; the input, the outputs and the weights
    n = c["n"]
    if kind == "resnet50":
        hw = lambda k: -(-c["hw"] // k)  # noqa: E731
        flops, wts, cin = 2 * n * hw(2) ** 2 * 64 * 147, 64 * 147, 64
        for stage, blocks in enumerate((3, 4, 6, 3)):
            mid, px = 64 << stage, hw(4 << stage) ** 2
            for i in range(blocks):
                wide = px if i or not stage else hw(2 << stage) ** 2
                wt = [cin * mid, 9 * mid * mid, 4 * mid * mid] + ([cin * 4 * mid] if i == 0 else [])
                flops += 2 * n * (wt[0] * wide + sum(wt[1:]) * px)
                wts += sum(wt)
                cin = 4 * mid
        return {"bytes": 4 * n * (3 * c["hw"] ** 2 + 1000) + 2 * (wts + 2048000), "flops": flops + 2 * n * 2048000}
    px = c["h"] * c["w"]
    if kind == "mnv3_block":
        cr = max(8, (c["e"] // 4 + 7) // 8 * 8)
        return {"bytes": 4 * n * c["c"] * px * 2 + 2 * c["e"] * (2 * c["c"] + c["k"] ** 2 + 2 * cr),
                "flops": 2 * n * px * c["e"] * (2 * c["c"] + c["k"] ** 2) + 4 * n * c["e"] * cr}
    wt = c["c"] ** 2 + c["reps"] * 18 * (c["c"] // 2) ** 2 + (2 + c["reps"]) * (c["c"] // 2) * c["c"]
    return {"bytes": 4 * n * c["c"] * px * 2 + 2 * wt, "flops": 2 * n * px * wt}


def tolerance(case):
    """About four times the measured distance from float64, which is at most 2.5e-4 (2-norm) for a
    layer that rounds once to fp16, 3.1e-4 for the squeeze-excite's second product, 4.2e-4 for the
    blocks and 3.4e-4 for the network, which round every intermediate tensor. Single values: two
    fp16 steps (1e-3 each) of a layer, and what the blocks' longer chains of roundings add up to."""
    return {"boundary": "exact",
            "conv": {"rel": 1e-3, "max": 4e-3}, "dwconv": {"rel": 1e-3, "max": 4e-3}, "dwpw": {"rel": 1e-3, "max": 8e-3},
            "se": {"rel": 1.3e-3, "max": 8e-3}, "mnv3_block": {"rel": 1.7e-3, "max": 2e-2}, "c2f": {"rel": 1.7e-3, "max": 2e-2},
            "resnet50": {"rel": 1.5e-3, "max": 2e-2}}[case["kind"]]
