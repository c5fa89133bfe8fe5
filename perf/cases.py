"""What users of this library have it do, as cases that can be timed: whole int8 networks from the float image to the float
features, single ConvBias calls in every layout and sparsity, large convolutions between two layout conversions, and the
same arithmetic as separate operators.  Every case goes through the public entry points (megengine_amd.ops, and the plan
helpers of megengine_amd.workloads that an inference program calls once at load time).

A case is a dict with a "kind":

    resnet50      float images -> quantize -> NCHW4 -> stem -> max-pool -> NCHW32 -> 52 ConvBias layers -> mean -> float
    mobilenetv2   the inverted-residual blocks in NCHW4 (expand, depthwise, project) on a quantized 16-channel input
    conv          one ConvBias call with default arguments: the operator as a graph without weight pre-processing calls it
    relayout_conv NCHW -> NCHW32, one large ConvBias with a residual and a pre-processed filter, NCHW32 -> NCHW
    unfused       the convolution, its requantisation, the residual add, the activation and the pooling as operators of their own

Values: weights are Gaussian (32 steps of their scale), activations Gaussian or rectified Gaussian, and every layer's scales
put its outputs at about 40 quantization steps, so that few of them saturate, as in a calibrated network.
"""
import math

import numpy as np
import torch

from megengine_amd import _abi, ops, workloads

WEIGHT_STD = 32.0   # steps of the filter scale
OUT_STD = 40.0      # steps of the output scale


def listed():
    return [
        # one image, answered at once: 58 short launches, the time is latency and the host's
        dict(name="resnet50_b1", kind="resnet50", batch=1, size=224),
        # a serving batch of images of a size that no tile divides (193 -> 97 -> 49 -> 25 -> 13 -> 7)
        dict(name="resnet50_b7_odd", kind="resnet50", batch=7, size=193),
        # throughput: the batch of the benchmark
        dict(name="resnet50_b64", kind="resnet50", batch=64, size=224),
        # the mobile network on one image
        dict(name="mobilenetv2_b1", kind="mobilenetv2", batch=1, size=224),
        # the mobile network at the batch of the benchmark: depthwise and narrow pointwise layers, bytes more than products
        dict(name="mobilenetv2_b64", kind="mobilenetv2", batch=64, size=224),
        # the smallest call in use: a pointwise layer of one small feature map
        dict(name="conv_pw_small", kind="conv", fmt="NCHW32", n=1, ic=64, h=28, w=28, oc=64, f=1, stride=1, group=1,
             nonline="RELU", z=False),
        # one NCHW4 3x3 layer at batch 16 (configuration 0 of the benchmark)
        dict(name="conv_nchw4_3x3", kind="conv", fmt="NCHW4", n=16, ic=64, h=56, w=56, oc=64, f=3, stride=1, group=1,
             nonline="RELU", z=False),
        # plain NCHW with channel counts and an image size that nothing divides, with a residual: what a converted model brings
        dict(name="conv_nchw_odd", kind="conv", fmt="NCHW", n=6, ic=75, h=61, w=45, oc=150, f=3, stride=1, group=1,
             nonline="RELU", z=True),
        # a grouped bottleneck layer: 32 groups of 4 channels
        dict(name="conv_group32", kind="conv", fmt="NCHW4", n=16, ic=128, h=56, w=56, oc=128, f=3, stride=1, group=32,
             nonline="RELU", z=False),
        # depthwise beyond 3x3, odd image
        dict(name="conv_depthwise_5x5", kind="conv", fmt="NCHW4", n=16, ic=240, h=57, w=57, oc=240, f=5, stride=2, group=240,
             nonline="H_SWISH", z=False),
        # the large 3x3 of the benchmark's stress configuration, layout conversions included
        dict(name="relayout_conv_large", kind="relayout_conv", n=128, ic=256, h=64, w=64, oc=256, f=3, stride=1),
        # a graph whose fuser left everything apart
        dict(name="unfused", kind="unfused", n=32, ic=128, h=28, w=28, oc=256, f=1),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["resnet50", "mobilenetv2", "conv", "conv", "conv", "conv", "relayout_conv", "unfused"])
    while True:
        if kind in ("resnet50", "mobilenetv2"):
            c = dict(kind=kind, batch=_log(rng, 1, 64), size=rng.randint(112, 288))
        elif kind == "relayout_conv":
            c = dict(kind=kind, n=_log(rng, 8, 128), ic=32 * _log(rng, 2, 16), h=rng.randint(20, 80), w=rng.randint(20, 80),
                     oc=32 * _log(rng, 2, 32), f=rng.choice([1, 3, 3, 5]), stride=rng.choice([1, 1, 2]))
        elif kind == "unfused":
            c = dict(kind=kind, n=_log(rng, 1, 64), ic=32 * _log(rng, 1, 16), h=rng.randint(7, 57), w=rng.randint(7, 57),
                     oc=32 * _log(rng, 1, 16), f=rng.choice([1, 3]))
        else:
            sort = rng.choice(["NCHW32", "NCHW4", "NCHW", "group4", "group32", "depthwise"])
            c = dict(kind="conv", fmt=sort, n=_log(rng, 1, 64), ic=0, h=_log(rng, 7, 112), w=_log(rng, 7, 112), oc=0,
                     f=rng.choice([1, 3, 3, 5]), stride=rng.choice([1, 1, 2]), group=1,
                     nonline=rng.choice(["IDENTITY", "RELU", "RELU", "H_SWISH"]), z=rng.choice([False, False, True]))
            if sort == "NCHW32":
                c.update(ic=32 * _log(rng, 1, 32), oc=32 * _log(rng, 1, 32))
            elif sort == "NCHW4":
                c.update(ic=4 * _log(rng, 4, 128), oc=4 * _log(rng, 4, 128))
            elif sort == "NCHW":
                c.update(ic=_log(rng, 3, 256), oc=_log(rng, 8, 256))
            elif sort == "group4":
                g, per = _log(rng, 2, 64), rng.choice([4, 8, 16])
                c.update(fmt="NCHW4", group=g, ic=g * per, oc=g * per, f=3)
            elif sort == "group32":
                g, per = _log(rng, 2, 16), rng.choice([32, 64])
                c.update(fmt="NCHW32", group=g, ic=g * per, oc=g * per, f=3)
            else:
                ch = 4 * _log(rng, 4, 240)
                c.update(fmt="NCHW4", group=ch, ic=ch, oc=ch, f=rng.choice([3, 3, 5]))
        w = work(c)
        most = 0.55e12 if kind != "conv" else 0.1e12
        if w["flops"] <= most and w["bytes"] <= (1.6e9 if kind in ("resnet50", "mobilenetv2") else 0.6e9):
            return c


# ---- the networks -----------------------------------------------------------------------------------------------------

def _resnet50(batch, size):
    """workloads.resnet50 for any image size: every stage takes the size that its strided layers leave."""
    layer = workloads.Layer
    stem = layer("stem", "NCHW4", batch, 4, size, size, 64, 7, stride=2, pad=3)
    out = [stem]
    cin, h, prev = 64, _abi.out_size(stem.oh, 3, 1, 2, 1), "input:pool"
    for si, (mid, cout, blocks, stride) in enumerate([(64, 256, 3, 1), (128, 512, 4, 2), (256, 1024, 6, 2), (512, 2048, 3, 2)]):
        for b in range(blocks):
            s, p = stride if b == 0 else 1, "s%db%d" % (si + 1, b)
            ho = _abi.out_size(h, 3, 1, s, 1)
            out.append(layer(p + "c1", "NCHW32", batch, cin, h, h, mid, 1, src=prev))
            out.append(layer(p + "c2", "NCHW32", batch, mid, h, h, mid, 3, stride=s, pad=1, src=p + "c1"))
            if b == 0:
                out.append(layer(p + "ds", "NCHW32", batch, cin, h, h, cout, 1, stride=s, nonline="IDENTITY", src=prev))
            out.append(layer(p + "c3", "NCHW32", batch, mid, ho, ho, cout, 1, z=p + "ds" if b == 0 else prev, src=p + "c2"))
            prev, cin, h = p + "c3", cout, ho
    return out


def _mobilenetv2(batch, size):
    """workloads.mobilenet_v2 for any image size, with the residuals wired to the blocks' inputs."""
    layer = workloads.Layer
    out, cin, h, prev = [], 16, _abi.out_size(size, 3, 1, 2, 1), "input:first"
    for c, n, stride in [(24, 2, 2), (32, 3, 2), (64, 4, 2), (96, 3, 1), (160, 3, 2), (320, 1, 1)]:
        for i in range(n):
            s, hid, p = stride if i == 0 else 1, cin * 6, "c%d_%d" % (c, i)
            ho = _abi.out_size(h, 3, 1, s, 1)
            out.append(layer(p + "_expand", "NCHW4", batch, cin, h, h, hid, 1, src=prev))
            out.append(layer(p + "_dw", "NCHW4", batch, hid, h, h, hid, 3, stride=s, pad=1, group=hid, src=p + "_expand"))
            out.append(layer(p + "_project", "NCHW4", batch, hid, ho, ho, c, 1, nonline="IDENTITY",
                             z=prev if s == 1 and cin == c else None, src=p + "_dw"))
            prev, cin, h = p + "_project", c, ho
    return out


def _layers(case):
    return (_resnet50 if case["kind"] == "resnet50" else _mobilenetv2)(case["batch"], case["size"])


def _conv_layer(case):
    z = "input:z" if case.get("z") else None
    return workloads.Layer("conv", case.get("fmt", "NCHW32"), case["n"], case["ic"], case["h"], case["w"], case["oc"], case["f"],
                           stride=case.get("stride", 1), pad=case["f"] // 2, group=case.get("group", 1),
                           nonline=case.get("nonline", "IDENTITY"), z=z)


def work(case):
    """Every tensor that goes in or comes out of an operator once; two operations per multiply-add."""
    kind = case["kind"]
    if kind in ("resnet50", "mobilenetv2"):
        layers = _layers(case)
        b, f = sum(l.bytes for l in layers), sum(l.ops for l in layers)
        if kind == "resnet50":
            image, stem, last = case["batch"] * case["size"] ** 2, layers[0], layers[-1]
            pool = layers[1].n * 64 * layers[1].ih * layers[1].iw
            b += image * (3 * 5 + 7)                          # quantize, relayout to NCHW4
            b += stem.n * 64 * stem.oh * stem.ow + 3 * pool   # max-pool, relayout to NCHW32
            b += last.n * 2048 * (last.oh * last.ow + 6)      # mean, dequantize
        return dict(bytes=b, flops=f)
    l = _conv_layer(case)
    out = l.n * l.oc * l.oh * l.ow
    if kind == "conv":
        return dict(bytes=l.bytes, flops=l.ops)
    if kind == "relayout_conv":
        return dict(bytes=l.bytes + out + 2 * l.n * l.ic * l.ih * l.iw + 2 * out, flops=l.ops)
    pooled = l.n * l.oc * (l.oh // 2) * (l.ow // 2)
    # int32 convolution, requantisation, three-operand add and activation, pooling, dequantize
    return dict(bytes=l.bytes + 3 * out + 5 * out + 3 * out + 2 * out + out + pooled + 5 * pooled, flops=l.ops)


def tolerance(case):
    return "exact"


# ---- tensors ----------------------------------------------------------------------------------------------------------

class _Source:
    """Seeded tensors on the GPU and seeded scales on the host."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)
        self.r = np.random.RandomState(seed % (1 << 32))

    def s8(self, shape, std, relu=False):
        x = torch.randn(shape, generator=self.g, device="cuda").mul_(std).round_().clamp_(-127, 127)
        return (x.clamp_(min=0) if relu else x).to(torch.int8)

    def s32(self, shape, most):
        most = max(1, int(most))
        return torch.randint(-most, most + 1, shape, generator=self.g, device="cuda", dtype=torch.int32)

    def scale(self, lo=0.01, hi=0.06):
        return float(np.float32(math.exp(self.r.uniform(math.log(lo), math.log(hi)))))


def _layer_tensors(src, layer, s_src, mean_square, z=None):
    """Filter, bias and descriptor of a layer whose input has the given scale and mean square (in steps); z: scale and mean
    square of the residual.  The accumulators' spread is put at OUT_STD output steps (with a residual: 30, on top of the
    residual at 0.8 of its own steps).  -> (desc, filter, bias, output scale, mean square of the output)"""
    spread = math.sqrt((layer.ic // layer.group) * layer.f * layer.f * mean_square) * WEIGHT_STD
    if z is None:
        s_dst, steps, ms = src.scale(), OUT_STD, OUT_STD ** 2
    else:
        s_dst, steps = float(np.float32(z[0] * 1.25)), 30.0
        ms = 30.0 ** 2 + 0.64 * z[1]
    s_flt = float(np.float32(steps * s_dst / (spread * s_src)))
    desc = layer.desc(float(np.float32(s_src) * np.float32(s_flt)), z[0] if z else 1.0, s_dst)
    _, flt_s, bias_s, _ = _abi.conv_shapes(desc)
    flt, bias = src.s8(flt_s, WEIGHT_STD), src.s32(bias_s, 0.5 * spread)
    if layer.nonline == "RELU":
        ms *= 0.5 if z is None else 0.8
    return desc, flt, bias, s_dst, ms


def _prepare_net(case, src):
    """The plan of an inference program: weights, algorithms and pre-processed filters once, activations in one arena laid
    out by liveness (a layer that reads its residual for the last time writes over it), one bound launch per layer."""
    layers = _layers(case)
    at = {l.name: i for i, l in enumerate(layers)}
    last = {}
    for i, l in enumerate(layers):
        for name in (l.src, l.z):
            last[name] = i
    size = [l.n * l.oc * l.oh * l.ow for l in layers]
    specs = []
    for i, l in enumerate(layers):
        over = at[l.z] if l.z in at and last[l.z] == i and size[at[l.z]] == size[i] and l.z != l.src else None
        specs.append((size[i], i, last.get(l.name, i), over))
    offsets, top = workloads.first_fit_offsets(specs)
    arena = torch.zeros(top, dtype=torch.int8, device="cuda")

    st = dict(arena=arena)
    if case["kind"] == "resnet50":
        n, s = case["batch"], case["size"]
        st["image"] = torch.randn((n, 3, s, s), generator=src.g, device="cuda")
        st["s_image"] = s_image = float(np.float32(1 / 40.0))
        st["to_nchw4"] = ops.relayout_desc(_abi.RL_NCHW_NCHW4_IC_SMALL, (n, 3, s, s))
        first = layers[1]
        oh = layers[0].oh
        st["pool"] = _abi.make_pooling_desc("MAX", "NCHW4", n, 64, oh, oh, 3, 2, 1)
        st["to_nchw32"] = ops.relayout_desc(_abi.RL_NCHW4_NCHW32, (n, 16, first.ih, first.iw, 4))
        h = layers[-1].oh
        st["mean"] = _abi.make_pooling_desc("AVERAGE", "NCHW32", n, 2048, h, h, h, h, 0)
        st["q"] = torch.empty((n, 3, s, s), dtype=torch.int8, device="cuda")
        st["q4"] = torch.empty((n, 1, s, s, 4), dtype=torch.int8, device="cuda")
        st["pool4"] = torch.empty((n, 16, first.ih, first.iw, 4), dtype=torch.int8, device="cuda")
        pool32 = torch.empty((n, 2, first.ih, first.iw, 32), dtype=torch.int8, device="cuda")
        known = {None: (st["q4"], s_image, 0.75 * 1600.0)}
    else:
        l = layers[0]
        x = src.s8((l.n, l.ic // 4, l.ih, l.iw, 4), OUT_STD)
        known = {"input:first": (x, src.scale(), OUT_STD ** 2)}

    plan = []
    for i, l in enumerate(layers):
        x, s_x, ms_x = known[l.src]
        z = known[l.z] if l.z else None
        desc, flt, bias, s_dst, ms = _layer_tensors(src, l, s_x, ms_x, z[1:] if z else None)
        shape = _abi.conv_shapes(desc)[3]
        dst = arena[offsets[i]:offsets[i] + size[i]].view(shape)
        known[l.name] = (dst, s_dst, ms)
        if l.name == "stem":
            known["input:pool"] = (pool32, s_dst, 2.0 * ms)
        plan.append(dict(layer=l, desc=desc, src=x, flt=flt, bias=bias, z=z[0] if z else None, dst=dst))
    workloads.choose_algorithms(plan)
    st.update(calls=workloads.bind_plan(plan), plan=plan, s_out=known[layers[-1].name][1])
    if case["kind"] == "resnet50":
        st["pool32"] = pool32
    return st


def prepare(case, seed):
    src = _Source(seed)
    kind = case["kind"]
    st = dict(kind=kind)
    if kind in ("resnet50", "mobilenetv2"):
        st.update(_prepare_net(case, src))
        return st
    l = _conv_layer(case)
    s_src = src.scale()
    s_z = src.scale()
    has_z = kind == "relayout_conv" or bool(case.get("z"))
    if kind == "relayout_conv":
        l.z, l.nonline = "input:z", "H_SWISH"
    st["desc"], st["flt"], st["bias"], st["s_dst"], ms = _layer_tensors(src, l, s_src, OUT_STD ** 2, (s_z, OUT_STD ** 2) if has_z else None)
    src_s, _, _, dst_s = _abi.conv_shapes(st["desc"])
    if kind == "conv":
        st["src"] = src.s8(src_s, OUT_STD)
        st["z"] = src.s8(dst_s, OUT_STD) if has_z else None
    elif kind == "relayout_conv":
        st["x"] = src.s8((l.n, l.ic, l.ih, l.iw), OUT_STD)
        st["z"] = src.s8(dst_s, OUT_STD)
        st["to"] = ops.relayout_desc(_abi.RL_NCHW_NCHW32, (l.n, l.ic, l.ih, l.iw))
        st["back"] = ops.relayout_desc(_abi.RL_NCHW32_NCHW, dst_s)
        st["algo"], _ = ops.conv_bias_query(st["desc"], _abi.ALGO_HEURISTIC_PREPROCESS)
        st["pre"] = ops.conv_bias_preprocess(st["desc"], st["flt"], st["algo"])
        st["packed"] = torch.empty(src_s, dtype=torch.int8, device="cuda")
        st["y"] = torch.empty(dst_s, dtype=torch.int8, device="cuda")
        st["out"] = torch.empty((l.n, l.oc, l.oh, l.ow), dtype=torch.int8, device="cuda")
    else:
        # the convolution's int32 result is requantised by an operator of its own, so it keeps the accumulator scale
        st["s_acc"] = st["desc"].scale_bias
        st["desc"].dst_dtype = _abi.DT_QS32
        st["desc"].scale_dst = st["s_acc"]
        st["src"] = src.s8(src_s, OUT_STD)
        st["z"], st["s_z"] = src.s8(dst_s, OUT_STD), s_z
        st["gate"], st["s_gate"] = src.s8(dst_s, OUT_STD), src.scale()
        st["pool"] = _abi.make_pooling_desc("AVERAGE", "NCHW32", l.n, l.oc, l.oh, l.ow, 2)
    return st


def run(st):
    kind = st["kind"]
    if kind == "conv":
        return ops.conv_bias_exec(st["desc"], st["src"], st["flt"], st["bias"], st["z"])
    if kind == "resnet50":
        ops.typecvt_exec(st["image"], st["s_image"], st["q"])
        ops.relayout_exec(st["to_nchw4"], st["q"], st["q4"])
        calls = st["calls"]
        calls[0]()
        ops.pooling_exec(st["pool"], st["plan"][0]["dst"], st["pool4"])
        ops.relayout_exec(st["to_nchw32"], st["pool4"], st["pool32"])
        for call in calls[1:]:
            call()
        mean = ops.pooling_exec(st["mean"], st["plan"][-1]["dst"])
        return dict(features=ops.typecvt_exec(mean, st["s_out"]), activations=st["arena"], pooled=st["pool32"])
    if kind == "mobilenetv2":
        for call in st["calls"]:
            call()
        return dict(features=st["plan"][-1]["dst"], activations=st["arena"])
    if kind == "relayout_conv":
        ops.relayout_exec(st["to"], st["x"], st["packed"])
        if st["pre"] is not None:
            ops.conv_bias_exec_preprocessed(st["desc"], st["packed"], st["pre"], st["bias"], st["z"], st["y"], st["algo"])
        else:
            ops.conv_bias_exec(st["desc"], st["packed"], st["flt"], st["bias"], st["z"], st["y"], st["algo"])
        return ops.relayout_exec(st["back"], st["y"], st["out"])
    acc = ops.conv_bias_exec(st["desc"], st["src"], st["flt"], st["bias"])
    y = ops.requant_exec(acc, st["s_acc"], st["s_dst"], "RELU", st["z"], st["s_z"])
    gated = ops.elemwise_q_exec("FUSE_MUL_ADD3", [y, st["gate"], st["z"]], [st["s_dst"], st["s_gate"], st["s_z"]], st["s_dst"])
    act = ops.elemwise_q_exec("H_SWISH", [gated], [st["s_dst"]], st["s_dst"])
    total = ops.requant_exec(act, st["s_dst"], st["s_dst"], "RELU", y, st["s_dst"])
    pooled = ops.pooling_exec(st["pool"], total)
    return dict(acc=acc, y=y, gated=gated, act=act, total=total, pooled=pooled, floats=ops.typecvt_exec(pooled, st["s_dst"]))
