"""Performance cases: what a user of this framework has it do, through its public entry points.

Kinds
  conv       one convolution layer from Python: fp32, 16-bit storage, W8A32 (fp32 in and out) or the int8 chain form
  matmul     one fp32 MatMul with the bias and the table GELU of a linear layer fused in
  net        a whole .one model through the device-resident runtime: ResNet-50, MobileNetV2, ViT-Tiny; fp32 or W8A32
  stack      every convolution of YOLOv8s on operands of its own, int8 in both forms
  resnet16   ResNet-50 with 16-bit storage: the image's conversion, the stem, the four stages with their residual Adds
  vit16      transformer encoder blocks with 16-bit storage: projections, attention, MLP with their skip connections

`listed()` names twelve of them, `draw()` gives more over the same ranges, odd sizes among them.
"""
import math

import numpy as np
import torch

from onenew_amd import abi, hip, onefile, rt, stacks

ACTS = {"none": abi.NOT_ACT, "relu": abi.RELU, "clip": abi.CLIP, "silu": abi.SILU}
COMPUTE = {"f32": abi.COMPUTE_F32, "bf16": abi.COMPUTE_BF16, "f16": abi.COMPUTE_F16, "w8a32": abi.COMPUTE_F32, "w8a8": abi.COMPUTE_F32}
IN_SCALE, OUT_SCALE = 1.0 / 127, 0.03


def listed():
    return [
        # one convolution of a 56 x 56 feature map, batch 1: the latency of a single call
        dict(name="conv_f32_b1", kind="conv", dtype="f32", n=1, cin=64, h=56, w=56, cout=64, k=3, stride=1, act="relu", depthwise=False),
        # a single image through a whole model: interactive use, bound by launches
        dict(name="resnet50_f32_b1", kind="net", model="resnet50", dtype="f32", batch=1, image=224),
        # batch inference in the reference's own arithmetic
        dict(name="resnet50_f32_b32", kind="net", model="resnet50", dtype="f32", batch=32, image=224),
        # the bandwidth-bound model: depthwise and pointwise convolutions
        dict(name="mobilenetv2_f32_b64", kind="net", model="mobilenetv2", dtype="f32", batch=64, image=224),
        # a transformer encoder: linear layers, attention, layer norms, Transposes
        dict(name="vit_tiny_f32_b64", kind="net", model="vit_tiny", dtype="f32", batch=64, image=224),
        # the same models after the offline quantiser
        dict(name="resnet50_w8a32_b32", kind="net", model="resnet50", dtype="w8a32", batch=32, image=224),
        dict(name="mobilenetv2_w8a32_b8", kind="net", model="mobilenetv2", dtype="w8a32", batch=8, image=224),
        # 16-bit storage: convolutions with residual Adds, batch inference
        dict(name="resnet50_bf16_b32", kind="resnet16", dtype="bf16", batch=32, image=224),
        # 16-bit storage: transformer blocks, 197 tokens (a prime, so no tile divides it)
        dict(name="vit_bf16_b64", kind="vit16", dtype="bf16", batch=64, tokens=197, heads=3, depth=6),
        # a detector's convolutions, large images: int8 from layer to layer, a batch
        dict(name="yolov8s_w8a8_b16", kind="stack", dtype="w8a8", batch=16, image=640),
        # the same with the reference's own interface (fp32 between the layers), one image
        dict(name="yolov8s_w8a32_b1", kind="stack", dtype="w8a32", batch=1, image=640),
        # a linear layer that no tile divides
        dict(name="matmul_f32_ragged", kind="matmul", m=4099, kdim=1031, ncols=2053, bias=True, gelu=True),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["conv"] * 5 + ["net"] * 3 + ["matmul", "stack", "resnet16", "vit16"])
    if kind == "conv":
        while True:
            dtype = rng.choice(["f32", "f32", "f32", "bf16", "f16", "w8a32", "w8a8"])
            depthwise = dtype in ("f32", "w8a32", "w8a8") and rng.random() < 0.25
            cin = spread(3, 1024)
            c = dict(kind="conv", dtype=dtype, n=spread(1, 64), cin=cin, h=spread(7, 160), w=spread(7, 160),
                     cout=cin if depthwise else spread(16, 1024), k=3 if depthwise else rng.choice([1, 1, 3, 3, 5]),
                     stride=rng.choice([1, 1, 2]), act=rng.choice(["none", "relu", "clip", "silu"]), depthwise=depthwise)
            if work(c)["flops"] <= 60e9 and work(c)["bytes"] <= 1e9:
                return c
    if kind == "matmul":
        while True:
            c = dict(kind="matmul", m=spread(16, 16384), kdim=spread(32, 4096), ncols=spread(32, 4096), bias=rng.random() < 0.7, gelu=False)
            c["gelu"] = c["bias"] and rng.random() < 0.5
            if work(c)["flops"] <= 60e9:
                return c
    if kind == "net":
        model, dtype = rng.choice([("resnet50", "f32"), ("resnet50", "w8a32"), ("mobilenetv2", "f32"), ("mobilenetv2", "w8a32"), ("vit_tiny", "f32")])
        image = 16 * rng.randint(8, 16) if model == "vit_tiny" else rng.randint(128, 224)
        return dict(kind="net", model=model, dtype=dtype, batch=spread(1, 32 if model == "resnet50" else 48), image=image)
    if kind == "stack":
        return dict(kind="stack", dtype=rng.choice(["w8a8", "w8a32"]), batch=spread(1, 16), image=32 * rng.randint(10, 20))
    if kind == "resnet16":
        return dict(kind="resnet16", dtype=rng.choice(["bf16", "f16"]), batch=spread(1, 32), image=rng.randint(128, 224))
    heads = rng.choice([3, 6, 12])
    return dict(kind="vit16", dtype=rng.choice(["bf16", "f16"]), batch=spread(1, 96 // heads), tokens=rng.randint(50, 256), heads=heads,
                depth=6)


# ---- inputs -------------------------------------------------------------------------------------------------------

def _table(gelu):
    """the activation tables of the reference host: 8192 values over [-8, 8)"""
    x = torch.arange(8192, dtype=torch.float64) / 512 - 8
    y = x * 0.5 * (1 + torch.erf(x / math.sqrt(2.0))) if gelu else x * torch.sigmoid(x)
    return y.float().cuda()


class _Gen:
    """tensors on the GPU from one seed"""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, shape, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda") * std

    def uniform(self, shape, lo=-1.0, hi=1.0):
        return torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def int8(self, shape):
        """int8 weights as the offline quantiser leaves them: a bell whose ends are the type's"""
        return (torch.randn(shape, generator=self.g, device="cuda") * 32).clamp(-127, 127).to(torch.int8)


def _conv_desc(n, cin, h, w, cout, k, stride, act, dtype, depthwise=False, bias=True):
    d = abi.ConvDesc(n=n, cin=cin, h=h, w=w, cout=cout, kh=k, kw=k, stride_h=stride, stride_w=stride, pad_t=k // 2, pad_l=k // 2,
                     pad_b=k // 2, pad_r=k // 2, group=cin if depthwise else 1, has_bias=int(bias), act_type=ACTS[act])
    d.clip_min, d.clip_max = 0.0, 6.0
    d.compute = COMPUTE[dtype]
    if dtype in ("w8a32", "w8a8"):
        d.input_scale, d.output_scale, d.out_s8 = IN_SCALE, OUT_SCALE, int(dtype == "w8a8")
    return d


def _conv_layer(gen, d, dtype, lut):
    """a layer's operands as a program holds them between calls: activations, weights laid out once, result, workspace"""
    oh, ow = d.out_hw()
    kc = d.cin if d.group == 1 else 1
    L = dict(d=d, dtype=dtype, lut=lut if d.act_type == abi.SILU else None)
    if dtype in ("w8a32", "w8a8"):
        w8 = gen.int8((d.cout, kc, d.kh, d.kw))
        # the result's spread is about one: sums of kc * k * k products of a 73-wide uniform and a 32-wide bell
        spread = 73.0 * 32.0 * math.sqrt(kc * d.kh * d.kw) * d.input_scale
        L["aux"] = gen.uniform((d.cout,), 0.6, 1.4) * (127.0 / spread)
        L["b32"] = torch.round(gen.normal((d.cout,), 0.05 * spread / d.input_scale)).to(torch.int32)
        packed = hip.pack_conv_weights_w8(d, w8)
        L["w"], L["packed"] = (w8, False) if packed is None else (packed, True)
        x = gen.uniform((d.n, d.cin, d.h, d.w))
        if dtype == "w8a8":
            L["x"] = hip.quantize_nhwc_s8(x, d.input_scale)
            L["y"] = torch.empty((d.n, oh, ow, (d.cout + 15) // 16 * 16), dtype=torch.int8, device="cuda")
        else:
            L["x"] = x
            L["y"] = torch.empty((d.n, d.cout, oh, ow), device="cuda")
            L["ws"] = torch.empty(max(16, hip.conv2d_w8a32_workspace(d)), dtype=torch.uint8, device="cuda")
        return L
    w = gen.normal((d.cout, kc, d.kh, d.kw), math.sqrt(2.0 / (kc * d.kh * d.kw)))
    x = gen.uniform((d.n, d.cin, d.h, d.w))
    L["b"] = gen.normal((d.cout,), 0.01)
    if dtype == "f32":
        packed = hip.pack_conv_weights(d, w)
        L["w"], L["packed"] = (w, False) if packed is None else (packed, True)
        L["x"], L["y"] = x, torch.empty((d.n, d.cout, oh, ow), device="cuda")
    else:
        L["w"], L["x"] = hip.h16_pack_conv_weights(d, w), hip.h16_from_nchw(x, d.compute)
        L["y"] = torch.empty((d.n, oh, ow, hip.h16_pitch(d.cout)), dtype=L["x"].dtype, device="cuda")
    return L


def _run_layer(L):
    d = L["d"]
    if L["dtype"] == "w8a8":
        return hip.conv2d_w8a8_nhwc(d, L["x"], L["w"], L["b32"], L["aux"], L["lut"], out=L["y"])
    if L["dtype"] == "w8a32":
        return hip.conv2d_w8a32(d, L["x"], L["w"], L["b32"], L["aux"], L["lut"], out=L["y"], workspace=L["ws"], packed=L["packed"])
    if L["dtype"] == "f32":
        return hip.conv2d_f32(d, L["x"], L["w"], L["b"], L["lut"], out=L["y"], packed=L["packed"])
    return hip.conv2d_h16(d, L["x"], L["w"], L["b"], L["lut"], out=L["y"])


def _stack_descs(case):
    out = []
    for _, d in stacks.with_batch(stacks.yolov8s(), case["batch"]):
        d.h, d.w = d.h * case["image"] // 640, d.w * case["image"] // 640
        d.input_scale, d.output_scale, d.out_s8 = IN_SCALE, OUT_SCALE, int(case["dtype"] == "w8a8")
        out.append(d)
    return out


RESNET50 = [(64, 3, 1), (128, 4, 2), (256, 6, 2), (512, 3, 2)]
MOBILENETV2 = [(1, 16, 1, 1), (6, 24, 2, 2), (6, 32, 3, 2), (6, 64, 4, 2), (6, 96, 3, 1), (6, 160, 3, 2), (6, 320, 1, 1)]


class _ModelWriter:
    """a convolutional model as the reference's offline tools leave it (batch norm folded, activations fused, W8A32 on
    request), with seeded He-scaled weights; counts its own work on the way"""

    def __init__(self, rng, dtype, batch, image):
        self.m, self.rng, self.q = onefile.OneModel(), rng, dtype == "w8a32"
        self.batch, self.flops, self.bytes = batch, 0.0, 0.0
        self.x = self.m.input("input", (batch, 3, image, image)) if rng is not None else "input"
        self.hw = image

    def conv(self, name, x, cin, cout, k, stride, hw, act, group=1, gain=1.0, second_moment=1.0):
        """second_moment: of the input's values; an int8 convolution's input_scale covers five times their spread"""
        kc = cin if group == 1 else 1
        out_hw = (hw + 2 * (k // 2) - k) // stride + 1
        self.flops += 2.0 * self.batch * cout * out_hw * out_hw * kc * k * k
        self.bytes += (1 if self.q else 4) * cout * kc * k * k
        if self.rng is None:
            return name, out_hw
        w = self.rng.standard_normal((cout, kc, k, k), dtype=np.float32) * np.float32(gain * math.sqrt(2.0 / (kc * k * k)))
        b = self.rng.standard_normal(cout, dtype=np.float32) * np.float32(0.01)
        quant = None
        if self.q:
            w, _, aux = hip.quant_weight_bias(w, b)
            scale = 5.0 * math.sqrt(second_moment) / 127
            b = np.round(b / (scale * aux / 127)).astype(np.int32)
            quant = (aux, scale)
        return self.m.conv(name, x, w, b, name + "_out", stride=stride, pad=k // 2, group=group, act=act, clip=(0.0, 6.0), quant=quant), out_hw

    def head(self, x, features, classes=1000):
        self.flops += 2.0 * self.batch * classes * features
        self.bytes += 4 * classes * features + 4 * self.batch * classes
        if self.rng is None:
            return self
        x = self.m.flatten("flatten", self.m.global_avgpool("avgpool", x, "avgpool_out"), "flatten_out", axis=1)
        std = math.sqrt(1.0 / features)
        self.m.gemm("fc", x, self.rng.standard_normal((classes, features), dtype=np.float32) * np.float32(std),
                    self.rng.standard_normal(classes, dtype=np.float32) * np.float32(0.01), "logits")
        self.m.output("logits", (self.batch, classes))
        return self


def _resnet50(rng, dtype, batch, image):
    W = _ModelWriter(rng, dtype, batch, image)
    x, hw = W.conv("stem", W.x, 3, 64, 7, 2, image, abi.RELU, second_moment=1.0)
    if rng is not None:
        x = W.m.maxpool("maxpool", x, "maxpool_out", 3, 2, 1)
    hw, cin, mom = (hw + 2 - 3) // 2 + 1, 64, 2.0
    for si, (planes, blocks, stride) in enumerate(RESNET50):
        for b in range(blocks):
            p, s = f"s{si}.{b}", stride if b == 0 else 1
            y, _ = W.conv(p + ".conv1", x, cin, planes, 1, 1, hw, abi.RELU, second_moment=mom)
            y, out = W.conv(p + ".conv2", y, planes, planes, 3, s, hw, abi.RELU, second_moment=mom)
            skip = W.conv(p + ".down", x, cin, planes * 4, 1, s, hw, abi.NOT_ACT, gain=0.7, second_moment=mom)[0] if b == 0 else x
            y, _ = W.conv(p + ".conv3", y, planes, planes * 4, 1, 1, out, abi.NOT_ACT, gain=0.3, second_moment=mom)
            if rng is not None:
                x = W.m.relu(p + ".relu", W.m.add(p + ".add", y, skip, p + ".add_out"), p + ".relu_out")
            hw, cin, mom = out, planes * 4, mom * (1.18 if b else 0.6)
    return W.head(x, 2048)


def _mobilenetv2(rng, dtype, batch, image):
    W = _ModelWriter(rng, dtype, batch, image)
    x, hw = W.conv("stem", W.x, 3, 32, 3, 2, image, abi.CLIP)
    cin, bi = 32, 0
    for t, c, n, s in MOBILENETV2:
        for i in range(n):
            bi += 1
            stride, hidden, y = s if i == 0 else 1, cin * t, x
            if t != 1:
                y, _ = W.conv(f"b{bi}.expand", y, cin, hidden, 1, 1, hw, abi.CLIP)
            y, out = W.conv(f"b{bi}.dw", y, hidden, hidden, 3, stride, hw, abi.CLIP, group=hidden)
            y, _ = W.conv(f"b{bi}.project", y, hidden, c, 1, 1, out, abi.NOT_ACT, gain=0.7)
            x = W.m.add(f"b{bi}.add", y, x, f"b{bi}.add_out") if stride == 1 and cin == c and rng is not None else y
            hw, cin = out, c
    x, _ = W.conv("last", x, 320, 1280, 1, 1, hw, abi.CLIP)
    return W.head(x, 1280)


def _vit_tiny(rng, dtype, batch, image, blocks=12, D=192, H=3):
    """a ViT-Tiny/16 encoder (mean over the tokens in the place of a class token)"""
    W = _ModelWriter(rng, dtype, batch, image)
    m, g = W.m, image // 16
    T, hd = g * g, D // H
    W.flops += 2.0 * batch * T * D * 768 + blocks * (2.0 * batch * T * 12 * D * D + 4.0 * batch * H * T * T * hd)
    W.bytes += 4 * (768 * D + T * D + blocks * 12 * D * D)
    if rng is None:
        return W.head("x", D)

    def n(shape, std):
        return rng.standard_normal(shape, dtype=np.float32) * np.float32(std)

    def linear(name, x, k, cols, gain=1.0, gelu=False):
        y = m.add(name + ".bias", m.matmul(name, x, n((k, cols), gain / math.sqrt(k)), name + "_mm"), n((cols,), 0.02), name + "_out")
        return m.gelu(name + ".gelu", y, name + "_act") if gelu else y

    def norm(name, x):
        return m.layernorm(name, x, 1 + n((D,), 0.05), n((D,), 0.05), name + "_out")

    x = m.conv("patch", W.x, n((D, 3, 16, 16), 1 / math.sqrt(768)), n((D,), 0.02), "patch_out", stride=16)
    x = m.transpose("tokens.t", m.reshape("tokens.flat", x, "tokens_flat", (batch, D, T, 1)), "tokens_t", (0, 2, 1, 3))
    x = m.add("pos", m.reshape("tokens", x, "tokens", (batch, T, D)), n((T, D), 0.02), "embedded")
    for b in range(blocks):
        p = f"b{b}."
        y, heads = norm(p + "ln1", x), {}
        for which in "qkv":
            t = m.reshape(p + which + ".split", linear(p + which, y, D, D, gain=0.125 if which == "q" else 1.0), p + which + "_split", (batch, T, H, hd))
            heads[which] = m.transpose(p + which + ".heads", t, p + which + "_heads", (0, 2, 1, 3))
        kt = m.transpose(p + "k.t", heads["k"], p + "k_t", (0, 1, 3, 2))
        a = m.softmax(p + "attn", m.matmul(p + "scores", heads["q"], kt, p + "scores_out"), p + "attn_out")
        c = m.transpose(p + "merge", m.matmul(p + "ctx", a, heads["v"], p + "ctx_out"), p + "merged", (0, 2, 1, 3))
        c = linear(p + "proj", m.reshape(p + "merge.flat", c, p + "merged_flat", (batch, T, D)), D, D, gain=0.5)
        x = m.add(p + "res1", c, x, p + "res1_out")
        y = linear(p + "fc2", linear(p + "fc1", norm(p + "ln2", x), D, 4 * D, gelu=True), 4 * D, D, gain=0.5)
        x = m.add(p + "res2", y, x, p + "res2_out")
    x = m.reshape("pool.shape", norm("ln", x), "pool_in_t", (batch, T, D, 1))
    return W.head(m.reshape("pool.grid", m.transpose("pool.t", x, "pool_in", (0, 2, 1, 3)), "pool_grid", (batch, D, g, g)), D)


MODELS = {"resnet50": _resnet50, "mobilenetv2": _mobilenetv2, "vit_tiny": _vit_tiny}


def _resnet16_shapes(case):
    """(stem, [stage: [(conv1, conv2, conv3, down or None)]]) as descriptors"""
    n, image, dt = case["batch"], case["image"], case["dtype"]
    stem = _conv_desc(n, 3, image, image, 64, 7, 2, "relu", dt)
    hw, cin, stages = (stem.out_hw()[0] + 2 - 3) // 2 + 1, 64, []
    for planes, blocks, stride in RESNET50:
        stage = []
        for b in range(blocks):
            s = stride if b == 0 else 1
            c1 = _conv_desc(n, cin, hw, hw, planes, 1, 1, "relu", dt)
            c2 = _conv_desc(n, planes, hw, hw, planes, 3, s, "relu", dt)
            down = _conv_desc(n, cin, hw, hw, planes * 4, 1, s, "none", dt) if b == 0 else None
            hw, cin = c2.out_hw()[0], planes * 4
            stage.append((c1, c2, _conv_desc(n, planes, hw, hw, planes * 4, 1, 1, "none", dt), down))
        stages.append(stage)
    return stem, stages


def prepare(case, seed):
    gen = _Gen(seed)
    kind, S = case["kind"], dict(case=case)
    if kind == "conv":
        d = _conv_desc(case["n"], case["cin"], case["h"], case["w"], case["cout"], case["k"], case["stride"], case["act"], case["dtype"], case["depthwise"])
        S["layer"] = _conv_layer(gen, d, case["dtype"], _table(False))
    elif kind == "stack":
        lut = _table(False)
        S["layers"] = [_conv_layer(gen, d, case["dtype"], lut) for d in _stack_descs(case)]
    elif kind == "matmul":
        m, k, n = case["m"], case["kdim"], case["ncols"]
        S["a"], S["b"], S["y"] = gen.normal((m, k)), gen.normal((k, n), 1 / math.sqrt(k)), torch.empty((m, n), device="cuda")
        S["bias"], S["lut"] = gen.normal((n,), 0.02) if case["bias"] else None, _table(True) if case["gelu"] else None
    elif kind == "net":
        W = MODELS[case["model"]](np.random.Generator(np.random.SFC64(seed)), case["dtype"], case["batch"], case["image"])
        S["net"] = rt.Net(W.m.tobytes())
        S["x"] = gen.normal((case["batch"], 3, case["image"], case["image"]))
        S["y"] = torch.empty((case["batch"], 1000), device="cuda")
    elif kind == "resnet16":
        stem, stages = _resnet16_shapes(case)

        def layer(d, gain=1.0):
            w = gen.normal((d.cout, d.cin, d.kh, d.kw), gain * math.sqrt(2.0 / (d.cin * d.kh * d.kw)))
            oh, ow = d.out_hw()
            return dict(d=d, w=hip.h16_first_pack_weights(d, w) if d.cin == 3 else hip.h16_pack_conv_weights(d, w), b=gen.normal((d.cout,), 0.01),
                        y=torch.empty((d.n, oh, ow, hip.h16_pitch(d.cout)), dtype=torch.bfloat16 if case["dtype"] == "bf16" else torch.float16, device="cuda"))

        S["image"], S["stem"] = gen.normal((stem.n, 3, stem.h, stem.w)), layer(stem)
        S["stages"] = [[[layer(c1), layer(c2), layer(c3, 0.3), layer(down, 0.7) if down is not None else None] for c1, c2, c3, down in stage] for stage in stages]
        # what the stem's pooling would hand on (pooling has no 16-bit form: a program keeps the pooled tensor)
        first = stages[0][0][0]
        S["pooled"] = hip.h16_from_nchw(gen.normal((first.n, first.cin, first.h, first.w)).abs(), first.compute)
    else:
        H, T, n = case["heads"], case["tokens"], case["batch"]
        D, rows, comp = 64 * H, n * T, COMPUTE[case["dtype"]]

        def linear(k, cols, gain=1.0):
            return hip.h16_pack_matmul_weights(gen.normal((k, cols), gain / math.sqrt(k)), comp), k, cols, gen.normal((cols,), 0.02)

        S["blocks"] = [dict(qkv=linear(D, 3 * D), proj=linear(D, D, 0.35), fc1=linear(D, 4 * D), fc2=linear(4 * D, D, 0.35)) for _ in range(case["depth"])]
        S["x"], S["lut"] = hip.h16_from_rows(gen.normal((rows, D)), comp), _table(True)
        e = lambda cols: torch.empty((rows, cols), dtype=S["x"].dtype, device="cuda")  # noqa: E731
        S["qkv"], S["ctx"], S["mid"], S["wide"], S["out"] = e(3 * D), e(D), e(D), e(4 * D), [e(D), e(D)]
    return S


def run(S):
    case = S["case"]
    kind = case["kind"]
    if kind == "conv":
        return _run_layer(S["layer"])
    if kind == "stack":
        return [_run_layer(L) for L in S["layers"]]
    if kind == "matmul":
        return hip.matmul(S["a"], S["b"], S["bias"], S["lut"], out=S["y"])
    if kind == "net":
        S["net"].enqueue_raw([S["x"].data_ptr()], [S["y"].data_ptr()])
        return S["y"]
    if kind == "resnet16":
        L = S["stem"]
        outs = [hip.conv2d_h16_first(L["d"], hip.h16_first_from_nchw(L["d"], S["image"]), L["w"], L["b"], out=L["y"])]
        x = S["pooled"]
        for stage in S["stages"]:
            for c1, c2, c3, down in stage:
                y = hip.conv2d_h16(c1["d"], x, c1["w"], c1["b"], out=c1["y"])
                y = hip.conv2d_h16(c2["d"], y, c2["w"], c2["b"], out=c2["y"])
                skip = x if down is None else hip.conv2d_h16(down["d"], x, down["w"], down["b"], out=down["y"])
                x = hip.conv2d_h16(c3["d"], y, c3["w"], c3["b"], residual=skip, residual_relu=True, out=c3["y"])
            outs.append(x)
        return outs
    x, comp = S["x"], COMPUTE[case["dtype"]]
    n, T, H = case["batch"], case["tokens"], case["heads"]
    for b in S["blocks"]:
        w, k, cols, bias = b["qkv"]
        qkv = hip.linear_h16(x, w, k, cols, comp, bias=bias, out=S["qkv"])
        q, kk, v = qkv.view(n, T, 3, H, 64).permute(2, 0, 3, 1, 4).unbind(0)
        ctx = hip.attention(q, kk, v, scale=0.125, out=S["ctx"].view(n, T, 64 * H))
        w, k, cols, bias = b["proj"]
        mid = hip.linear_h16(ctx.view(n * T, 64 * H), w, k, cols, comp, bias=bias, residual=x, out=S["mid"])
        w, k, cols, bias = b["fc1"]
        wide = hip.linear_h16(mid, w, k, cols, comp, bias=bias, gelu_lut=S["lut"], out=S["wide"])
        w, k, cols, bias = b["fc2"]
        x = hip.linear_h16(wide, w, k, cols, comp, bias=bias, residual=mid, out=S["out"][0 if x is not S["out"][0] else 1])
    return x


# ---- what a pass cannot do without -----------------------------------------------------------------------------------

def _conv_work(d, eb_x, eb_w, eb_y):
    return {"bytes": float(d.algorithmic_bytes(eb_x=eb_x, eb_w=eb_w, eb_y=eb_y)), "flops": float(d.flops())}


def work(case):
    """2 operations per multiply-accumulate; a model's bytes are its input, its weights and its result, since the tensors
    between its layers need not leave the chip"""
    kind = case["kind"]
    widths = {"f32": (4, 4, 4), "bf16": (2, 2, 2), "f16": (2, 2, 2), "w8a32": (4, 1, 4), "w8a8": (1, 1, 1)}.get(case.get("dtype"))
    if kind == "conv":
        d = _conv_desc(case["n"], case["cin"], case["h"], case["w"], case["cout"], case["k"], case["stride"], case["act"], case["dtype"], case["depthwise"])
        return _conv_work(d, *widths)
    if kind == "stack":
        each = [_conv_work(d, *widths) for d in _stack_descs(case)]
        return {k: sum(e[k] for e in each) for k in ("bytes", "flops")}
    if kind == "matmul":
        m, k, n = case["m"], case["kdim"], case["ncols"]
        return {"bytes": 4.0 * (m * k + k * n + m * n + (n if case["bias"] else 0)), "flops": 2.0 * m * k * n}
    if kind == "net":
        W = MODELS[case["model"]](None, case["dtype"], case["batch"], case["image"])
        return {"bytes": W.bytes + 12.0 * case["batch"] * case["image"] ** 2, "flops": W.flops}
    if kind == "resnet16":
        stem, stages = _resnet16_shapes(case)
        first, last = stages[0][0][0], stages[-1][-1][2]
        convs = [stem] + [d for stage in stages for block in stage for d in block if d is not None]
        moved = 12.0 * stem.n * stem.h * stem.w + 2.0 * stem.n * 64 * math.prod(stem.out_hw()) + 2.0 * first.n * first.cin * first.h * first.w
        moved += sum(2.0 * s[-1][2].n * s[-1][2].cout * math.prod(s[-1][2].out_hw()) for s in stages)
        return {"bytes": moved + sum(2.0 * d.cout * d.cin * d.kh * d.kw for d in convs), "flops": float(sum(d.flops() for d in convs))}
    n, T, D = case["batch"], case["tokens"], 64 * case["heads"]
    return {"bytes": 4.0 * n * T * D + case["depth"] * 24.0 * D * D, "flops": case["depth"] * (24.0 * n * T * D * D + 4.0 * n * T * T * D)}


def tolerance(case):
    """int8 sums are whole numbers and the operations on them separately rounded ones: those results are the same for every
    order.  The others state about four times what was seen: fp32 with another tile and K split (another order of the sums;
    where a result goes through a table, a value next to a step of the table takes the neighbouring entry), 16 bits against
    64-bit sums with the same roundings of every stored tensor."""
    kind, dtype = case["kind"], case.get("dtype")
    if kind in ("conv", "stack") and (dtype in ("w8a8", "w8a32") or case.get("depthwise")):
        return "exact"
    if kind == "net":
        return {"rel": 2e-4, "max": 1e-3} if case["model"] == "vit_tiny" else {"rel": 3e-6, "max": 2e-5}
    if kind == "resnet16":
        return {"rel": 0.028, "max": 0.16} if dtype == "bf16" else {"rel": 4e-3, "max": 0.025}
    if kind == "vit16":
        return {"rel": 0.018, "max": 0.12} if dtype == "bf16" else {"rel": 3e-3, "max": 0.02}
    if dtype in ("bf16", "f16"):
        return {"rel": 1.6e-4, "max": 0.03} if dtype == "bf16" else {"rel": 1.1e-4, "max": 0.013}
    if case.get("act") == "silu" or case.get("gelu"):
        return {"rel": 1.2e-4, "max": 1.3e-2}
    return {"rel": 3e-6, "max": 3e-5}
