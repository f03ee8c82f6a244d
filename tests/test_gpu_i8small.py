"""W8A32 layers that run as one launch: the same bits as the staged form (activations quantised by a launch of their own), whose results the
oracle pins elsewhere."""
import pytest

from onenew_amd import abi, hip
from onenew_amd.abi import ConvDesc

pytestmark = pytest.mark.gpu

N, R, C, S = abi.NOT_ACT, abi.RELU, abi.CLIP, abi.SILU
# (n, cin, h, w, cout, filter, stride, pad, activation): channels below and off sixteen (odd counts of 16-byte units), rows and pixels off
# every tile, fewer steps of K than wavefronts, filters of even size, strides that leave pixels out, more padding than the filter needs,
# a wide pixel, one output pixel; then the four workgroup shapes in their own sizes
LAYERS = [(1, 3, 9, 11, 5, 3, 1, 1, R), (1, 16, 7, 7, 33, 1, 1, 0, N), (2, 40, 13, 9, 64, 3, 2, 1, S), (1, 72, 20, 20, 128, 3, 1, 1, S), (1, 31, 17, 23, 30, 5, 1, 2, C),
          (1, 48, 14, 14, 70, 7, 2, 3, S), (3, 20, 5, 6, 17, 2, 1, 0, R), (1, 33, 12, 10, 40, 3, 3, 4, S), (1, 592, 6, 6, 40, 3, 1, 1, S), (5, 24, 3, 3, 20, 3, 1, 0, S),
          (1, 64, 80, 80, 64, 3, 1, 1, S), (1, 128, 80, 80, 128, 1, 1, 0, S), (4, 128, 40, 40, 128, 3, 1, 1, S), (1, 512, 20, 20, 70, 3, 1, 1, S), (2, 144, 52, 51, 100, 1, 1, 0, S)]


def layer(torch, n, cin, h, w, cout, k, stride, pad, act, bias=1):
    d = ConvDesc(n=n, cin=cin, h=h, w=w, cout=cout, kh=k, kw=k, stride_h=stride, stride_w=stride, pad_t=pad, pad_l=pad, pad_b=pad, pad_r=pad, group=1,
                 has_bias=bias, act_type=act, compute=abi.COMPUTE_F32)
    d.input_scale, d.clip_min, d.clip_max = 0.0123, 0.0, 6.0
    g = torch.Generator(device="cuda").manual_seed(cin * 7 + cout)
    w8 = torch.randint(-127, 128, (cout, cin, k, k), generator=g, device="cuda", dtype=torch.int8)
    x = torch.randn((n, cin, h, w), generator=g, device="cuda")
    x.view(-1)[::7] = torch.round(x.view(-1)[::7] / 0.0123 + 0.5) * 0.0123   # ties of the quantiser and their neighbours
    b32 = torch.randint(-9999, 9999, (cout,), generator=g, device="cuda", dtype=torch.int32)
    aux = torch.rand((cout,), generator=g, device="cuda") * 0.2 / (cin ** 0.5 * k)
    lut = torch.arange(8192, device="cuda", dtype=torch.float32) / 512 - 8
    return d, x, hip.pack_conv_weights_w8(d, w8), b32, aux, lut * torch.sigmoid(lut)


def both(torch, monkeypatch, d, x, wp, b32, aux, lut):
    before = hip.set_tuning(0)
    try:
        y = hip.conv2d_w8a32(d, x, wp, b32, aux, lut, packed=True)
        ran = hip.last_launch_choice()
        monkeypatch.setenv("ONHIP_NO_PATCH", "1")
        staged = hip.conv2d_w8a32(d, x, wp, b32, aux, lut, packed=True)
        assert hip.last_launch_choice()[4] == 0
    finally:
        monkeypatch.delenv("ONHIP_NO_PATCH", raising=False)
        hip.set_tuning(before)
    return y, staged, ran


@pytest.mark.parametrize("case", LAYERS, ids=[str(c) for c in LAYERS])
def test_layer(case, monkeypatch):
    import torch
    hip.init(0)
    print("i8small", case, flush=True)
    y, staged, ran = both(torch, monkeypatch, *layer(torch, *case))
    assert ran[4] == 4
    assert torch.equal(y, staged) and bool((y != 0).any())


def test_the_layers_take_every_workgroup_shape():
    import torch
    hip.init(0)
    seen, before = set(), hip.set_tuning(0)
    try:
        for case in LAYERS:
            hip.conv2d_w8a32(*layer(torch, *case), packed=True)
            seen.add(tuple(hip.last_launch_choice()[:2]))
    finally:
        hip.set_tuning(before)
    assert seen >= {(32, 32), (64, 32), (128, 32), (64, 64)}


# the forms either side: int8 or fp32 in; int8, fp32, or fp32 after an Add (and Relu) with its int8 twin out
FORMS = ["s8 to s8", "f32 to s8", "s8 to f32", "s8 add", "s8 add relu"]
LINKS = [(1, 16, 7, 7, 33, 1, 1, 0, N), (2, 40, 13, 9, 64, 3, 2, 1, R), (1, 72, 20, 20, 128, 3, 1, 1, S), (1, 576, 7, 7, 160, 1, 1, 0, N), (8, 960, 7, 7, 176, 1, 1, 0, C),
         (1, 512, 20, 20, 80, 3, 1, 1, S), (8, 256, 14, 14, 256, 3, 1, 1, R), (1, 48, 14, 14, 70, 7, 2, 3, S), (5, 24, 3, 3, 20, 3, 1, 0, C), (3, 2048, 7, 7, 272, 1, 1, 0, N)]


def link_fits(case, form):
    """a twin has channels in sixteens, an Add follows no table activation here"""
    return "add" not in form or (case[4] % 16 == 0 and case[8] != S)


def run_link(torch, case, form):
    """-> result, its int8 twin (of an Add) or None, the kernel that ran"""
    d, x, wp, b32, aux, lut = layer(torch, *case)
    d.output_scale, d.out_s8 = 0.031, int(form.endswith("to s8"))
    add = "add" in form
    src = dict(x=x) if form.startswith("f32") else dict(xq=hip.quantize_nhwc_s8(x, d.input_scale))
    oh, ow = d.out_hw()
    g = torch.Generator(device="cuda").manual_seed(5)
    addend = torch.randn((d.n, d.cout, oh, ow), generator=g, device="cuda") if add else None
    twin = torch.full((d.n, oh, ow, d.cout), 55, dtype=torch.int8, device="cuda") if add else None
    out = torch.full((d.n, oh, ow, (d.cout + 15) // 16 * 16), 55, dtype=torch.int8, device="cuda") if d.out_s8 else torch.full((d.n, d.cout, oh, ow), 55.0, device="cuda")
    before = hip.set_tuning(0)
    try:
        hip.conv2d_w8_link(d, wp, b32, aux, lut, addend=addend, relu_after="relu" in form, out=out, twin=twin, **src)
    finally:
        hip.set_tuning(before)
    return out, twin, hip.last_launch_choice()[4]


@pytest.mark.parametrize("case,form", [(c, f) for c in LINKS for f in FORMS if link_fits(c, f)], ids=str)
def test_link(case, form, monkeypatch):
    import torch
    hip.init(0)
    print("i8small", form, case, flush=True)
    out, twin, _ = run_link(torch, case, form)
    monkeypatch.setenv("ONHIP_NO_PATCH", "1")
    staged, staged_twin, ran = run_link(torch, case, form)
    assert ran == 0 and torch.equal(out, staged) and bool((out != 0).any())
    assert twin is None or torch.equal(twin, staged_twin)


@pytest.mark.parametrize("form", FORMS)
def test_two_layers_or_more_take_each_form(form):
    import torch
    hip.init(0)
    assert sum(run_link(torch, case, form)[2] == 4 for case in LINKS if link_fits(case, form)) >= 2


def test_no_bias_leaves_the_activation_out(monkeypatch):
    import torch
    hip.init(0)
    d, x, wp, b32, aux, lut = layer(torch, 1, 48, 10, 10, 40, 3, 1, 1, S, bias=0)
    y, staged, ran = both(torch, monkeypatch, d, x, wp, None, aux, lut)
    assert ran[4] == 4 and torch.equal(y, staged) and bool((y < -1e-3).any())


def test_values_that_are_not_finite_and_beyond_the_clamp(monkeypatch):
    import torch
    hip.init(0)
    d, x, wp, b32, aux, lut = layer(torch, 1, 40, 9, 9, 33, 3, 1, 1, R)
    flat = x.view(-1)
    for i, v in enumerate([float("nan"), float("inf"), float("-inf"), 3.4e38, -3.4e38, 1e9, -1e9, -0.0, 127.5 * 0.0123, -128.5 * 0.0123, 1e-45]):
        flat[i * 37::463] = v
    y, staged, ran = both(torch, monkeypatch, d, x, wp, b32, aux, lut)
    assert ran[4] == 4 and torch.equal(y, staged)


def test_many_tiles_stay_staged():
    """more workgroups than compute units: quantised once, by a launch of its own"""
    import torch
    hip.init(0)
    d, x, wp, b32, aux, lut = layer(torch, 4, 64, 112, 112, 64, 3, 1, 1, R)
    hip.conv2d_w8a32(d, x, wp, b32, aux, lut, packed=True)
    assert hip.last_launch_choice()[4] != 4


@pytest.mark.parametrize("case,ours", [((4, 1198, 5, 5, 248, 7, 3, 3, N), False), ((1, 832, 11, 11, 35, 7, 1, 3, R), False), ((2, 1844, 5, 5, 147, 5, 3, 2, S), False),
                                       ((1, 154, 11, 11, 1146, 7, 2, 3, R), True), ((4, 784, 6, 6, 948, 3, 3, 1, N), True), ((2, 811, 7, 7, 795, 3, 3, 1, S), True),
                                       ((1, 512, 7, 7, 96, 3, 1, 1, R), True), ((1, 800, 7, 7, 64, 3, 1, 1, N), True), ((2, 1366, 13, 13, 172, 3, 1, 1, R), True)])
def test_long_reductions_are_cut_into_slices(case, ours):
    """from int8 activations: where the other kernels cut K, one launch is the slower form of a long one"""
    import torch
    hip.init(0)
    print("i8small, long K", case, flush=True)
    d, x, wp, b32, aux, lut = layer(torch, *case)
    xq = hip.quantize_nhwc_s8(x, d.input_scale)
    y = hip.conv2d_w8_link(d, wp, b32, aux, lut, xq=xq)
    assert (hip.last_launch_choice()[4] == 4) == ours, hip.last_launch_choice()
    assert torch.equal(y, hip.conv2d_w8a32(d, x, wp, b32, aux, lut, packed=True))
