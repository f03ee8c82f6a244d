"""First-layer convolutions (stem.hip): output channels off a row tile of 32, one and two of them, widths off a segment of 128 pixels, one and several segments
a row, fewer items than workgroups and several a workgroup, either side of where segments of 64 pixels
take over, both weight layouts, planes and paddings so large that masked rows have to be bounded; against 64-bit sums, within what a chain of fp32 multiply-adds can be off."""
import pytest

from onenew_amd import abi, hip
from onenew_amd.abi import ConvDesc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("n,h,w,cout,k,stride,pad,act", [(1, 20, 33, 13, 7, 2, 3, abi.RELU), (5, 230, 224, 64, 7, 2, 3, abi.RELU), (3, 190, 257, 40, 7, 1, 3, abi.NOT_ACT), (9, 125, 300, 32, 7, 2, 0, abi.NOT_ACT),
                                                         (1, 224, 224, 64, 7, 2, 3, abi.RELU), (1, 20, 261, 50, 7, 1, 3, abi.NOT_ACT), (4, 63, 99, 33, 7, 2, 3, abi.RELU), (3, 85, 99, 33, 7, 2, 3, abi.RELU),
                                                         (1, 9, 7, 5, 3, 1, 1, abi.NOT_ACT), (2, 64, 260, 33, 3, 2, 1, abi.RELU), (2, 40, 129, 64, 3, 1, 1, abi.NOT_ACT), (1, 300, 128, 24, 3, 2, 1, abi.RELU)])
def test_stem(n, h, w, cout, k, stride, pad, act, packed):
    import torch
    hip.init(0)
    print(f"{n} x 3 x {h} x {w} -> {cout}, filter {k}, stride {stride}, packed {packed}", flush=True)
    d = ConvDesc(n=n, cin=3, h=h, w=w, cout=cout, kh=k, kw=k, stride_h=stride, stride_w=stride, pad_t=pad, pad_l=pad, pad_b=pad, pad_r=pad, group=1, has_bias=1, act_type=act,
                 compute=abi.COMPUTE_F32)
    g = torch.Generator().manual_seed(cout + w)
    x, wt, b = torch.randn((n, 3, h, w), generator=g), torch.randn((cout, 3, k, k), generator=g), torch.randn(cout, generator=g)
    wk = wt.cuda()
    guard = torch.full((n * cout * d.out_hw()[0] * d.out_hw()[1] + 64,), 7.0, device="cuda")
    y = guard[:-64].view(n, cout, *d.out_hw())
    hip.conv2d_f32(d, x.cuda(), hip.pack_conv_weights(d, wk) if packed else wk, b.cuda(), packed=packed, out=y)
    torch.cuda.synchronize()
    conv = lambda x, w, b: torch.nn.functional.conv2d(x.double(), w.double(), b.double(), stride=stride, padding=pad)  # noqa: E731
    ref, mass = conv(x, wt, b), conv(x.abs(), wt.abs(), b.abs())
    if act == abi.RELU:
        ref = ref.clamp(min=0.0)
    assert bool(((y.cpu().double() - ref).abs() <= mass * (3 * k * k + 4) * 2.0 ** -24).all())
    assert bool((guard[-64:] == 7.0).all())


# row_offset.hpp, far_rows: rows past the last output channel 2 GiB away (one row tile and two), patch rows below an image and above one
@pytest.mark.parametrize("h,w,cout,k,stride,pad_t,pad_b", [(4106, 4100, 5, 7, 1, 3, 3), (2901, 2899, 33, 3, 1, 1, 1), (10, 30000, 1, 3, 2, 1, 18000), (10, 30000, 1, 7, 2, 18000, 3)])
def test_masked_rows_far_away(h, w, cout, k, stride, pad_t, pad_b):
    import torch
    hip.init(0)
    print(f"3 x {h} x {w} -> {cout}, filter {k}, stride {stride}, {pad_t} rows above, {pad_b} below", flush=True)
    pad = k // 2
    d = ConvDesc(n=1, cin=3, h=h, w=w, cout=cout, kh=k, kw=k, stride_h=stride, stride_w=stride, pad_t=pad_t, pad_l=pad, pad_b=pad_b, pad_r=pad, group=1, has_bias=1, act_type=abi.NOT_ACT,
                 compute=abi.COMPUTE_F32)
    oh, ow = d.out_hw()
    g = torch.Generator().manual_seed(cout + k)
    x, wt, b = torch.randn((1, 3, h, w), generator=g), torch.randn((cout, 3, k, k), generator=g), torch.randn(cout, generator=g)
    guard = torch.full((cout * oh * ow + 64,), 7.0, device="cuda")
    y = guard[:-64].view(cout, oh, ow)
    hip.conv2d_f32(d, x.cuda(), wt.cuda(), b.cuda(), out=y)
    torch.cuda.synchronize()
    assert bool((guard[-64:] == 7.0).all())
    # rows whose patch has nothing of the image are the bias; where the image starts, in the middle and where it ends, eight rows each
    first, last = max(0, (pad_t - k) // stride + 1), min(oh, (pad_t + h - 1) // stride + 1)
    outside = torch.cat([y[:, :first].reshape(cout, -1), y[:, last:].reshape(cout, -1)], 1)
    assert bool((outside == b.cuda()[:, None]).all())
    rows = torch.nn.functional.pad(x, (pad, pad, k, k))   # row i of x is row i + k
    for r0 in sorted({first, (first + last) // 2 - 4, last - 8}):
        r0 = max(r0, first)
        r1 = min(r0 + 8, last)
        lo = r0 * stride - pad_t
        part = rows[:, :, lo + k:lo + k + (r1 - r0 - 1) * stride + k]
        conv = lambda x, w, b: torch.nn.functional.conv2d(x.double(), w.double(), b.double(), stride=stride)[0]  # noqa: E731
        ref, mass = conv(part, wt, b), conv(part.abs(), wt.abs(), b.abs())
        assert ref.shape == (cout, r1 - r0, ow)
        assert bool(((y[:, r0:r1].cpu().double() - ref).abs() <= mass * (3 * k * k + 4) * 2.0 ** -24).all())
