"""First-layer convolutions (stem.hip): output channels off a row tile of 32, one and two of them, widths off a segment of 128 pixels, one and several segments
a row, fewer items than workgroups and several a workgroup, either side of where segments of 64 pixels
take over, both weight layouts; against 64-bit sums, within what a chain of fp32 multiply-adds can be off."""
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
