"""The launch that adds K slices up, four columns a thread from 2^18 sums on: the bits of the launch that adds one column a thread, which
runs for an image of the batch on its own.  Planes of a multiple of four pixels and others, slices up to more than eight, rows off the workgroup's four,
each activation, with and without a bias, an addend and the Relu behind it."""
import pytest

from onenew_amd import abi, hip
from onenew_amd.abi import ConvDesc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("split", [2, 5, 8, 12])
@pytest.mark.parametrize("cout,h,w,n", [(65, 14, 14, 24), (256, 14, 14, 6), (130, 7, 7, 44), (67, 6, 6, 120), (160, 9, 5, 40)])
@pytest.mark.parametrize("act,bias,addend,relu", [(abi.NOT_ACT, True, True, True), (abi.CLIP, True, False, False), (abi.NOT_ACT, False, True, False), (abi.SILU, True, True, True)])
def test_sums_of_slices(cout, h, w, n, split, act, bias, addend, relu, monkeypatch):
    import torch
    hip.init(0)
    assert n * cout * h * w >= 1 << 18 > cout * h * w
    print(f"{n} x {cout} x {h} x {w} in {split} slices, activation {act}", flush=True)
    monkeypatch.setenv("ONHIP_TILE", f"64x64x{split}x0x2")
    cin = 16 * 120   # K tiles that every count of slices divides
    d = ConvDesc(n=n, cin=cin, h=h, w=w, cout=cout, kh=1, kw=1, stride_h=1, stride_w=1, pad_t=0, pad_l=0, pad_b=0, pad_r=0, group=1, has_bias=int(bias), act_type=act,
                 compute=abi.COMPUTE_F32)
    d.clip_min, d.clip_max = -0.5, 0.75
    g = torch.Generator(device="cuda").manual_seed(cout + split)
    x = torch.randn((n, cin, h, w), generator=g, device="cuda")
    wt = torch.randn((cout, cin, 1, 1), generator=g, device="cuda") / cin ** 0.5
    b = torch.randn((cout,), generator=g, device="cuda") if bias else None
    r = torch.randn((n, cout, h, w), generator=g, device="cuda") if addend else None
    lut = (lambda t: t * torch.sigmoid(t))(torch.arange(8192, dtype=torch.float64) / 512 - 8).float().cuda() if act == abi.SILU else None
    run = lambda d, x, r: hip.conv2d_f32_add(d, x, wt, r, b, lut, relu=relu) if addend else hip.conv2d_f32(d, x, wt, b, lut)  # noqa: E731
    whole = run(d, x, r)
    torch.cuda.synchronize()
    choice = hip.last_launch_choice()
    assert choice[2] == split and choice[4] == 2, choice
    d.n = 1
    parts = torch.cat([run(d, x[i:i + 1].contiguous(), r[i:i + 1].contiguous() if addend else None) for i in range(n)])
    assert torch.equal(whole, parts)
