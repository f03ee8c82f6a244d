"""W8A32 layers with few tiles and a long reduction: cut along K by the cost model, the same values as in one piece."""
import pytest

from onenew_amd import abi, hip
from onenew_amd.abi import ConvDesc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cin,hw,cout", [(256, 20, 256), (512, 20, 64), (251, 19, 130)])
def test_few_tiles_long_reduction(cin, hw, cout, monkeypatch):
    import torch
    hip.init(0)
    print(f"int8 {cin} -> {cout} {hw}x{hw}", flush=True)
    d = ConvDesc(n=1, cin=cin, h=hw, w=hw, cout=cout, kh=3, kw=3, stride_h=1, stride_w=1, pad_t=1, pad_l=1, pad_b=1, pad_r=1, group=1, has_bias=1,
                 act_type=abi.RELU, compute=abi.COMPUTE_F32)
    d.input_scale = 1.0 / 127
    g = torch.Generator(device="cuda").manual_seed(cin + cout)
    w8 = torch.randint(-127, 128, (cout, cin, 3, 3), generator=g, device="cuda", dtype=torch.int8)
    x = torch.rand((1, cin, hw, hw), generator=g, device="cuda") * 2 - 1
    b32, aux = torch.randint(-9999, 9999, (cout,), generator=g, device="cuda", dtype=torch.int32), torch.rand((cout,), generator=g, device="cuda")
    wp = hip.pack_conv_weights_w8(d, w8)
    before = hip.set_tuning(0)
    try:
        y = hip.conv2d_w8a32(d, x, wp, b32, aux, packed=True)
        assert hip.last_launch_choice()[2] > 1
        monkeypatch.setenv("ONHIP_TILE", "64x64x1")
        whole = hip.conv2d_w8a32(d, x, wp, b32, aux, packed=True)
        assert hip.last_launch_choice()[2] == 1
    finally:
        hip.set_tuning(before)
    torch.cuda.synchronize()
    assert torch.equal(y, whole) and bool((y > 0).any())
