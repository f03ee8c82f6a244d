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


def test_tile_of_a_short_reduction(monkeypatch):
    """a layer whose K has nothing to cut: the tile is chosen by the time of its K tiles all the same"""
    import torch
    hip.init(0)
    print("int8 96 -> 24 56x56 batch 8", flush=True)
    d = ConvDesc(n=8, cin=96, h=56, w=56, cout=24, kh=1, kw=1, stride_h=1, stride_w=1, group=1, has_bias=1, act_type=abi.NOT_ACT, compute=abi.COMPUTE_F32)
    d.input_scale = 1.0 / 127
    g = torch.Generator(device="cuda").manual_seed(96)
    w8 = torch.randint(-127, 128, (24, 96, 1, 1), generator=g, device="cuda", dtype=torch.int8)
    x = torch.rand((8, 96, 56, 56), generator=g, device="cuda") * 2 - 1
    b32, aux = torch.randint(-9999, 9999, (24,), generator=g, device="cuda", dtype=torch.int32), torch.rand((24,), generator=g, device="cuda")
    wp, before = hip.pack_conv_weights_w8(d, w8), hip.set_tuning(0)
    try:
        y = hip.conv2d_w8a32(d, x, wp, b32, aux, packed=True)
        assert hip.last_launch_choice()[:3] == (64, 64, 1)
        monkeypatch.setenv("ONHIP_TILE", "32x128x1")
        other = hip.conv2d_w8a32(d, x, wp, b32, aux, packed=True)
        assert hip.last_launch_choice()[:2] == (32, 128)
    finally:
        hip.set_tuning(before)
    assert torch.equal(y, other) and bool((y > 0).any())


def test_slices_stay_in_the_callers_workspace():
    """Layers that run in K slices on two streams at once, each with a workspace of its own: nothing of the process is shared or
    allocated.  With a workspace that holds the int8 activations alone they run in one piece."""
    import ctypes as C

    import torch
    hip.init(0)
    print("int8 slices on two streams", flush=True)
    before, jobs, scratch = hip.set_tuning(0), [], hip.load().onhip_scratch_bytes()
    try:
        for cin, hw, cout in ((256, 20, 256), (512, 20, 64)):
            d = ConvDesc(n=1, cin=cin, h=hw, w=hw, cout=cout, kh=3, kw=3, stride_h=1, stride_w=1, pad_t=1, pad_l=1, pad_b=1, pad_r=1, group=1, has_bias=1,
                         act_type=abi.NOT_ACT, compute=abi.COMPUTE_F32)
            d.input_scale = 1.0 / 127
            g = torch.Generator(device="cuda").manual_seed(cin)
            w8 = torch.randint(-127, 128, (cout, cin, 3, 3), generator=g, device="cuda", dtype=torch.int8)
            x = torch.rand((1, cin, hw, hw), generator=g, device="cuda") * 2 - 1
            b32, aux = torch.zeros(cout, device="cuda", dtype=torch.int32), torch.rand((cout,), generator=g, device="cuda")
            wp, whole = hip.pack_conv_weights_w8(d, w8), torch.empty((1, cout, hw, hw), device="cuda")
            q = torch.empty(hw * hw * cin, device="cuda", dtype=torch.uint8)
            rc = hip.load().onhip_conv2d_w8a32_packed(C.byref(d), x.data_ptr(), wp.data_ptr(), b32.data_ptr(), aux.data_ptr(), None, whole.data_ptr(), None,
                                                      q.data_ptr(), (hw * hw * cin + 255) // 256 * 256, None)
            assert rc == 0 and hip.last_launch_choice()[2] == 1
            jobs.append((d, x, wp, b32, aux, whole, [torch.zeros_like(whole) for _ in range(50)],
                         torch.empty(hip.conv2d_w8a32_workspace(d), dtype=torch.uint8, device="cuda"), torch.cuda.Stream()))
        torch.cuda.synchronize()
        for i in range(50):
            for d, x, wp, b32, aux, _, y, ws, stream in jobs:
                with torch.cuda.stream(stream):
                    hip.conv2d_w8a32(d, x, wp, b32, aux, out=y[i], workspace=ws, packed=True)
                assert hip.last_launch_choice()[2] > 1
    finally:
        hip.set_tuning(before)
    torch.cuda.synchronize()
    assert hip.load().onhip_scratch_bytes() == scratch
    for job in jobs:
        assert all(torch.equal(y, job[5]) for y in job[6])
