"""Patch layers (filters of more than 64 taps whose windows all lie inside the image) on the fp32 kernel on the 16-bit matrix cores, against
64-bit sums; bounds as in test_gpu_f3."""
import pytest

from onenew_amd import hip
from test_gpu_f3 import check, conv_desc, conv_ref

pytestmark = pytest.mark.gpu

# (n, cin, h, w, cout, filter, stride, pad): windows that end with the image and that leave rows and columns over, K off sixteen, overlapping
# windows, one window an image
LAYERS = [(2, 3, 64, 48, 70, 16, 16, 0), (1, 3, 50, 37, 33, 9, 5, 0), (3, 5, 20, 20, 40, 10, 1, 0), (70, 2, 12, 13, 66, 12, 3, 0), (1, 3, 224, 224, 192, 16, 16, 0)]


@pytest.mark.parametrize("tile", [(64, 64), (192, 64), (256, 128)], ids=str)
@pytest.mark.parametrize("special", [False, True], ids=["finite", "special"])
@pytest.mark.parametrize("layer", LAYERS, ids=str)
def test_patch_layer(layer, special, tile, monkeypatch):
    import torch
    hip.init(0)
    print("f3 patch", layer, special, tile, flush=True)
    monkeypatch.setenv("ONHIP_TILE", "%dx%dx1x0x2" % tile)
    d = conv_desc(*layer)
    g = torch.Generator().manual_seed(layer[1] + layer[4])
    x = torch.randn(d.n, d.cin, d.h, d.w, generator=g)
    w, b = torch.randn(d.cout, d.cin, d.kh, d.kw, generator=g) / (d.cin * d.kh * d.kw) ** 0.5, torch.randn(d.cout, generator=g)
    if special:
        x[0, 0, 1, 2], x[-1, 1, 2, 1], w[5, 1, 0, 0] = float("inf"), float("nan"), -3.4e38
    y = hip.conv2d_f32(d, x.cuda(), w.cuda(), b.cuda())
    assert hip.last_launch_choice()[:2] == tile and hip.last_launch_choice()[4] == 2
    ref, magnitude = conv_ref(torch, d, x, w, b)
    ok = (magnitude < 1e38) | ~magnitude.isfinite()
    check(y.cpu()[ok], ref[ok], magnitude[ok], d.cin * d.kh * d.kw)


def test_windows_over_the_edge_stay_with_the_other_kernels(monkeypatch):
    import torch
    hip.init(0)
    monkeypatch.setenv("ONHIP_TILE", "64x64x1x0x2")
    d = conv_desc(1, 3, 40, 40, 40, 9, 4, 2)
    hip.conv2d_f32(d, torch.randn(1, 3, 40, 40, device="cuda"), torch.randn(40, 3, 9, 9, device="cuda"), torch.randn(40, device="cuda"))
    assert hip.last_launch_choice()[4] != 2
