"""The fp32 kernel whose wavefronts share K, on weights as given and on weights kept split, every tile at ragged sizes, against 64-bit
sums.  Bounds as in test_gpu_f3: a chain of fp32 multiply-adds (K 2^-24 sum |a b|), and what the left-out partial products can reach."""
import numpy as np
import pytest

from onenew_amd import abi, hip
from test_gpu_f3 import check, conv_desc, conv_ref

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    hip.init(0)
    return torch


SHAPES = [(16, 16, 4), (32, 32, 4), (32, 32, 8), (64, 32, 4)]   # tile, wavefronts
# (n, cin, h, w, cout, filter, stride, pad): rows and columns off every tile, one step of K, fewer steps than wavefronts, a count of steps
# that neither the wavefronts nor the ring of loads divides, columns of several images in a tile
LAYERS = [(1, 32, 5, 7, 16, 1, 1, 0), (2, 96, 9, 11, 37, 1, 1, 0), (3, 416, 5, 5, 97, 1, 2, 0), (1, 64, 14, 13, 70, 3, 1, 1), (2, 32, 11, 9, 33, 3, 2, 1),
          (5, 160, 3, 3, 129, 3, 1, 1), (1, 32, 12, 13, 66, 7, 1, 3)]


def operands(torch, d, seed, special):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(d.n, d.cin, d.h, d.w, generator=g)
    w, b = torch.randn(d.cout, d.cin, d.kh, d.kw, generator=g) / (d.cin * d.kh * d.kw) ** 0.5, torch.randn(d.cout, generator=g)
    if special:   # an infinity, a NaN, values that round to bf16 infinities (products with them stay finite)
        x[0, 0, 1, 2], x[-1, 1, 2, 1], x[0, 2, 2, 2], w[5, 3] = float("inf"), float("nan"), 3.4e38, -3.4e38
        x[:, 3] *= 1e-3
    return x, w, b


def compare(torch, d, y, x, w, b):
    ref, magnitude = conv_ref(torch, d, x, w, b)
    ok = (magnitude < 1e38) | ~magnitude.isfinite()   # sums that may overflow on the way are left to the infinities' and NaNs' own check
    check(y.cpu()[ok], ref[ok], magnitude[ok], d.cin * d.kh * d.kw)


@pytest.mark.parametrize("kept", [False, True], ids=["given", "split"])
@pytest.mark.parametrize("special", [False, True], ids=["finite", "special"])
@pytest.mark.parametrize("bm,bn,waves", SHAPES)
@pytest.mark.parametrize("layer", LAYERS, ids=[str(i) for i in range(len(LAYERS))])
def test_layer(layer, bm, bn, waves, special, kept, torch_dev, monkeypatch):
    from onenew_amd import ops
    torch = torch_dev
    print(f"kw {layer} tile {bm}x{bn}, {waves} wavefronts, special {special}, split {kept}", flush=True)
    monkeypatch.setenv("ONHIP_TILE", f"{bm}x{bn}x{waves}x0x3")
    d = conv_desc(*layer)
    x, w, b = operands(torch, d, bm + layer[1], special)
    if kept:
        y = torch.from_numpy(ops.Conv(ops.Plugin(hip.plugin_path("Conv")).eval, d, w.numpy(), b.numpy())(x.numpy()))
    else:
        packed = d.kh > 1
        y = hip.conv2d_f32(d, x.cuda(), hip.pack_conv_weights(d, w.cuda()) if packed else w.cuda(), b.cuda(), packed=packed)
    assert hip.last_launch_choice()[:3] == (bm, bn, waves) and hip.last_launch_choice()[4] == 3
    compare(torch, d, y, x, w, b)


@pytest.mark.parametrize("bm,bn,waves", SHAPES)
def test_stores(bm, bn, waves, torch_dev, monkeypatch):
    """the residual operand and the activations, bit for bit what the operators do to the plain store's result; the same bits again"""
    torch = torch_dev
    monkeypatch.setenv("ONHIP_TILE", f"{bm}x{bn}x{waves}x0x3")
    d = conv_desc(2, 96, 9, 11, 37, 1, 1, 0)
    x, w, b = (t.cuda() for t in operands(torch, d, 7, False))
    y = hip.conv2d_f32(d, x, w, b)
    r = torch.randn(y.shape, generator=torch.Generator().manual_seed(1)).cuda()
    for relu in (False, True):
        z = hip.conv2d_f32_add(d, x, w, r, b, relu=relu)
        assert hip.last_launch_choice()[4] == 3
        assert torch.equal(z, (y + r).clamp(min=0) if relu else y + r)
    d.act_type = abi.RELU
    assert torch.equal(hip.conv2d_f32(d, x, w, b), y.clamp(min=0))
    d.act_type, d.clip_min, d.clip_max = abi.CLIP, -0.5, 0.75
    assert torch.equal(hip.conv2d_f32(d, x, w, b), y.clamp(-0.5, 0.75))
    d.act_type = abi.SILU
    table = torch.linspace(-8, 8, 8192, device="cuda")
    z = hip.conv2d_f32(d, x, w, b, table)
    assert torch.equal(z, table[((y + 8) * 512).int().clamp(0, 8191).long()])   # |y| < 8
    d.act_type, d.has_bias = abi.NOT_ACT, 0
    assert torch.allclose(hip.conv2d_f32(d, x, w, None), y - b.view(1, -1, 1, 1), rtol=0, atol=1e-5)


@pytest.mark.parametrize("values", ["normal", "uneven", "spread"])
@pytest.mark.parametrize("cin,filt,hw", [(256, 1, 14), (1024, 1, 14), (64, 3, 28), (256, 3, 14)])
def test_error_no_larger_than_of_fp32_matrix_instructions(cin, filt, hw, values, torch_dev, monkeypatch):
    """both forms of the weights against the launches these layers ran as before, rms error over sum |a b|; operands spread over 2^+-4, and over
    2^+-24, where a term decides the sum and its own rounding the error (as in test_gpu_f3)"""
    from onenew_amd import ops
    torch = torch_dev
    d = conv_desc(1, cin, hw, hw, 128, filt, 1, filt // 2)
    x, w, b = operands(torch, d, cin, False)
    if values != "normal":
        g, e = torch.Generator().manual_seed(cin + 1), 4 if values == "uneven" else 24
        x, w = (t * 2.0 ** (2 * e * torch.rand(t.shape, generator=g) - e) for t in (x, w))
    b.zero_()
    ref, magnitude = conv_ref(torch, d, x, w, b)
    rms = lambda y: float(((y.double().cpu() - ref) / magnitude).square().mean().sqrt())  # noqa: E731
    xg, wg, bg = x.cuda(), w.cuda(), b.cuda()
    wk = hip.pack_conv_weights(d, wg) if filt > 1 else wg
    monkeypatch.setenv("ONHIP_TILE", "64x64x4")
    theirs = rms(hip.conv2d_f32(d, xg, wk, bg, packed=filt > 1))
    for bm, bn, waves in SHAPES:
        monkeypatch.setenv("ONHIP_TILE", f"{bm}x{bn}x{waves}x0x3")
        given = rms(hip.conv2d_f32(d, xg, wk, bg, packed=filt > 1))
        split = rms(torch.from_numpy(ops.Conv(ops.Plugin(hip.plugin_path("Conv")).eval, d, w.numpy(), b.numpy())(x.numpy())))
        assert hip.last_launch_choice()[4] == 3
        print(f"kw error K {cin * filt * filt} {values} {bm}x{bn}x{waves}: given {given:.2e}, split {split:.2e}, sliced {theirs:.2e}", flush=True)
        # rms over a few thousand outputs repeats within 10 %
        assert given <= 1.1 * theirs and split <= (1.25 if values == "spread" else 1.1) * theirs


def test_choice(torch_dev, monkeypatch):
    """a layer with few tiles takes the kernel by itself, a large one does not"""
    torch = torch_dev
    monkeypatch.delenv("ONHIP_TILE", raising=False)
    for layer, ours in (((1, 64, 56, 56, 64, 3, 1, 1), True), ((16, 64, 56, 56, 64, 3, 1, 1), False)):
        d = conv_desc(*layer)
        x, w, b = operands(torch, d, 3, False)
        y = hip.conv2d_f32(d, x.cuda(), hip.pack_conv_weights(d, w.cuda()), b.cuda(), packed=True)
        assert (hip.last_launch_choice()[4] == 3) == ours
        if ours:
            compare(torch, d, y, x, w, b)


@pytest.mark.parametrize("layer,ours", [((29, 848, 1, 1, 299, 1, 1, 0), False), ((96, 1280, 1, 1, 1000, 1, 1, 0), False), ((2, 16, 15, 15, 618, 1, 1, 0), False),
                                        ((8, 8, 24, 24, 47, 1, 1, 0), False), ((16, 432, 4, 4, 176, 1, 2, 0), False), ((64, 48, 1, 1, 1760, 3, 1, 1), (32, 32)), ((4, 64, 1, 1, 746, 1, 1, 0), (16, 16)), ((4, 1376, 2, 2, 110, 1, 1, 0), (16, 16))])
def test_choice_where_loads_or_steps_do_not_fit_it(layer, ours, torch_dev, monkeypatch):
    """one-pixel images (a cache line for each column of a load) and reductions of fewer steps than wavefronts"""
    torch = torch_dev
    monkeypatch.delenv("ONHIP_TILE", raising=False)
    d = conv_desc(*layer)
    x, w, b = (t.cuda() for t in operands(torch, d, 3, False))
    y = hip.conv2d_f32(d, x, hip.pack_conv_weights(d, w) if d.kh > 1 else w, b, packed=d.kh > 1)
    ran = hip.last_launch_choice()
    compare(torch, d, y, x.cpu(), w.cpu(), b.cpu())
    assert (ran[4] == 3 and ran[:2] == ours) if ours else ran[4] != 3, ran
