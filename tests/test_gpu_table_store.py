"""Table activations in the store of fp32 results: the table read from LDS or from memory, by tile and count of workgroups, on both sides of the
counts at which it changes.  What the store gives is the table's entry for the result without an activation, bit for bit."""
import pytest

from onenew_amd import abi, hip
from onenew_amd.abi import ConvDesc

pytestmark = pytest.mark.gpu


def through_table(torch, y, table):
    """conv.c's rule: zero below -8, the value itself from 8 on, between them entry (v + 8) * 512"""
    z = table[((y + 8.0) * 512.0).int().clamp(0, 8191).long()]
    return torch.where(y < -8.0, torch.zeros_like(y), torch.where(y >= 8.0, y, z))


# (tile, rows, columns, K): 512 and 513 workgroups of 32 x 128, 768 and 769 of 64 x 64 (with more, a K on either side of the one up to which the table
# is in LDS: 24, and 64 with a residual operand), one, and more than a round of a tile that always has it in LDS
SIZES = [("32x128", 32, 512 * 128, 20), ("32x128", 29, 512 * 128 + 1, 20), ("32x128", 7, 40, 20), ("64x64", 64, 768 * 64, 20), ("64x64", 61, 768 * 64 + 3, 20),
         ("64x64", 64, 768 * 64, 65), ("64x64", 61, 768 * 64 + 3, 25), ("64x64", 61, 768 * 64 + 3, 64), ("64x64", 61, 768 * 64 + 3, 65), ("64x64", 200, 50, 20),
         ("64x64x2", 130, 385 * 64, 20), ("64x128", 64, 1025 * 128, 20), ("128x128", 100, 300 * 128, 20)]


@pytest.mark.parametrize("kind", ["f32", "w8a32", "add"])
@pytest.mark.parametrize("tile,rows,cols,k", SIZES)
def test_table(tile, rows, cols, k, kind, monkeypatch):
    import torch
    hip.init(0)
    if kind == "w8a32" and tile.endswith("x2"):
        pytest.skip("one K tile: nothing to cut")
    print("table store", tile, rows, cols, k, kind, flush=True)
    monkeypatch.setenv("ONHIP_TILE", tile)
    d = ConvDesc(n=1, cin=k, h=1, w=cols, cout=rows, kh=1, kw=1, stride_h=1, stride_w=1, group=1, has_bias=1, act_type=abi.NOT_ACT, compute=abi.COMPUTE_F32)
    g = torch.Generator(device="cuda").manual_seed(rows + cols)
    x = torch.randn((1, d.cin, 1, cols), generator=g, device="cuda")
    table = torch.randn(8192, generator=g, device="cuda")
    if kind == "w8a32":
        d.input_scale = 0.02
        w = hip.pack_conv_weights_w8(d, torch.randint(-127, 128, (rows, d.cin, 1, 1), generator=g, device="cuda", dtype=torch.int8))
        b, aux = torch.randint(-999, 999, (rows,), generator=g, device="cuda", dtype=torch.int32), torch.rand(rows, generator=g, device="cuda") * 5
        run = lambda: hip.conv2d_w8a32(d, x, w, b, aux, table, packed=True)   # noqa: E731
    else:
        w, b = torch.randn((rows, d.cin, 1, 1), generator=g, device="cuda"), torch.randn(rows, generator=g, device="cuda")
        r = torch.randn((1, rows, 1, cols), generator=g, device="cuda")
        run = lambda: hip.conv2d_f32(d, x, w, b, table) if kind == "f32" else hip.conv2d_f32_add(d, x, w, r, b, table)   # noqa: E731
    y = hip.conv2d_f32(d, x, w, b) if kind == "add" else run()
    d.act_type = abi.SILU
    ref = through_table(torch, y, table)
    assert bool((y < -8).any()) and bool((y > 8).any()) or cols < 100
    assert torch.equal(run(), ref + r if kind == "add" else ref)
    ran = hip.last_launch_choice()
    assert f"{ran[0]}x{ran[1]}" == tile.removesuffix("x2") and (ran[2] == 2) == tile.endswith("x2"), ran


@pytest.mark.parametrize("tiles", [40, 257], ids=["alone", "several a unit"])
@pytest.mark.parametrize("tile", ["128x128", "128x64", "64x128", "64x64"])
@pytest.mark.parametrize("kind,cin", [("w8a32", 64), ("w8a32", 128), ("bf16", 32), ("bf16", 64)])
def test_table_of_the_direct_to_lds_kernel(kind, cin, tile, tiles, monkeypatch):
    """stages of 64 and of 128 bytes; the table in LDS of its own with up to 256 workgroups, in the ring's memory with more, where the per-row
    constants move out of it"""
    import torch
    hip.init(0)
    print("table, direct to LDS", kind, cin, tile, tiles, flush=True)
    monkeypatch.setenv("ONHIP_TILE", tile + "x1x0x0x0x1")
    bm, bn = map(int, tile.split("x"))
    d = ConvDesc(n=1, cin=cin, h=1, w=(tiles - 1) * bn + 5, cout=bm - 3, kh=1, kw=1, stride_h=1, stride_w=1, group=1, has_bias=1, act_type=abi.NOT_ACT,
                 compute=abi.COMPUTE_F32)
    g = torch.Generator(device="cuda").manual_seed(cin + tiles)
    x, table = torch.randn((1, cin, 1, d.w), generator=g, device="cuda"), torch.randn(8192, generator=g, device="cuda")
    if kind == "w8a32":
        d.input_scale = 0.02
        w = hip.pack_conv_weights_w8(d, torch.randint(-127, 128, (d.cout, cin, 1, 1), generator=g, device="cuda", dtype=torch.int8))
        b, aux = torch.randint(-999, 999, (d.cout,), generator=g, device="cuda", dtype=torch.int32), torch.rand(d.cout, generator=g, device="cuda")
        run = lambda: hip.conv2d_w8a32(d, x, w, b, aux, table, packed=True)   # noqa: E731
    else:
        d.compute = abi.COMPUTE_BF16
        xh, w = hip.h16_from_nchw(x, d.compute), hip.h16_pack_conv_weights(d, torch.randn((d.cout, cin, 1, 1), generator=g, device="cuda"))
        b = torch.randn(d.cout, generator=g, device="cuda")
        run = lambda: hip.conv2d_h16(d, xh, w, b, table, y_kind=hip.H16_OUT_F32_NCHW)   # noqa: E731
    y = run()
    d.act_type = abi.SILU
    assert torch.equal(run(), through_table(torch, y, table)) and bool((y < -8.0).any()) and bool((y > 8.0).any())
    assert tuple(hip.last_launch_choice()) == (bm, bn, 1, 0, 0, 0, 1)
