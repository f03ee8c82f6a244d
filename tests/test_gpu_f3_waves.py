"""fp32 on the 16-bit matrix cores, the tile of 192 x 64 on either side of one workgroup a compute unit, where it takes twelve wavefronts instead of four:
the bits of the 64 x 64 tile, whose wavefronts are the same everywhere, and of each other.  Rows, 1x1 and 3x3 convolutions, with an addend, a table
activation, ragged rows and columns, slices of K."""
import pytest

from onenew_amd import abi, hip
from onenew_amd.abi import ConvDesc

pytestmark = pytest.mark.gpu


def table(torch):
    x = torch.arange(8192, dtype=torch.float64) / 512 - 8
    return (x * 0.5 * (1 + torch.erf(x / 2 ** 0.5))).float().cuda()


def both(tile, other, run, monkeypatch, torch):
    got = []
    for t in (tile, other):
        monkeypatch.setenv("ONHIP_TILE", t)
        got.append(run())
        assert list(hip.last_launch_choice()[:2]) == [int(v) for v in t.split("x")[:2]] and hip.last_launch_choice()[4] == 2
    torch.cuda.synchronize()
    assert torch.equal(got[0].view(torch.int32), got[1].view(torch.int32))


# (tiles of a product cannot be asked for; the model takes it for the first three and others for the rest)
@pytest.mark.parametrize("rows,k,n", [(12544, 192, 192), (12481, 767, 187), (16384, 200, 190), (6272, 1024, 250), (17000, 520, 187), (33000, 192, 192)])
def test_product(rows, k, n):
    import torch
    hip.init(0)
    g = torch.Generator(device="cuda").manual_seed(rows + k)
    a, b, bias = torch.randn((rows, k), generator=g, device="cuda"), torch.randn((k, n), generator=g, device="cuda") / k ** 0.5, torch.randn(n, generator=g, device="cuda")
    add = torch.randn((rows, n), generator=g, device="cuda")
    ref, mass = torch.matmul(a.double(), b.double()) + bias, torch.matmul(a.abs().double(), b.abs().double()) + bias.abs()
    # a chain of fp32 multiply-adds, what the left-out partial products can reach, the roundings of the bias and the result (and of the addend's sum)
    bound = mass * ((k + 4) * 2.0 ** -24 + 2.0 ** -23)
    y = hip.matmul(a, b, bias=bias)
    plain = list(hip.last_launch_choice())
    print(rows, k, n, plain, flush=True)
    assert bool(((y.double() - ref).abs() <= bound).all())
    z = hip.matmul(a, b, bias=bias, addend=add)
    if list(hip.last_launch_choice()) == plain:   # a choice of its own, so perhaps other sums
        assert torch.equal(z, y + add)
    else:
        assert bool(((z.double() - ref - add).abs() <= bound + 2.0 ** -23 * add.abs()).all())
    t = table(torch)
    i = ((y + 8.0) * 512.0).to(torch.int32).clamp(0, 8191)
    z = hip.matmul(a, b, bias=bias, gelu_lut=t)
    assert list(hip.last_launch_choice()) == plain and torch.equal(z, torch.where(y < -8.0, 0.0, torch.where(y >= 8.0, y, t[i.long()])))


# Tiles of a product cannot be asked for: with the one that the model takes.  192 x 64 in twelve wavefronts up to 16384 rows and in four above, then others.
@pytest.mark.parametrize("rows,k,n,tile", [(12544, 192, 192, (192, 64)), (12481, 767, 187, (192, 64)), (16384, 200, 190, (192, 64)), (33000, 520, 187, (192, 64)),
                                           (32961, 768, 192, (192, 64)), (6272, 1024, 250, None), (17000, 520, 187, (64, 64)), (33000, 192, 192, (64, 64))])
def test_product_tiles(rows, k, n, tile):
    import torch
    hip.init(0)
    g = torch.Generator(device="cuda").manual_seed(rows + k)
    a, b, bias = torch.randn((rows, k), generator=g, device="cuda"), torch.randn((k, n), generator=g, device="cuda") / k ** 0.5, torch.randn(n, generator=g, device="cuda")
    add = torch.randn((rows, n), generator=g, device="cuda")
    ref, mass = torch.matmul(a.double(), b.double()) + bias, torch.matmul(a.abs().double(), b.abs().double()) + bias.abs()
    # a chain of fp32 multiply-adds, what the left-out partial products can reach, the roundings of the bias and the result (and of the addend's sum)
    bound = mass * ((k + 4) * 2.0 ** -24 + 2.0 ** -23)
    y = hip.matmul(a, b, bias=bias)
    plain = list(hip.last_launch_choice())
    print(rows, k, n, plain, flush=True)
    assert plain[4] == 2 and (tile is None or tuple(plain[:2]) == tile)
    assert bool(((y.double() - ref).abs() <= bound).all())
    if rows > 16384:   # the first rows alone, in twelve wavefronts: the same products in the same order
        part = hip.matmul(a[:12481], b, bias=bias)
        assert tuple(hip.last_launch_choice()[:2]) == (192, 64) and hip.last_launch_choice()[4] == 2
        assert torch.equal(y[:12481].view(torch.int32), part.view(torch.int32))
    z = hip.matmul(a, b, bias=bias, addend=add)
    assert tile != (192, 64) or list(hip.last_launch_choice()) == plain
    if list(hip.last_launch_choice()) == plain:   # a choice of its own, so perhaps other sums
        assert torch.equal(z, y + add)
    else:
        assert bool(((z.double() - ref - add).abs() <= bound + 2.0 ** -23 * add.abs()).all())
    t = table(torch)
    i = ((y + 8.0) * 512.0).to(torch.int32).clamp(0, 8191)
    z = hip.matmul(a, b, bias=bias, gelu_lut=t)
    assert list(hip.last_launch_choice()) == plain and torch.equal(z, torch.where(y < -8.0, 0.0, torch.where(y >= 8.0, y, t[i.long()])))


@pytest.mark.parametrize("cin,k,hw,split", [(40, 1, 63, 1), (513, 1, 64, 1), (60, 3, 62, 1), (60, 3, 66, 1), (520, 1, 30, 3)])
def test_convolution(cin, k, hw, split, monkeypatch):
    import torch
    hip.init(0)
    n, cout, tile = 4, 185, "192x64"
    print(f"{n} x {cin} x {hw}^2 -> {cout}, filter {k}, {tile} in {split}", flush=True)
    d = ConvDesc(n=n, cin=cin, h=hw, w=hw, cout=cout, kh=k, kw=k, stride_h=1, stride_w=1, pad_t=k // 2, pad_l=k // 2, pad_b=k // 2, pad_r=k // 2, group=1,
                 has_bias=1, act_type=abi.NOT_ACT, compute=abi.COMPUTE_F32)
    g = torch.Generator(device="cuda").manual_seed(cin + hw)
    x, w, bias = torch.randn((n, cin, hw, hw), generator=g, device="cuda"), torch.randn((cout, cin, k, k), generator=g, device="cuda") / (cin * k * k) ** 0.5, torch.randn(cout, generator=g, device="cuda")
    x[0, 1, 2, 3] = float("inf")
    add = torch.randn((n, cout, hw, hw), generator=g, device="cuda")
    both(f"{tile}x{split}x0x2", f"64x64x{split}x0x2", lambda: hip.conv2d_f32(d, x, w, bias), monkeypatch, torch)
    both(f"{tile}x{split}x0x2", f"64x64x{split}x0x2", lambda: hip.conv2d_f32_add(d, x, w, add, bias, relu=True), monkeypatch, torch)
