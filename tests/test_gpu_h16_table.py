"""Table activations stored in 16 bits (table_h16): bit for bit the rounding of the same layer's fp32 result, whose table is read by other code, on
every tile of the direct-to-LDS kernel, at both ends of the table and beyond, on its entries' edges, at infinities and NaN, with the last tile's
channels beyond the result zero."""
import pytest

from onenew_amd import abi, hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("compute", [abi.COMPUTE_BF16, abi.COMPUTE_F16])
@pytest.mark.parametrize("tile", ["128x128", "128x64", "64x128", "64x64"])
def test_stored_rounding(tile, compute, monkeypatch):
    import torch
    hip.init(0)
    print(tile, compute, flush=True)
    rows, k, cols = 1030, 96, 170   # 170 columns: a last tile of 42 of 64 or 128, in a row of 192
    x = torch.zeros((rows, k))
    x[:, 0] = torch.arange(rows) / 64 - 8.04   # from below the table to above it, rounded; the columns' biases reach every entry's edge
    x[3, 0], x[4, 0], x[5, 0], x[6, 0], x[7, 0] = float("inf"), float("-inf"), float("nan"), 300.0, -300.0
    x[:, 1] = torch.randn(rows, generator=torch.Generator().manual_seed(1)) * 5
    b = torch.arange(cols).float() / 512 * (8 / 3) - 0.3
    w = torch.zeros((k, cols))
    w[0], w[1, ::3] = 1.0, 1.0
    t = torch.arange(8192, dtype=torch.float64) / 512 - 8
    t = (t * 0.5 * (1 + torch.erf(t / 2 ** 0.5))).float().cuda()
    x, w, b = hip.h16_from_rows(x.cuda(), compute), hip.h16_pack_matmul_weights(w.cuda(), compute), b.cuda()
    monkeypatch.setenv("ONHIP_TILE", tile + "x1x0x0x0x1")
    y = hip.linear_h16(x, w, k, cols, compute, bias=b, gelu_lut=t)
    assert list(hip.last_launch_choice()[:2]) == [int(v) for v in tile.split("x")]
    whole = hip.linear_h16(x, w, k, cols, compute, bias=b, gelu_lut=t, y_kind=hip.H16_OUT_F32_NHWC)
    torch.cuda.synchronize()
    assert torch.equal(y[:, :cols].view(torch.int16), whole.to(y.dtype).view(torch.int16))
    assert not y[:, cols:].view(torch.int16).any()
