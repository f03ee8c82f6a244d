"""Gemm over the rows of a batch: both kernels of gemm_nt.hip and the sizes at which they hand over, against 64-bit sums.  Bound: a chain of
K fp32 multiply-adds in any order and the bias, (K + 1) 2^-24 (sum |a w| + |bias|)."""
import pytest

from onenew_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    hip.init(0)
    return torch


# (rows, K, columns): every row count the vector kernel is compiled for and the ones between, K below a wavefront's share, past two turns of
# it and off four; the matrix kernel's tiles with one row or column over, K below a step, past its ring; more workgroups than it takes
SHAPES = [(1, 2048, 1000), (1, 3, 1), (2, 260, 5), (3, 2052, 7), (4, 1027, 33), (5, 4096, 6), (8, 1280, 1000), (8, 31, 9), (7, 6148, 4),
          (9, 4, 16), (9, 2048, 17), (16, 36, 1), (17, 2052, 130), (32, 2048, 1000), (63, 192, 31), (64, 1280, 1000), (97, 64, 1000), (33, 2049, 20)]


@pytest.mark.parametrize("special", [False, True], ids=["finite", "special"])
@pytest.mark.parametrize("shape", SHAPES, ids=[str(s) for s in SHAPES])
def test_gemm_rows(shape, special, torch_dev):
    torch = torch_dev
    m, k, n = shape
    print("gemm", shape, special, flush=True)
    g = torch.Generator().manual_seed(m * 131 + k + n)
    a, w, b = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g), torch.randn(n, generator=g)
    if special:   # one row and one column that are not finite: their neighbours stay as they are
        a[m - 1, k - 1], w[n - 1, 0] = float("nan"), float("inf")
    y = hip.gemm_f32(a.cuda(), w.cuda(), b.cuda()).cpu().double()
    a, w, b = a.double(), w.double(), b.double()
    ref, bound = a @ w.T + b, (k + 1) * 2.0 ** -24 * (a.abs() @ w.abs().T + b.abs())
    if special:
        assert bool(y[m - 1].isnan().all()) and not bool(y[:, n - 1].isfinite().any())
        y, ref, bound = y[:m - 1, :n - 1], ref[:m - 1, :n - 1], bound[:m - 1, :n - 1]
    assert bool(((y - ref).abs() <= bound).all())


@pytest.mark.parametrize("m", [3, 20])
def test_gemm_operands_off_sixteen_bytes(m, torch_dev):
    """operands at four-byte addresses: no 16-byte loads of them"""
    torch = torch_dev
    g = torch.Generator().manual_seed(m)
    a, w, b = torch.randn(m * 64 + 1, generator=g).cuda()[1:].view(m, 64), torch.randn(19 * 64 + 1, generator=g).cuda()[1:].view(19, 64), torch.randn(19, generator=g).cuda()
    y = hip.gemm_f32(a, w, b).double()
    bound = 65 * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T + b.double().abs())
    assert bool(((y - (a.double() @ w.double().T + b.double())).abs() <= bound).all())


@pytest.mark.parametrize("m,k,n,tiled", [(16, 25088, 512, True), (64, 4096, 512, True), (16, 8192, 2048, True), (17, 1028, 5000, True), (16, 4096, 4096, False), (21, 2544, 1641, False), (46, 1796, 311, False), (130, 2100, 28, False), (68, 3752, 642, False),
                                         (48, 2048, 1000, False), (9, 2048, 1000, False), (64, 192, 1000, False)])
def test_gemm_hand_over(m, k, n, tiled, torch_dev):
    """a K that the tiled kernels are faster on, cut into slices, goes there (they leave a launch choice, the kernels of a batch's rows do not)"""
    torch = torch_dev
    x, filt = torch.randn(1, 8, 4, 4, device="cuda"), torch.randn(4, 8, 1, 1, device="cuda")
    hip.conv2d_f32(hip.ConvDesc(n=1, cin=8, h=4, w=4, cout=4, kh=1, kw=1, stride_h=1, stride_w=1, group=1), x, filt)
    before = hip.last_launch_choice()
    a, w, b = torch.randn(m, k, device="cuda"), torch.randn(n, k, device="cuda"), torch.randn(n, device="cuda")
    y = hip.gemm_f32(a, w, b).double()
    bound = (k + 1) * 2.0 ** -24 * (a.abs().double() @ w.abs().double().T + b.abs().double())
    assert bool(((y - (a.double() @ w.double().T + b.double())).abs() <= bound).all())
    assert (hip.last_launch_choice() != before) == tiled
