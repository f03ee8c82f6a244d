"""The one-launch kernel for a convolution and the 1x1 convolution over its result on the 16-bit matrix cores (igemm_f3_pw.hip), which
the Conv plugin runs on weights that stay as they are: against the oracle's operator chain, against 64-bit sums with the bound of the fp32
kernels, and on operands that are not finite or out of the split form's range against the fp32 kernel."""
import numpy as np
import pytest

from onenew_amd import abi, hip, ops
from test_gpu_conv_pw import SHAPES, close, descs, dev, operands

pytestmark = pytest.mark.gpu
N, R, CL = abi.NOT_ACT, abi.RELU, abi.CLIP


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    hip.init(0)
    return torch


def plugin_pair(a, b, wa, ba, wb, bb):
    return ops.ConvPair(ops.Plugin(hip.plugin_path("Conv")), (a, b), (wa, wb), (ba, bb))


# SHAPES: tiles and steps that are not full in every direction; here one row, one and two steps of the second reduction, its last row alone
MORE = [(1, 4, 1, 9, 9, 1, 3, 1, 1, R, N, True, True), (1, 8, 16, 11, 13, 32, 3, 1, 1, R, R, True, False),
        (2, 12, 17, 8, 8, 65, 3, 1, 1, N, CL, False, False), (1, 16, 64, 17, 19, 129, 3, 2, 1, R, N, True, True)]


@pytest.mark.parametrize("shape", SHAPES + MORE)
def test_pair_on_kept_weights(shape, torch_dev, oracle):
    n, cin, cmid, h, w, cout, k, s, p, act_a, act_b, with_res, relu = shape
    print(f"conv + 1x1, split {shape}", flush=True)
    a, b = descs(n, cin, cmid, h, w, cout, k, s, p, act_a, act_b)
    x, wa, ba, wb, bb = operands(f"convpw_split{shape}", a, b)
    oh, ow = a.out_hw()
    res = np.random.default_rng(7).standard_normal((n, cout, oh, ow), dtype=np.float32) if with_res else None
    y = plugin_pair(a, b, wa, ba, wb, bb)(x, addend=res, relu=relu).copy()
    ref = oracle.conv2d_f32(b, oracle.conv2d_f32(a, x, wa, ba), wb, bb).astype(np.float64)
    if with_res:
        ref = np.maximum(ref + res, 0.0) if relu else ref + res
    close(y, ref)


@pytest.mark.parametrize("values", ["normal", "uneven", "spread"])
def test_error_against_64_bits_is_that_of_the_fp32_kernel(values, torch_dev):
    """the first stage of ResNet-50: the split form is no further from 64-bit sums than fp32 matrix instructions; operands spread over 2^+-4, and
    over 2^+-24, where a term decides a sum and its own rounding the error (as in test_gpu_f3)"""
    torch = torch_dev
    a, b = descs(2, 64, 64, 56, 56, 256, 3, 1, 1, R, N)
    x, wa, ba, wb, bb = operands("convpw_split_error", a, b)
    if values != "normal":
        rng, e = np.random.default_rng(11), 4 if values == "uneven" else 24
        x, wa, wb = (v * np.exp2(rng.uniform(-e, e, v.shape)).astype(np.float32) for v in (x, wa, wb))
    y = torch.from_numpy(plugin_pair(a, b, wa, ba, wb, bb)(x).copy()).double()
    plain = hip.conv2d_pw_f32(a, b, dev(torch, x), hip.pack_conv_weights(a, dev(torch, wa)), dev(torch, ba), hip.conv2d_pw_pack_weights(b, dev(torch, wb)),
                              dev(torch, bb)).cpu().double()
    t = lambda v: torch.from_numpy(v).double()   # noqa: E731
    conv = lambda f: torch.nn.functional.conv2d(torch.relu(torch.nn.functional.conv2d(f(t(x)), f(t(wa)), f(t(ba)), padding=1)), f(t(wb)), f(t(bb)))   # noqa: E731
    ref, magnitude = conv(lambda v: v), conv(torch.abs)
    # spread operands: a share of the magnitudes, element by element (a norm would be the largest sums' error alone)
    err = lambda v: float((v - ref).norm() / ref.norm()) if values == "normal" else float(((v - ref) / magnitude).square().mean().sqrt())   # noqa: E731
    print(f"conv + 1x1, error of {values} values: split {err(y):.3e}, fp32 {err(plain):.3e}, ratio {err(y) / err(plain):.3f}", flush=True)
    assert not torch.equal(y, plain)   # it is the other kernel
    assert err(y) <= (1.25 if values == "spread" else 1.02) * err(plain)


@pytest.mark.parametrize("what", ["input", "weights", "large", "middle"])
def test_operands_without_finite_parts(what, torch_dev):
    """infinities, NaN and values of 2^104 and more in either product: what the fp32 kernel gives, in every element"""
    torch = torch_dev
    a, b = descs(1, 8, 40, 10, 13, 70, 3, 1, 1, N, N)
    x, wa, ba, wb, bb = operands("convpw_split_range", a, b)
    if what == "input":
        x[0, 2, 3, 4], x[0, 5, 8, 8] = np.inf, np.nan
    elif what == "weights":
        wb[3, 7, 0, 0], wb[69, 1, 0, 0] = np.nan, -np.inf
    elif what == "large":
        x *= np.float32(2.0 ** 100)
        wb *= np.float32(2.0 ** -60)
    else:
        ba[5] = np.float32(2.0 ** 110)   # one row of the first result leaves the range, its products do not overflow
    y = torch.from_numpy(plugin_pair(a, b, wa, ba, wb, bb)(x).copy())
    plain = hip.conv2d_pw_f32(a, b, dev(torch, x), hip.pack_conv_weights(a, dev(torch, wa)), dev(torch, ba), hip.conv2d_pw_pack_weights(b, dev(torch, wb)),
                              dev(torch, bb)).cpu()
    assert torch.equal(y.isnan(), plain.isnan()) and torch.equal(y.isinf(), plain.isinf())
    ok = plain.isfinite()
    assert bool(ok.any()) and torch.equal(y[plain.isinf()], plain[plain.isinf()])
    # both sum at most 72 and 40 products in fp32: 112 roundings of the sum of magnitudes
    scale = plain[ok].abs().max().double()
    assert float((y[ok].double() - plain[ok].double()).abs().max()) <= 112 * 2.0 ** -24 * float(scale) * 8


def test_split_weights_out_of_reach(torch_dev):
    """more rows of the second product than the split form's 32-bit offsets reach, fewer than the fp32 one's: the fp32 kernel runs"""
    torch = torch_dev
    rows, mid = 2_800_001, 64
    print(f"conv + 1x1, {rows} rows of the second product", flush=True)
    a, b = descs(1, 4, mid, 1, 2, rows, 3, 1, 1, R, N)
    x, wa, ba, _, _ = operands("convpw_split_rows", a, descs(1, 4, mid, 1, 2, 1, 3, 1, 1, R, N)[1])
    g = torch.Generator(device="cuda").manual_seed(3)
    wb, bb = torch.randn((rows, mid, 1, 1), generator=g, device="cuda"), torch.randn(rows, generator=g, device="cuda")
    y = plugin_pair(a, b, wa, ba, wb.cpu().numpy(), bb.cpu().numpy())(x)
    t = lambda v: torch.from_numpy(v).double()   # noqa: E731
    conv = lambda f: torch.nn.functional.conv2d(f(t(x)), f(t(wa)), f(t(ba)), padding=1).view(mid, 2).cuda()   # noqa: E731
    product = lambda f, m: f(wb.view(rows, mid).double()) @ m + f(bb.double())[:, None]   # noqa: E731
    ref, magnitude = product(lambda v: v, torch.relu(conv(lambda v: v))), product(torch.abs, conv(torch.abs))
    got = torch.from_numpy(y).cuda().view(rows, 2).double()
    # 36 and 64 products and a bias each: at most 102 roundings to fp32 of what the magnitudes add up to
    assert bool(((got - ref).abs() <= 102 * 2.0 ** -24 * magnitude).all())


@pytest.mark.parametrize("n,cin,cmid,hw,split", [(1, 4, 24, 40, False), (1, 4, 24, 128, False), (2, 4, 24, 93, True), (1, 8, 8, 40, True)])
def test_choice(n, cin, cmid, hw, split, torch_dev):
    """a short first reduction in one round of workgroups stays with fp32 matrix instructions: the bits of the fp32 kernel"""
    torch = torch_dev
    a, b = descs(n, cin, cmid, hw, hw, 16, 3, 1, 1, R, N)
    x, wa, ba, wb, bb = operands("convpw_split_choice", a, b)
    y = torch.from_numpy(plugin_pair(a, b, wa, ba, wb, bb)(x).copy())
    plain = hip.conv2d_pw_f32(a, b, dev(torch, x), hip.pack_conv_weights(a, dev(torch, wa)), dev(torch, ba), hip.conv2d_pw_pack_weights(b, dev(torch, wb)),
                              dev(torch, bb)).cpu()
    assert torch.equal(y, plain) != split
