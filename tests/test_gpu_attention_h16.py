"""16-bit attention against float64 on the same operands: tokens at the edges of a tile of 32 keys, of a workgroup's queries and of each size the kernel is
built for, one copy of k and v a head and several, scales of either sign and zero, a result with a pitch; values near the type's largest, infinities and NaN."""
import numpy as np
import pytest

from onenew_amd import hip

pytestmark = pytest.mark.gpu

SHAPES = [(2, 3, 1, 0.125), (5, 2, 31, -0.5), (1, 3, 32, 0.125), (2, 2, 33, 1.0), (1, 1, 64, 0.0), (64, 3, 65, 0.125), (2, 3, 128, -0.125), (50, 3, 129, 0.125),
          (2, 3, 197, 0.125), (64, 3, 197, -0.25), (1, 5, 224, 0.125), (3, 1, 225, 0.125), (48, 3, 225, 0.125), (43, 3, 256, 0.125), (1, 3, 256, 0.0)]


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("b,h,t,scale", SHAPES)
def test_error(b, h, t, scale, dtype):
    import torch
    hip.init(0)
    tdt = getattr(torch, dtype)
    print(f"{b} x {h} heads of {t} tokens, scale {scale}, {dtype}", flush=True)
    g = torch.Generator().manual_seed(t * 100 + b)
    qkv = torch.randn((b, t, 3, h, 64), generator=g).to(tdt)
    dev = qkv.cuda()
    out = torch.full((b, t, h * 64 + 8), 7.0, dtype=tdt, device="cuda")
    hip.attention(*(dev[:, :, i].permute(0, 2, 1, 3) for i in range(3)), scale=scale, out=out)
    torch.cuda.synchronize()
    assert bool((out[..., h * 64:] == 7.0).all())
    got = out[..., :h * 64].double().cpu().reshape(b, t, h, 64).permute(0, 2, 1, 3)
    q, k, v = (qkv[:, :, i].permute(0, 2, 1, 3).double().contiguous() for i in range(3))
    p = torch.softmax(torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale, -1)
    ref, mass = torch.matmul(p, v), torch.matmul(p, v.abs())
    # a half unit of the type for each rounded probability and for the result, 2^-25 where they are below f16's normal numbers; the scores' 64 fp32 additions
    # and what the exponential adds (its argument's rounding and two units), once in the weight and once in the sum
    u, tiny = (2.0 ** -8, 0.0) if dtype == "bfloat16" else (2.0 ** -11, 2.0 ** -25)
    top = float(torch.matmul(q.abs(), k.abs().transpose(-1, -2).contiguous()).max()) * abs(scale)
    score = 2 * (66 * top + 16 + t) * 2.0 ** -24
    bound = u * ref.abs() + (u + score) * (1 + u) * mass + tiny * (1 + v.abs().sum(-2, keepdim=True))
    assert bool(((got - ref).abs() <= bound).all()), float(((got - ref).abs() / bound).max())


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
def test_far_values(dtype):
    import torch
    hip.init(0)
    tdt = getattr(torch, dtype)
    print(dtype, flush=True)
    t, big = 256, float(torch.finfo(tdt).max) * 0.98
    q, k = torch.zeros((2, 1, 1, t, 64), dtype=tdt, device="cuda")
    k[0, 0, 7, 0] = 1.0
    v = torch.full((1, 1, t, 64), big, dtype=tdt, device="cuda")
    run = lambda: hip.attention(q, k, v, merged_out=False)[0, 0].float().cpu().numpy()  # noqa: E731
    assert np.allclose(run(), big, rtol=1e-2), "the mean of values near the largest"
    v.zero_()
    v[0, 0, :, 0] = 1.0
    v[0, 0, 9, 3], v[0, 0, 9, 4], v[0, 0, 200, 5] = float("inf"), float("-inf"), float("nan")
    y = run()
    assert np.allclose(y[:, 0], 1.0, rtol=1e-2) and (y[:, 3] == np.inf).all() and (y[:, 4] == -np.inf).all() and np.isnan(y[:, 5]).all() and not y[:, 6:].any()
    v.zero_()
    v[0, 0, :, 0] = 1.0
    q[0, 0, 3, 0], q[0, 0, 4, 0], q[0, 0, 5, 0] = float("nan"), 200.0, -200.0   # a row of its own each
    v[0, 0, 7, 1] = 2.0
    y = run()
    assert np.isnan(y[3]).all() and np.allclose(y[4, :2], [1.0, 2.0], rtol=1e-2) and np.allclose(y[5, :2], [1.0, 0.0], rtol=1e-2)
    assert np.isfinite(np.delete(y, 3, 0)).all() and np.allclose(np.delete(y, 3, 0)[:, 0], 1.0, rtol=1e-2)
