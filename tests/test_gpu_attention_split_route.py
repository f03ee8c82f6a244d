"""fp32 attention on the 16-bit matrix cores (attention_f3.hip: head dimension 64, more than 64 tokens, more 64-query workgroups than compute units)
against 64-bit arithmetic: sizes at the edges of its tiles of 32 keys, of its workgroups of 128 and 256 queries and of its two widths, strides
of a projection's output and of tensors of their own, scores of every size: which calls run on it, and
bounds on each element that a lost partial product does not meet.

Which kernel a call ran on shows in its bits: the same heads in calls of at most one workgroup a compute unit run on fp32 matrix instructions
(attention.hip), whose sums are others."""
import pytest

from onenew_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    hip.init(0)
    return torch


def reference(torch, q, k, v, scale):
    """the result, the sum of its terms' absolute values and of a score's, in 64 bits"""
    q, k, v = (x.double().contiguous() for x in (q, k, v))
    p = torch.softmax(torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale, -1)
    top = torch.matmul(q.abs(), k.abs().transpose(-1, -2).contiguous()).amax(-1, keepdim=True) * scale
    return torch.matmul(p, v), torch.matmul(p, v.abs()), top


def on_fp32_instructions(torch, q, k, v, scale):
    """the same heads, some images at a time"""
    b, h, t, _ = q.shape
    step = max(1, 256 // (h * ((t + 63) // 64)))
    assert step * h * ((t + 63) // 64) <= 256
    return torch.cat([hip.attention(q[i:i + step], k[i:i + step], v[i:i + step], scale=scale, merged_out=False) for i in range(0, b, step)])


def operands(torch, b, h, t, std, seed=0):
    g = torch.Generator(device="cuda").manual_seed(1000 * t + 10 * h + seed)
    qkv = torch.randn((b, t, 3, h, 64), generator=g, device="cuda") * std
    return [qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3)]


@pytest.mark.parametrize("b,h,t", [(130, 1, 65), (45, 3, 65), (129, 1, 95), (130, 1, 96), (130, 1, 97), (130, 1, 127), (65, 2, 128), (30, 3, 129), (43, 3, 129), (43, 3, 160), (65, 1, 193), (65, 1, 196),
                                   (64, 3, 196), (90, 1, 196), (43, 3, 224), (43, 3, 225), (65, 1, 255), (65, 1, 256), (128, 1, 256)])
@pytest.mark.parametrize("std", [1.0, 3.0])
def test_attention_against_64_bits(b, h, t, std, torch_dev):
    torch = torch_dev
    print(f"attention {b} x {h} heads, {t} tokens", flush=True)
    q, k, v = operands(torch, b, h, t, std)
    ref, mass, top = reference(torch, q, k, v, 0.125)
    out = hip.attention(q, k, v, scale=0.125, merged_out=False)
    out2 = hip.attention(q.contiguous(), k.contiguous(), v.contiguous(), scale=0.125, merged_out=False)
    merged = hip.attention(q, k, v, scale=0.125)
    other = on_fp32_instructions(torch, q, k, v, 0.125)
    torch.cuda.synchronize()
    assert torch.equal(out, out2) and torch.equal(merged, out.permute(0, 2, 1, 3).reshape(b, t, 64 * h))
    assert not torch.equal(out, other)
    # a score: 64 products and their fp32 additions, three partial products left out of each (2^-23 of it together), and what the exponential adds (its
    # argument's rounding and two units); once in the weight and once in the sum of t of them; then t products and additions of the second product
    score = ((68 * top + 16) + t) * 2.0 ** -24
    assert bool(((out.double() - ref).abs() <= (2 * score + (t + 8) * 2.0 ** -24) * mass).all())
    # no further off than with fp32 matrix instructions (0.71-0.91 measured; one of the six partial products less is 10 times as far)
    error = lambda y: float((y.double() - ref).norm() / ref.norm())  # noqa: E731
    assert error(out) <= error(other), (error(out), error(other))


@pytest.mark.parametrize("b,h,t", [(260, 1, 64), (768, 1, 64), (300, 2, 33), (520, 1, 16), (600, 1, 1), (130, 2, 5), (260, 1, 31), (90, 3, 32), (260, 1, 33), (90, 3, 63), (64, 4, 33), (64, 2, 65), (32, 2, 200), (60, 1, 196), (64, 1, 256)])
def test_calls_for_fp32_instructions(b, h, t, torch_dev):
    """up to 64 tokens, and up to one workgroup a compute unit"""
    torch = torch_dev
    print(f"attention {b} x {h} heads, {t} tokens", flush=True)
    q, k, v = operands(torch, b, h, t, 1.0)
    out = hip.attention(q, k, v, scale=0.125, merged_out=False)
    other = on_fp32_instructions(torch, q, k, v, 0.125)
    assert torch.equal(out, other)
    ref = reference(torch, q, k, v, 0.125)[0]
    assert float((out.double() - ref).norm() / ref.norm()) <= 1e-6


@pytest.mark.parametrize("t", [72, 196, 256])
def test_scores_that_grow_from_tile_to_tile(t, torch_dev):
    """the largest score moves on by hundreds with every tile of keys, or stands in the first one"""
    torch = torch_dev
    b = 260
    print(f"growing scores, {t} tokens", flush=True)
    for order in (1, -1):
        q, k, v = operands(torch, b, 1, t, 1.0, seed=order)
        ramp = torch.arange(t, device="cuda", dtype=torch.float32)
        ramp = ramp if order == 1 else ramp.flip(0)
        q = q.contiguous()
        q[..., 0] = 8.0
        k = k.contiguous()
        k[..., 0] = ramp * 10.0
        ref = reference(torch, q, k, v, 1.0)[0]
        out = hip.attention(q, k, v, scale=1.0, merged_out=False)
        other = on_fp32_instructions(torch, q, k, v, 1.0)
        torch.cuda.synchronize()
        assert not torch.equal(out, other)
        # scores of up to 20000 are 2^-24 of that off, 1e-3, and so is a probability
        assert (out.double() - ref).abs().max() <= 5e-3 * ref.abs().max()
