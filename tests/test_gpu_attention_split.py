"""fp32 attention on the 16-bit matrix cores (attention_f3.hip: head dimension 64, more than 64 tokens, more 64-query workgroups than compute
units) and, up to those, on fp32 matrix instructions
against 64-bit arithmetic: sizes at the edges of its tiles of 32 keys, of its workgroups of 128 and 256 queries and of its two widths, strides
of a projection's output and of tensors of their own, scores of every size, operands that are not finite.

Tolerance: sums of up to 256 products with fp32 accumulation err by about 2^-24 sqrt(256) of the terms' spread, and an error d of a
score is one of d in its exponential.  Scores of a spread of 1 to 9 make that 1e-6 to 1e-5 of the result; 4e-5 is stated."""
import pytest

from onenew_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    hip.init(0)
    return torch


def reference(torch, q, k, v, scale):
    q, k, v = (x.double().contiguous() for x in (q, k, v))
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    return torch.matmul(torch.softmax(s, -1), v)


def operands(torch, b, h, t, std, seed=0):
    g = torch.Generator(device="cuda").manual_seed(1000 * t + 10 * h + seed)
    qkv = torch.randn((b, t, 3, h, 64), generator=g, device="cuda") * std
    return [qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3)]


@pytest.mark.parametrize("b,h,t", [(260, 1, 1), (130, 2, 5), (260, 1, 31), (90, 3, 32), (260, 1, 33), (90, 3, 63), (260, 1, 64), (45, 3, 65), (130, 1, 96),
                                   (130, 1, 127), (65, 2, 128), (30, 3, 129), (43, 3, 129), (43, 3, 160), (60, 1, 196), (64, 3, 196), (43, 3, 224), (43, 3, 225),
                                   (65, 1, 255), (65, 1, 256), (128, 1, 256)])
@pytest.mark.parametrize("std", [1.0, 3.0])
def test_attention_against_64_bits(b, h, t, std, torch_dev):
    torch = torch_dev
    print(f"attention {b} x {h} heads, {t} tokens", flush=True)
    q, k, v = operands(torch, b, h, t, std)
    ref = reference(torch, q, k, v, 0.125)
    out = hip.attention(q, k, v, scale=0.125, merged_out=False)
    out2 = hip.attention(q.contiguous(), k.contiguous(), v.contiguous(), scale=0.125, merged_out=False)
    merged = hip.attention(q, k, v, scale=0.125)
    torch.cuda.synchronize()
    assert (out.double() - ref).abs().max() <= 4e-5 * ref.abs().max()
    assert torch.equal(out, out2) and torch.equal(merged, out.permute(0, 2, 1, 3).reshape(b, t, 64 * h))


@pytest.mark.parametrize("t", [40, 196, 256])
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
        ref = reference(torch, q, k, v, 1.0)
        out = hip.attention(q, k, v, scale=1.0, merged_out=False)
        torch.cuda.synchronize()
        # scores of up to 20000 are 2^-24 of that off, 1e-3, and so is a probability
        assert (out.double() - ref).abs().max() <= 5e-3 * ref.abs().max()


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3e38, 2.0 ** 110])
@pytest.mark.parametrize("where", ["q", "k", "v"])
def test_operands_without_finite_parts(value, where, torch_dev):
    """an element that is not finite, or too large for its parts: every other query, head and channel as without it, its own as in fp32"""
    torch = torch_dev
    b, t = 90, 196
    print(f"{value} in {where}", flush=True)
    q, k, v = (x.contiguous() for x in operands(torch, b, 1, t, 1.0))
    clean = hip.attention(q, k, v, scale=0.125, merged_out=False)
    x = {"q": q, "k": k, "v": v}[where]
    x[3, 0, 57, 5] = value
    out = hip.attention(q, k, v, scale=0.125, merged_out=False)
    torch.cuda.synchronize()
    s = torch.matmul(q[3].double(), k[3].double().transpose(-1, -2).contiguous()).float() * 0.125
    ref = torch.matmul(torch.softmax(s, -1).double(), v[3].double()).float()
    others = [i for i in range(b) if i != 3]
    assert torch.equal(out[others], clean[others])
    finite = torch.isfinite(ref)
    assert torch.equal(torch.isnan(out[3]), torch.isnan(ref))
    assert torch.equal(out[3][torch.isinf(ref)], ref[torch.isinf(ref)])
    top = ref[finite].abs().max() if finite.any() else 1.0
    assert ((out[3][finite] - ref[finite]).abs() <= 4e-5 * torch.maximum(ref[finite].abs(), torch.full_like(ref[finite], float(min(top, 10.0))))).all()
