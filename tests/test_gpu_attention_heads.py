"""16-bit attention with enough heads for one workgroup each (eight wavefronts on one copy of k and v): token counts at the
edges of the 32-query and 32-key tiles against a float64 model, 1.5 units in the last place of the type."""
import pytest

from onenew_amd import hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("b,h,t", [(43, 3, 129), (32, 4, 161), (11, 12, 193), (64, 2, 224), (128, 1, 225), (33, 4, 256)])
def test_one_workgroup_per_head(b, h, t, dtype):
    import torch
    hip.init(0)
    print(f"attention {dtype} {b} x {h} heads, {t} tokens", flush=True)
    dt = getattr(torch, dtype)
    qkv = torch.randn(b, t, 3, h, 64, generator=torch.Generator().manual_seed(t)).cuda().to(dt)
    q, k, v = (qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3))
    got = hip.attention(q, k, v, scale=0.125).double()
    torch.cuda.synchronize()
    q, k, v = (x.double().contiguous() for x in (q, k, v))
    pr = torch.softmax(torch.matmul(q, k.transpose(-1, -2).contiguous()) * 0.125, -1).to(dt).double()
    ref = torch.matmul(pr, v).permute(0, 2, 1, 3).reshape(b, t, h * 64)
    ulp = 2.0 ** -8 if dtype == "bfloat16" else 2.0 ** -11
    assert float((got - ref).abs().max()) <= 1.5 * ulp * float(ref.abs().max()) + 1e-6
