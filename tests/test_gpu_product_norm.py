"""A product with a bias and a skip connection whose result goes into a LayerNormalization: the runtime has the product's call make both tensors,
in one launch where a tile of the product holds whole rows.  The bits of the net run operator by operator."""
import numpy as np
import pytest

from onenew_amd import hip, onefile, rt

pytestmark = pytest.mark.gpu

# (rows, k, n, in one launch): rows that end inside a tile of 64, alone in one, and full; the widest row a tile holds and narrower ones, off 32 and off 16
# columns, in twelve wavefronts up to 16384 rows and in four above; then products that run in another tile, rows that no tile holds (196, 256), of three columns more than a multiple of four, and few rows, where
# the normalisation is a launch of its own
CASES = [(12544, 192, 192, 1), (12544, 768, 192, 1), (12481, 192, 192, 1), (12481, 201, 180, 1), (12544, 192, 164, 1), (16001, 201, 132, 1), (14001, 200, 148, 1),
         (33001, 768, 192, 1), (32961, 520, 180, 1), (33024, 600, 164, 1),
         (9999, 201, 180, 0), (12544, 64, 164, 0), (20001, 96, 132, 0), (9999, 96, 100, 0), (12544, 64, 196, 0), (9999, 192, 256, 0), (9999, 64, 163, 0),
         (12544, 192, 163, 0), (50, 192, 192, 0), (65, 64, 64, 0)]


@pytest.mark.parametrize("rows,k,n,one_launch", CASES)
def test_product_norm(rows, k, n, one_launch, monkeypatch):
    hip.init(0)
    print("product + LayerNormalization", rows, k, n, flush=True)
    m, rng = onefile.OneModel(), np.random.default_rng(rows + k + n)
    w = lambda *s: (rng.normal(size=s) / s[0] ** 0.5).astype(np.float32)   # noqa: E731
    m.input("x", (1, rows, k))
    m.matmul("skip", "x", w(k, n), "skip_out")
    m.matmul("p", "x", w(k, n), "p_mm")
    m.add("p_bias", "p_mm", w(n), "p_out")
    m.add("res", "p_out", "skip_out", "y")
    m.layernorm("ln", "y", 1 + w(n), w(n), "z")
    m.matmul("after", "z", w(n, 32), "u")
    for name, cols in (("y", n), ("z", n), ("u", 32)):
        m.output(name, (1, rows, cols))
    data = m.tobytes()
    fused = rt.Net(data)
    monkeypatch.setenv("ONENEW_RT_FUSE", "0")
    plain = rt.Net(data)
    for special in (False, True):
        x = rng.normal(size=(1, rows, k)).astype(np.float32)
        if special:
            x[0, rows - 1, 3], x[0, rows // 2, 5] = np.inf, np.nan
        before = hip.load().onhip_product_norm_launches()
        got = fused.run(x)
        assert hip.load().onhip_product_norm_launches() - before == one_launch
        for a, b in zip(got, plain.run(x)):
            assert np.array_equal(a, b, equal_nan=True)
            assert special or np.isfinite(a).all()
    fused.close()
    plain.close()


def test_measured_choices(monkeypatch):
    """the product alone is measured; what is chosen then normalises its rows where its tile holds them: the bits of the separate launches"""
    hip.init(0)
    rows, k, n = 12544, 192, 192
    m, rng = onefile.OneModel(), np.random.default_rng(5)
    w = lambda *s: (rng.normal(size=s) / s[0] ** 0.5).astype(np.float32)   # noqa: E731
    m.input("x", (1, rows, k))
    m.input("s", (1, rows, n))
    m.matmul("p", "x", w(k, n), "p_mm")
    m.add("p_bias", "p_mm", w(n), "p_out")
    m.add("res", "p_out", "s", "y")
    m.layernorm("ln", "y", 1 + w(n), w(n), "z")
    m.output("y", (1, rows, n))
    m.output("z", (1, rows, n))
    x, skip = rng.normal(size=(1, rows, k)).astype(np.float32), rng.normal(size=(1, rows, n)).astype(np.float32)
    net = rt.Net(m.tobytes())
    before = hip.set_tuning(1)
    try:
        for _ in range(2):   # measured, and chosen from what was
            launches = hip.load().onhip_product_norm_launches()
            y, z = net.run(x, skip)
            ran = hip.last_launch_choice()
            assert hip.load().onhip_product_norm_launches() - launches == (1 if ran[4] == 2 and ran[:2] == (192, 64) else 0), ran
    finally:
        hip.set_tuning(before)
    import torch
    t = lambda name: torch.from_numpy(net.fetch(name)).cuda()   # noqa: E731
    assert np.array_equal(hip.layernorm_f32(torch.from_numpy(y).cuda(), t("ln.weight"), t("ln.bias")).cpu().numpy(), z)
    net.close()
