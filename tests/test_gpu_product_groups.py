"""Linear layers of one shape on one input, which the runtime runs as one call (and the library as one launch where that is faster): the bits of
the net run operator by operator."""
import numpy as np
import pytest

from onenew_amd import hip, onefile, rt

pytestmark = pytest.mark.gpu


# (rows, k, n, products, groups): rows and products for which each runs on its own and no copy of the weights is made; then one launch, with tiles that
# cover two products and end inside the last one, K off sixteen, rows off every tile, more products than a group takes
CASES = [(2099, 192, 192, 3, 0), (5000, 64, 96, 2, 0), (1500, 201, 224, 4, 0), (3000, 192, 160, 5, 0), (50, 96, 64, 3, 0),
         (12544, 192, 192, 3, 1), (12546, 192, 192, 2, 1), (9002, 201, 224, 4, 1), (12622, 192, 160, 5, 1), (3154, 384, 384, 3, 1)]


@pytest.mark.parametrize("rows,k,n,products,groups", CASES)
def test_group(rows, k, n, products, groups, monkeypatch):
    hip.init(0)
    print("product group", rows, k, n, products, flush=True)
    m, rng = onefile.OneModel(), np.random.default_rng(rows + n)
    w = lambda *s: (rng.normal(size=s) / s[0] ** 0.5).astype(np.float32)   # noqa: E731
    m.input("x", (2, rows // 2, k))
    for i in range(products):
        m.matmul(f"p{i}", "x", w(k, n), f"p{i}_mm")
        m.add(f"p{i}_bias", f"p{i}_mm", w(n), f"y{i}")
        if i == 0:   # another shape between them
            m.matmul("odd", "x", w(k, 33), "odd_mm")
            m.add("odd_bias", "odd_mm", w(33), "odd_y")
        m.output(f"y{i}", (2, rows // 2, n))
    m.output("odd_y", (2, rows // 2, 33))
    data = m.tobytes()
    fused = rt.Net(data)
    monkeypatch.setenv("ONENEW_RT_FUSE", "0")
    plain = rt.Net(data)
    assert fused.fused_linears() == products + 1
    assert fused.product_groups() == groups and plain.product_groups() == 0
    for scale in (1.0, -0.3):
        x = (rng.normal(size=(2, rows // 2, k)) * scale).astype(np.float32)
        if scale < 0:
            x[1, 3, 5] = np.inf
        got, ref = fused.run(x), plain.run(x)
        for i, (a, b) in enumerate(zip(got, ref)):
            assert np.array_equal(a, b, equal_nan=True), i
        assert np.isfinite(got[0][0]).all()
        for i in range(products):
            assert np.array_equal(fused.fetch(f"y{i}"), ref[i], equal_nan=True)
    fused.close()
    plain.close()


@pytest.mark.parametrize("measured", [0, 1], ids=["by the model", "measured choices"])
def test_one_launch(measured):
    """three products of 192 columns run as one of 576, in tiles that a product of 192 is not cut into; under measured choices as well"""
    hip.init(0)
    ran = []
    for products, tuning in ((1, 0), (3, measured)):
        m, rng = onefile.OneModel(), np.random.default_rng(3)
        m.input("x", (64, 196, 192))
        for i in range(products):
            m.matmul(f"p{i}", "x", (rng.normal(size=(192, 192)) * 0.07).astype(np.float32), f"p{i}_mm")
            m.add(f"p{i}_bias", f"p{i}_mm", rng.normal(size=192).astype(np.float32), f"y{i}")
            m.output(f"y{i}", (64, 196, 192))
        net = rt.Net(m.tobytes())
        before = hip.set_tuning(tuning)
        try:
            net.run(rng.normal(size=(64, 196, 192)).astype(np.float32))
        finally:
            hip.set_tuning(before)
        ran.append(tuple(hip.last_launch_choice()))
        net.close()
    assert ran[0][4] == ran[1][4] == 2 and ran[0][:2] != ran[1][:2], ran


def test_an_operand_with_the_name_of_the_weights_side_by_side(monkeypatch):
    """the copy that a group's weights and biases have is no operand: one of the model's that is called like it stays what it is"""
    hip.init(0)
    m, rng = onefile.OneModel(), np.random.default_rng(8)
    w = lambda *s: (rng.normal(size=s) / s[0] ** 0.5).astype(np.float32)   # noqa: E731
    rows, k, n = 12544, 192, 192
    m.input("x", (1, rows, k))
    for i in range(2):
        m.matmul(f"p{i}", "x", w(k, n), f"p{i}_mm")
        m.add(f"p{i}_bias", f"p{i}_mm", w(n), f"y{i}")
        m.output(f"y{i}", (1, rows, n))
    m.matmul("q", "x", m.init("y0/weights side by side", w(k, 2 * n)), "q_mm")
    m.add("q_bias", "q_mm", m.init("y0/biases side by side", w(2 * n)), "z")
    m.output("z", (1, rows, 2 * n))
    data, x = m.tobytes(), rng.normal(size=(1, rows, k)).astype(np.float32)
    fused = rt.Net(data)
    monkeypatch.setenv("ONENEW_RT_FUSE", "0")
    plain = rt.Net(data)
    assert fused.product_groups() == 1
    for a, b in zip(fused.run(x), plain.run(x)):
        assert np.array_equal(a, b)
    assert np.array_equal(fused.fetch("y0/weights side by side"), plain.fetch("y0/weights side by side"))
    fused.close()
    plain.close()
