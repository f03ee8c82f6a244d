"""1x1 fp32 convolutions with kept weights and more than 8 MB of activations on the kernel whose wavefronts share K: either side of 8 and 64 MB, of 96 rows
with a K of 1024 and of a K of 320 in 64 rows, rows, columns and K off the tiles, with an addend; the result against 64 bits, within what a chain of fp32
multiply-adds can be off."""
import numpy as np
import pytest

from onenew_amd import hip, onefile, rt

pytestmark = pytest.mark.gpu

# images, side, input and output channels, addend, this kernel or not (None: either)
CASES = [(64, 14, 384, 64, True, 1), (64, 14, 384, 64, False, None), (64, 7, 960, 160, True, 1), (32, 14, 381, 33, False, 1), (33, 14, 577, 130, False, 1), (8, 28, 960, 160, False, 1),
         (8, 56, 96, 24, False, None), (8, 56, 576, 24, True, 1), (64, 14, 192, 64, False, 0), (32, 14, 1500, 130, False, 0), (42, 28, 521, 20, False, 0), (10, 14, 1070, 70, True, None),
         (11, 14, 1070, 70, True, None)]


@pytest.mark.parametrize("n,hw,cin,cout,addend,ours", CASES)
def test_layer(n, hw, cin, cout, addend, ours):
    import torch
    hip.init(0)
    print(f"{n} x {cin} x {hw}^2 -> {cout}", flush=True)
    rng = np.random.default_rng(cin + cout)
    m, w, b = onefile.OneModel(), (rng.normal(size=(cout, cin, 1, 1)) / cin ** 0.5).astype(np.float32), rng.normal(size=cout).astype(np.float32)
    m.input("x", (n, cin, hw, hw))
    if addend:
        m.input("s", (n, cout, hw, hw))
        m.conv("c", "x", w, b, "c_out")
        m.add("a", "c_out", "s", "y")
    else:
        m.conv("c", "x", w, b, "y")
    m.output("y", (n, cout, hw, hw))
    net = rt.Net(m.tobytes())
    g = torch.Generator(device="cuda").manual_seed(cin)
    x, s = torch.randn((n, cin, hw, hw), generator=g, device="cuda"), torch.randn((n, cout, hw, hw), generator=g, device="cuda")
    y = torch.empty((n, cout, hw, hw), device="cuda")
    net.enqueue_raw([x.data_ptr()] + ([s.data_ptr()] if addend else []), [y.data_ptr()])
    torch.cuda.synchronize()
    choice = list(hip.last_launch_choice())
    assert ours is None or (choice[4] == 3) == bool(ours), choice
    wd, bd = torch.from_numpy(w).cuda().double(), torch.from_numpy(b).cuda().double()[:, None, None]
    conv = lambda x, w: torch.matmul(w.reshape(cout, cin), x.reshape(n, cin, hw * hw)).reshape(n, cout, hw, hw)  # noqa: E731
    ref, mass = conv(x.double(), wd) + bd, conv(x.double().abs(), wd.abs()) + bd.abs()
    if addend:
        ref, mass = ref + s, mass + s.abs()
    assert bool(((y.double() - ref).abs() <= mass * ((cin + 5) * 2.0 ** -24 + 2.0 ** -23)).all())
    net.close()
