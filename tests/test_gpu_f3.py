"""fp32 convolutions and products on the 16-bit matrix cores (operands as three bf16 parts): every tile and loader at ragged
sizes against 64-bit sums.  The bound is that of a chain of fp32 multiply-adds, K 2^-24 sum |a b|, plus what the three left-out
partial products can reach, 2^-23 sum |a b|, and the roundings of the bias and the result."""
import threading

import numpy as np
import pytest

from onenew_amd import abi, hip
from onenew_amd.abi import ConvDesc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    hip.init(0)
    return torch


def conv_desc(n, cin, h, w, cout, k, stride, pad):
    kh, kw = k if isinstance(k, tuple) else (k, k)
    return ConvDesc(n=n, cin=cin, h=h, w=w, cout=cout, kh=kh, kw=kw, stride_h=stride, stride_w=stride, pad_t=pad, pad_l=pad, pad_b=pad, pad_r=pad,
                    group=1, has_bias=1, act_type=abi.NOT_ACT, compute=abi.COMPUTE_F32)


def check(got, ref, magnitude, k):
    """got within the bound of ref (fp64), non-finite where ref is; magnitude: sum |a b| + |bias| in fp64"""
    got = got.double().cpu()
    bad = ~ref.isfinite()
    assert bool((got.isnan() == ref.isnan()).all()) and bool((got[bad & ~ref.isnan()] == ref[bad & ~ref.isnan()]).all())
    err = (got - ref).abs()[~bad]
    bound = (magnitude * ((k + 4) * 2.0 ** -24 + 2.0 ** -23))[~bad]
    assert bool((err <= bound + 1e-38).all()), float((err / bound).max())


def conv_ref(torch, d, x, w, b):
    conv = lambda x, w, b: torch.nn.functional.conv2d(x.double().cpu(), w.double().cpu(), b.double().cpu(), stride=d.stride_h, padding=d.pad_t)  # noqa: E731
    return conv(x, w, b), conv(x.abs(), w.abs(), b.abs())


TILES = [(256, 128), (256, 64), (192, 64), (128, 128), (128, 64), (64, 64)]
# loader, (n, cin, h, w, cout, filter, stride, pad): rows and columns off every tile, reductions off a K tile of 16 and off a unit of 4
SHAPES = [("plain", (2, 109, 9, 23, 67, 1, 1, 0)), ("plain", (1, 130, 16, 17, 259, 1, 1, 0)), ("tapc", (2, 13, 11, 9, 97, 3, 1, 1)),
          ("tapc", (1, 33, 15, 12, 260, 3, 2, 1)), ("gather", (1, 13, 13, 21, 65, 3, 1, 1)), ("tapc", (1, 20, 12, 13, 70, 7, 1, 3)), ("gather", (1, 6, 9, 14, 66, (5, 11), 2, 2)), ("gather", (2, 117, 14, 9, 40, 1, 2, 0))]


@pytest.mark.parametrize("special", [False, True], ids=["finite", "special"])
@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("bm,bn", TILES)
@pytest.mark.parametrize("loader,shape", SHAPES, ids=[f"{s[0]}{i}" for i, s in enumerate(SHAPES)])
def test_convolution(loader, shape, bm, bn, split, special, torch_dev, monkeypatch):
    torch = torch_dev
    print(f"f3 {loader} {shape} tile {bm}x{bn} split {split} special {special}", flush=True)
    monkeypatch.setenv("ONHIP_TILE", f"{bm}x{bn}x{split}x0x2")
    d = conv_desc(*shape)
    if special and loader == "tapc":
        d.cin += -d.cin % 4   # packed weights round the channels up to four; what lies there (the next image) meets zero weights
    g = torch.Generator().manual_seed(hash((shape, bm)) % 1000)
    x = torch.randn(d.n, d.cin, d.h, d.w, generator=g)
    w, b = torch.randn(d.cout, d.cin, d.kh, d.kw, generator=g) / (d.cin * d.kh * d.kw) ** 0.5, torch.randn(d.cout, generator=g)
    if special:   # an infinity, a NaN, values that round to bf16 infinities (products with them stay finite)
        x[0, 0, 1, 2], x[-1, 1, 3, 4], x[0, 2, 5, 5], w[5, 3] = float("inf"), float("nan"), 3.4e38, -3.4e38
        x[:, 3] *= 1e-3
    x, w, b = x.cuda(), w.cuda(), b.cuda()
    wk = hip.pack_conv_weights(d, w) if loader == "tapc" else w
    y = hip.conv2d_f32(d, x, wk, b, packed=loader == "tapc")
    assert hip.last_launch_choice()[4] == 2
    torch.cuda.synchronize()
    ref, magnitude = conv_ref(torch, d, x, w, b)
    if special:
        ok = magnitude < 1e38   # sums that may overflow on the way are left to the infinities' and NaNs' own check
        ref, got, magnitude = ref[ok | ~magnitude.isfinite()], y.cpu()[ok | ~magnitude.isfinite()], magnitude[ok | ~magnitude.isfinite()]
        return check(got, ref, magnitude, d.cin * d.kh * d.kw)
    check(y, ref, magnitude, d.cin * d.kh * d.kw)


@pytest.mark.parametrize("m,k,n", [(4099, 1031, 2053), (8195, 773, 1030), (8190, 1029, 1027), (12545, 193, 768)])
@pytest.mark.parametrize("special", [False, True], ids=["finite", "special"])
def test_product(m, k, n, special, torch_dev):
    torch = torch_dev
    print(f"f3 product {m} x {k} x {n} special {special}", flush=True)
    g = torch.Generator().manual_seed(m + k)
    a, b, bias = torch.randn(m, k, generator=g), torch.randn(k, n, generator=g) / k ** 0.5, torch.randn(n, generator=g)
    if special:
        a[3, 5], a[m - 1, k - 1], b[7, n - 1] = float("inf"), float("nan"), -float("inf")
    a, b, bias = a.cuda(), b.cuda(), bias.cuda()
    y = hip.matmul(a, b, bias)
    assert hip.last_launch_choice()[4] == 2
    torch.cuda.synchronize()
    check(y, (a.double() @ b.double() + bias.double()).cpu(), (a.double().abs() @ b.double().abs() + bias.double().abs()).cpu(), k)


@pytest.mark.parametrize("bm,bn", TILES)
@pytest.mark.parametrize("loader,shape", [SHAPES[i] for i in (0, 1, 3, 4, 7)], ids=["plain0", "plain1", "tapc3", "gather4", "gather7"])
def test_stores(loader, shape, bm, bn, torch_dev, monkeypatch):
    """the residual operand's kernels and the activations of a store, bit for bit what the operators do to the plain store's result"""
    torch = torch_dev
    print(f"f3 stores {loader} {shape} tile {bm}x{bn}", flush=True)
    monkeypatch.setenv("ONHIP_TILE", f"{bm}x{bn}x1x0x2")
    d = conv_desc(*shape)
    g = torch.Generator(device="cuda").manual_seed(bm + bn)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    x, w, b = rand(d.n, d.cin, d.h, d.w), rand(d.cout, d.cin, d.kh, d.kw) / (d.cin * d.kh * d.kw) ** 0.5, rand(d.cout)
    wk = hip.pack_conv_weights(d, w) if loader == "tapc" else w
    packed = loader == "tapc"
    y = hip.conv2d_f32(d, x, wk, b, packed=packed)
    r = rand(*y.shape)
    for relu in (False, True):
        z = hip.conv2d_f32_add(d, x, wk, r, b, relu=relu, packed=packed)
        assert hip.last_launch_choice()[4] == 2 and hip.last_launch_choice()[:2] == (bm, bn)
        assert torch.equal(z, (y + r).clamp(min=0) if relu else y + r)
    d.act_type = abi.RELU
    assert torch.equal(hip.conv2d_f32(d, x, wk, b, packed=packed), y.clamp(min=0))
    d.act_type, d.clip_min, d.clip_max = abi.CLIP, -0.5, 0.75
    assert torch.equal(hip.conv2d_f32(d, x, wk, b, packed=packed), y.clamp(-0.5, 0.75))
    assert hip.last_launch_choice()[4] == 2


@pytest.mark.parametrize("m,k,n", [(8195, 773, 1030), (12545, 193, 768), (8190, 1029, 193)])
def test_product_stores(m, k, n, torch_dev, oracle):
    """an addend with and without a bias, and the table GELU, bit for bit what the operators do to the plain store's result"""
    torch = torch_dev
    print(f"f3 product stores {m} x {k} x {n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    a, b, bias, r = rand(m, k), rand(k, n) / k ** 0.5, rand(n), rand(m, n)
    lut = torch.from_numpy(np.ascontiguousarray(oracle.gelu_lut())).cuda()
    for v in (None, bias):
        y = hip.matmul(a, b, v)
        assert hip.last_launch_choice()[4] == 2
        plain = hip.last_launch_choice()
        z = hip.matmul(a, b, v, addend=r)
        assert hip.last_launch_choice() == plain
        assert torch.equal(z, y + r)
        z = hip.matmul(a, b, v, gelu_lut=lut)
        assert hip.last_launch_choice() == plain
        assert torch.equal(z, hip.gelu_lut_f32(y, lut))


def test_time_on_nonfinite_data(torch_dev):
    """sums that are not finite are computed again at the rate of matrix instructions: 4.3 times the time where all of them are, 118 times
    with one multiply-add a lane and element"""
    torch = torch_dev
    print("f3 time on non-finite data", flush=True)
    a, b, y = torch.randn(4099, 1031, device="cuda"), torch.randn(1031, 2053, device="cuda"), torch.empty(4099, 2053, device="cuda")

    def ms():
        hip.matmul(a, b, out=y)
        assert hip.last_launch_choice()[4] == 2
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        times = []
        for _ in range(5):
            start.record()
            hip.matmul(a, b, out=y)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        return sorted(times)[2]

    finite = ms()
    a[:] = float("nan")
    assert ms() <= 16 * finite
    assert bool(y.isnan().all())


def test_product_under_a_tile_hint(torch_dev):
    """a hint restricts the choice to its tile, which this kernel's choice is not"""
    torch = torch_dev
    print("f3 product under a tile hint", flush=True)
    a, b = torch.randn(8195, 773, device="cuda"), torch.randn(773, 1030, device="cuda")
    lib = hip.load()
    assert lib.onhip_set_tile_hint(64, 128) == 1
    try:
        y = hip.matmul(a, b)
        assert hip.last_launch_choice()[:2] == (64, 128) and hip.last_launch_choice()[4] != 2
    finally:
        assert lib.onhip_set_tile_hint(0, 0) == 0
    hip.matmul(a, b)
    assert hip.last_launch_choice()[4] == 2
    check(y, (a.double() @ b.double()).cpu(), (a.double().abs() @ b.double().abs()).cpu(), 773)


MEASURED = """
import sys, torch
sys.path.insert(0, sys.argv[1])
from onenew_amd import hip
hip.init(0)
a, b = torch.randn(8195, 773, device="cuda"), torch.randn(773, 1030, device="cuda")
y = hip.matmul(a, b)
ref, scale = a.double() @ b.double(), a.double().abs() @ b.double().abs()
print("RAN", *hip.last_launch_choice(), float(((y.double() - ref).abs() / scale).max()))
"""


def measuring(program, cache):
    """a process of its own, as measured choices are kept for the life of one"""
    import os
    import subprocess
    import sys
    print("f3 measured choices", flush=True)
    env = {k: v for k, v in os.environ.items() if k != "ONHIP_TILE"}
    env.update(ONHIP_TUNE="1", ONHIP_TUNE_CACHE=str(cache))
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", program, root], env=env, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr[-2000:]
    return out


def test_product_measured(tmp_path):
    """with measured choices the product's launches of both forms are timed, the winner is kept, and a kept choice is obeyed"""
    cache = tmp_path / "tune.txt"

    def ran():
        out = measuring(MEASURED, cache)
        *choice, err = [line for line in out.stdout.splitlines() if line.startswith("RAN")][0].split()[1:]
        assert float(err) <= (773 + 4) * 2.0 ** -24 + 2.0 ** -23
        return [int(v) for v in choice]

    ran()
    lines = cache.read_text().splitlines()
    assert len(lines) == 1
    for choice in ("128 128 1 0 0 0 0", "192 64 1 0 2 0 0"):
        cache.write_text(lines[0].split(":")[0] + ": " + choice + "\n")
        got = ran()
        assert [got[0], got[1], got[4]] == [int(v) for v in (choice.split()[0], choice.split()[1], choice.split()[4])]
        assert len(cache.read_text().splitlines()) == 1


KEPT = """
import sys, numpy as np, torch
sys.path.insert(0, sys.argv[1])
from onenew_amd import hip, ops
hip.init(0)
d = ops.ConvDesc(n=4, cin=256, h=20, w=20, cout=128, kh=1, kw=1, stride_h=1, stride_w=1, group=1, has_bias=1)
x, w, b = (np.random.default_rng(0).standard_normal(s, dtype=np.float32) for s in ((4, 256, 20, 20), (128, 256, 1, 1), (128,)))
hip.conv2d_f32(d, *(torch.from_numpy(t).cuda() for t in (x, w, b)))
ops.Conv(ops.Plugin(hip.plugin_path("Conv")).eval, d, w, b)(x)
"""


def test_kept_weights_are_measured_apart(tmp_path):
    """a layer whose weights are kept split and one that splits them on the call do not share a measured choice"""
    measuring(KEPT, tmp_path / "tune.txt")
    keys = {line.split(":")[0] for line in (tmp_path / "tune.txt").read_text().splitlines()}
    assert len(keys) == 2, keys


@pytest.mark.parametrize("n,cin,hw,cout,ours", [(64, 384, 14, 64, False), (64, 96, 14, 576, True), (64, 320, 7, 1280, True)])
def test_layers_bound_by_their_activations(n, cin, hw, cout, ours, torch_dev):
    """1x1 layers of MobileNetV2 on kept weights: a lone workgroup per compute unit that waits for its activations gains too little from the
    16-bit matrix cores (16.8 -> 16.0 us for the first layer) for what they draw; the others gain a quarter"""
    from onenew_amd import ops
    torch = torch_dev
    print(f"f3 choice {n} x {cin} x {hw} -> {cout}", flush=True)
    d = conv_desc(n, cin, hw, hw, cout, 1, 1, 0)
    rng = np.random.default_rng(cin)
    x, w, b = (rng.standard_normal(s, dtype=np.float32) for s in ((n, cin, hw, hw), (cout, cin, 1, 1), (cout,)))
    y = torch.from_numpy(ops.Conv(ops.Plugin(hip.plugin_path("Conv")).eval, d, w, b)(x)).double()
    assert (hip.last_launch_choice()[4] == 2) == ours
    x, w, b = (torch.from_numpy(t) for t in (x, w, b))
    check(y, *conv_ref(torch, d, x, w, b), cin)


def test_streams_and_threads(torch_dev):
    """weights split on the call: more streams than there are slots for them, one after another, and two threads on one stream"""
    torch = torch_dev
    print("f3 streams and threads", flush=True)
    m, k, n = 8195, 773, 1030
    g = torch.Generator(device="cuda").manual_seed(3)
    jobs = []
    for _ in range(10):
        a, b = torch.randn(m, k, generator=g, device="cuda"), torch.randn(k, n, generator=g, device="cuda")
        jobs.append((a, b, torch.empty(m, n, device="cuda"), (a.double() @ b.double()).cpu(), (a.double().abs() @ b.double().abs()).cpu()))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in jobs]
    for s, (a, b, y, _, _) in zip(streams, jobs):   # no cut along K: nothing but the split weights could be shared
        with torch.cuda.stream(s):
            hip.matmul(a, b, out=y)
    torch.cuda.synchronize()

    def verify():
        for _, _, y, ref, magnitude in jobs:
            check(y, ref, magnitude, k)
            y.zero_()
        torch.cuda.synchronize()
    verify()

    def work(mine):
        for _ in range(8):
            for a, b, y, _, _ in mine:
                hip.matmul(a, b, out=y)
    threads = [threading.Thread(target=work, args=(jobs[i::2],)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    verify()


def test_capture(torch_dev, monkeypatch):
    """Split weights under capture: graphs recorded on one stream and replayed on two at once each have a slot of their own.
    33 captures are one more than there are slots for: the last ones run other kernels, cut nowhere, as nothing else may be
    allocated there."""
    torch = torch_dev
    print("f3 capture", flush=True)
    m, k, n = 8195, 773, 1030
    d = conv_desc(3, 300, 20, 19, 259, 1, 1, 0)
    g = torch.Generator(device="cuda").manual_seed(4)
    rand = lambda *shape: torch.randn(shape, generator=g, device="cuda")  # noqa: E731
    jobs = []
    for _ in range(2):
        a, b, x, w, bias = rand(m, k), rand(k, n), rand(d.n, d.cin, d.h, d.w), rand(d.cout, d.cin, 1, 1), rand(d.cout)
        jobs.append((a, b, x, w, bias, torch.empty(m, n, device="cuda"), torch.empty(d.n, d.cout, d.h, d.w, device="cuda"),
                     ((a.double() @ b.double()).cpu(), (a.double().abs() @ b.double().abs()).cpu()), conv_ref(torch, d, x, w, bias)))
    choices = []

    def work(job):
        a, b, x, w, bias, y, z = job[:7]
        choices.clear()
        hip.matmul(a, b, out=y)
        choices.append(hip.last_launch_choice())
        monkeypatch.setenv("ONHIP_TILE", "128x64x1x0x2")
        hip.conv2d_f32(d, x, w, bias, out=z)
        monkeypatch.delenv("ONHIP_TILE")
        choices.append(hip.last_launch_choice())

    stream, others = torch.cuda.Stream(), [torch.cuda.Stream() for _ in jobs]
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        work(jobs[0])
    assert all(c[4] == 2 for c in choices), choices
    torch.cuda.synchronize()

    def record(job):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            work(job)
        return graph

    def replay(graphs):
        for _ in range(3):
            for job in jobs:
                job[5].zero_()
                job[6].zero_()
            torch.cuda.synchronize()
            for graph, s in zip(graphs, others):
                with torch.cuda.stream(s):
                    graph.replay()
            with torch.cuda.stream(stream):   # the recording stream goes on with weights of its own
                hip.matmul(jobs[0][0], jobs[1][1])
                assert hip.last_launch_choice()[4] == 2
            torch.cuda.synchronize()
            for job in jobs:
                check(job[5], *job[7], k)
                check(job[6], *job[8], d.cin)

    first = []
    for job in jobs:
        first.append(record(job))
        assert all(c[4] == 2 for c in choices), choices
    replay(first)
    graphs = [record(jobs[i % 2]) for i in range(33)]
    assert all(c[4] != 2 and c[2] == 1 and c[3] == 0 for c in choices), choices
    replay(graphs[-2:])


# exponents of the left and the right operand: low bits below bf16's subnormals, subnormal fp32 numbers, operands and sums that
# overflow with the operands' scale on them
RANGES = [(-120, 0), (0, -120), (-66, -58), (-140, 20), (20, -140), (108, -20), (-20, 108), (50, 40)]


@pytest.mark.parametrize("form", ["plain", "tapc", "gather", "rows"])
@pytest.mark.parametrize("ea,eb", RANGES)
def test_ends_of_the_range(ea, eb, form, torch_dev, monkeypatch):
    """no operand that fp32 holds loses bits: the bound of a chain of fp32 multiply-adds, each of which may round at 2^-149"""
    torch = torch_dev
    print(f"f3 operands of 2^{ea} and 2^{eb}, {form}", flush=True)
    g = torch.Generator().manual_seed(5)
    scaled = lambda e, *shape: (torch.randn(shape, generator=g).double() * 2.0 ** e).float().cuda()  # noqa: E731
    if form == "rows":
        k = 773
        a, b = scaled(ea, 8195, k), scaled(eb, k, 1030)
        y, chosen = hip.matmul(a, b), hip.last_launch_choice()[4]
        ref, magnitude = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    else:
        d = conv_desc(2, 36, 13, 11, 70, 1 if form == "plain" else 3, 1, 0)
        d.has_bias = 0
        k = d.cin * d.kh * d.kw
        x, w = scaled(ea, d.n, d.cin, d.h, d.w), scaled(eb, d.cout, d.cin, d.kh, d.kw)
        monkeypatch.setenv("ONHIP_TILE", "64x64x1x0x2")
        y = hip.conv2d_f32(d, x, hip.pack_conv_weights(d, w) if form == "tapc" else w, None, packed=form == "tapc")
        chosen = hip.last_launch_choice()[4]
        zero = torch.zeros(d.cout)
        ref, magnitude = conv_ref(torch, d, x, w, zero)
    assert chosen == 2
    err, bound = (y.double().cpu() - ref.cpu()).abs(), magnitude.cpu() * ((k + 4) * 2.0 ** -24 + 2.0 ** -23) + k * 2.0 ** -149
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("values", ["normal", "positive", "uneven", "spread"])
@pytest.mark.parametrize("cin,filt", [(48, 1), (192, 1), (768, 1), (128, 3), (512, 3)])
def test_error_no_larger_than_of_fp32_matrix_instructions(cin, filt, values, torch_dev, monkeypatch):
    """both kernels of a layer against 64-bit sums, errors as a share of sum |a b|: the root mean square over the outputs.  0.63-0.88 on values
    as layers hold them (spread over 2^+-4 among them).  Where operands spread over 2^+-24 a single term decides the sum and its own
    rounding the error: 1.10-1.19, asked to stay below 1.25."""
    torch = torch_dev
    d = conv_desc(2, cin, 24, 24, 192, filt, 1, filt // 2)
    d.has_bias = 0
    g = torch.Generator().manual_seed(cin)
    x, w = torch.randn(d.n, cin, d.h, d.w, generator=g), torch.randn(d.cout, cin, filt, filt, generator=g)
    if values == "positive":
        x, w = x.abs(), w.abs()
    if values in ("uneven", "spread"):
        e = 4 if values == "uneven" else 24
        x, w = (t * 2.0 ** (2 * e * torch.rand(t.shape, generator=g) - e) for t in (x, w))
    ref, magnitude = conv_ref(torch, d, x, w, torch.zeros(d.cout))
    x, w = x.cuda(), w.cuda()
    wk = hip.pack_conv_weights(d, w) if filt > 1 else w

    def error(tile):
        monkeypatch.setenv("ONHIP_TILE", tile)
        y = hip.conv2d_f32(d, x, wk, None, packed=filt > 1).double().cpu()
        return float(((y - ref) / magnitude).square().mean().sqrt())

    ours, theirs = error("64x64x1x0x2"), error("64x64x1")
    print(f"f3 error K {cin * filt * filt} {values}: {ours:.3e}, of fp32 matrix instructions {theirs:.3e}, ratio {ours / theirs:.3f}", flush=True)
    assert ours <= (1.25 if values == "spread" else 1.0) * theirs
