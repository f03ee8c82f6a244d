"""Weights that the plugins keep split for the fp32 kernel on the 16-bit matrix cores: when the split form is made, and what
recorded graphs and other streams see of it.  Results against 64-bit sums within K 2^-24 sum |a b| and the roundings of bias and
result, as a chain of fp32 multiply-adds."""
import contextlib
import ctypes as C

import numpy as np
import pytest

from onenew_amd import abi, hip, ops
from onenew_amd.abi import ConvDesc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    hip.init(0)
    lib = hip.load()
    lib.onhip_plugin_set_stream.argtypes = [C.c_void_p]
    lib.onhip_plugin_set_async.argtypes = [C.c_int]
    return torch


@contextlib.contextmanager
def evals_on(stream):
    """evals queue on `stream` without waiting for their results"""
    lib = hip.load()
    assert lib.onhip_plugin_set_async(1) == 0 and lib.onhip_plugin_set_stream(C.c_void_p(stream.cuda_stream)) == 0
    try:
        yield
    finally:
        assert lib.onhip_plugin_set_stream(None) == 0 and lib.onhip_plugin_set_async(0) == 0


class Layer:
    """a 1x1 convolution or a linear layer on host weights, called with device buffers of any row count"""
    K, M = 256, 260

    def __init__(self, torch, kind, seed):
        self.torch, self.kind, self.g = torch, kind, torch.Generator().manual_seed(seed)
        self.w = torch.randn(self.M, self.K, generator=self.g) / self.K ** 0.5
        self.b = torch.randn(self.M, generator=self.g)
        if kind == "conv":
            d = ConvDesc(n=1, cin=self.K, h=4, w=4, cout=self.M, kh=1, kw=1, stride_h=1, stride_w=1, group=1, has_bias=1, act_type=abi.NOT_ACT,
                         compute=abi.COMPUTE_F32)
            self.op = ops.Conv(ops.Plugin(hip.plugin_path("Conv")).eval, d, self.w.numpy(), self.b.numpy())
        else:
            self.op = ops.MatMulFused(ops.Plugin(hip.plugin_path("MatMul")))
            self.host = [ops.aligned_empty(s) for s in ((self.K, self.M), (self.M,))]
            self.host[1][...] = self.b.numpy()
            self.set_weights(self.w)

    def set_weights(self, w):
        self.w = w
        if self.kind == "conv":
            self.op.weight[...] = w.reshape(self.op.weight.shape).numpy()
        else:
            self.host[0][...] = w.t().numpy()

    def hint(self, tile):
        """the model-wide tile, which narrows the choice of the Conv plugin's kernels"""
        if self.kind == "conv":
            info = self.op.useful.block_info
            info.cuda_gemm_tile_m = info.cuda_gemm_tile_n = tile

    def input(self, rows):
        n, hw = (rows // 256, 16) if rows >= 256 else (1, 4)
        shape = (n, self.K, hw, hw) if self.kind == "conv" else (rows, self.K)
        x = self.torch.randn(shape, generator=self.g).cuda()
        return x, self.torch.zeros((n, self.M, hw, hw) if self.kind == "conv" else (rows, self.M), device="cuda")

    def __call__(self, x, y):
        op = self.op
        if self.kind == "conv":
            for o, t in ((op.in_operand, x), (op.out_operand, y)):
                for i in range(4):
                    o.shapes[i] = t.shape[i]
            return op(x.data_ptr(), out=y.data_ptr())
        for i, o in enumerate([ops.make_operand(x.shape, b"a"), ops.make_operand((self.K, self.M), b"w", fixed=True),
                               ops.make_operand((self.M,), b"bias", fixed=True), ops.make_operand(y.shape, b"out")]):
            op._slot(op.params_vec, 1 + i, o)
        for i, t in enumerate((x.data_ptr(), *self.host)):
            op._slot(op.inputs_vec, i, t)
        op._slot(op.outputs_vec, 0, y.data_ptr())
        op._run(op.plugin.eval_bias, "eval_bias")

    def check(self, x, y):
        rows = x.double().cpu().permute(0, 2, 3, 1).reshape(-1, self.K) if self.kind == "conv" else x.double().cpu()
        got = y.double().cpu().permute(0, 2, 3, 1).reshape(-1, self.M) if self.kind == "conv" else y.double().cpu()
        w, b = self.w.double(), self.b.double()
        bound = (rows.abs() @ w.t().abs() + b.abs()) * ((self.K + 4) * 2.0 ** -24 + 2.0 ** -23)
        err = (got - (rows @ w.t() + b)).abs()
        assert bool((err <= bound).all()), float((err / bound).max())


def record(torch, layer, x, y, stream):
    graph = torch.cuda.CUDAGraph()
    with evals_on(stream), torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
        layer(x, y)
        assert hip.last_launch_choice()[4] == 2
    return graph


@pytest.mark.parametrize("kind", ["conv", "linear"])
def test_first_needed_under_capture(kind, torch_dev):
    """a layer whose split form is first asked for while a graph is recorded: an eval before the first replay is right, and so is
    every replay"""
    torch = torch_dev
    print(f"split weights first needed under capture: {kind}", flush=True)
    layer = Layer(torch, kind, 11)
    x, y = layer.input(16)
    layer.hint(64)
    layer(x, y)                       # weights on the device, no split form: a tile of the other kernels, or too little work
    layer.hint(16)
    assert hip.last_launch_choice()[4] != 2
    layer.check(x, y)
    x, y = layer.input(16384)
    recorded = torch.zeros_like(y)
    graph = record(torch, layer, x, recorded, torch.cuda.Stream())
    layer(x, y)
    assert hip.last_launch_choice()[4] == 2
    layer.check(x, y)
    for _ in range(3):
        recorded.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(recorded, y)
        layer(x, y)
        layer.check(x, y)


@pytest.mark.parametrize("kind", ["conv", "linear"])
def test_weights_changed_under_a_recorded_graph(kind, torch_dev):
    """host weights updated in place: the graph recorded before goes on reading its copy of them, which holds the new ones"""
    torch = torch_dev
    print(f"split weights changed under a graph: {kind}", flush=True)
    layer = Layer(torch, kind, 12)
    x, y = layer.input(16384)
    layer(x, y)
    layer.check(x, y)
    recorded = torch.zeros_like(y)
    graph = record(torch, layer, x, recorded, torch.cuda.Stream())
    for _ in range(3):
        layer.set_weights(torch.randn(layer.M, layer.K, generator=layer.g) / 16)
        layer(x, y)
        layer.check(x, y)
        recorded.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(recorded, y)


@pytest.mark.parametrize("kind", ["conv", "linear"])
def test_next_eval_on_another_stream(kind, torch_dev):
    """the split form is made behind other work of one stream; the next eval, on a second stream, does not run ahead of it"""
    torch = torch_dev
    print(f"split weights and a second stream: {kind}", flush=True)
    layer = Layer(torch, kind, 13)
    x, y = layer.input(16)
    layer.hint(64)
    layer(x, y)                       # weights on the device, no split form
    layer.hint(16)
    x, y = layer.input(16384)
    z = torch.zeros_like(y)
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        torch.cuda._sleep(20_000_000)   # about 10 ms
    for stream, out in ((first, y), (second, z)):
        with evals_on(stream):
            layer(x, out)
            assert hip.last_launch_choice()[4] == 2
    torch.cuda.synchronize()
    layer.check(x, z)
    assert torch.equal(y, z)


@pytest.fixture(scope="module")
def products(torch_dev):
    """products with enough work for weights split on the call, on operands of their own, and what they come to"""
    torch = torch_dev
    m, k, n = 8195, 773, 1030
    g = torch.Generator(device="cuda").manual_seed(5)
    jobs = []
    for _ in range(12):
        a, b = torch.randn(m, k, generator=g, device="cuda"), torch.randn(k, n, generator=g, device="cuda")
        bound = (a.double().abs() @ b.double().abs()) * ((k + 4) * 2.0 ** -24 + 2.0 ** -23)
        jobs.append((a, b, torch.zeros(m, n, device="cuda"), a.double() @ b.double(), bound))
    return jobs


def multiply(job):
    hip.matmul(job[0], job[1], out=job[2])
    assert hip.last_launch_choice()[4] == 2


def right(job):
    err = (job[2].double() - job[3]).abs()
    assert bool((err <= job[4]).all()), float((err / job[4]).max())
    job[2].zero_()


def test_more_streams_than_slots(products, torch_dev):
    """twelve streams at once, a second round in another order, and streams that come and go: every one splits on the call"""
    torch = torch_dev
    print("split weights: streams", flush=True)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in products]
    for order in (range(12), range(11, -1, -1)):
        for i in order:
            with torch.cuda.stream(streams[i]):
                multiply(products[i])
        torch.cuda.synchronize()
        for job in products:
            right(job)
    hiprt, old = C.CDLL(None), []
    for _ in range(3):   # nine new streams while the nine before are still there, which are destroyed then
        new = [C.c_void_p() for _ in range(9)]
        for handle in new:
            assert hiprt.hipStreamCreate(C.byref(handle)) == 0
        for handle in old:
            assert hiprt.hipStreamDestroy(handle) == 0
        for handle, job in zip(new, products):
            with torch.cuda.stream(torch.cuda.ExternalStream(handle.value)):
                multiply(job)
        torch.cuda.synchronize()
        for job in products[:9]:
            right(job)
        old = new
    for handle in old:
        assert hiprt.hipStreamDestroy(handle) == 0


def test_captures_that_come_and_go(products, torch_dev):
    """graphs recorded and dropped, more of them than there are slots: each has a slot, and the one that lives keeps its own"""
    torch = torch_dev
    print("split weights: captures", flush=True)
    stream = torch.cuda.Stream()

    def graph_of(job):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            multiply(job)
        return graph

    torch.cuda.synchronize()
    kept = graph_of(products[0])
    for i in range(70):
        job = products[1 + i % 11]
        graph = graph_of(job)
        graph.replay()
        kept.replay()
        torch.cuda.synchronize()
        if i % 10 == 9:
            right(job)
            right(products[0])
        del graph
    assert hip.load().onhip_plugin_release() == 0   # slots that no graph holds are given back, not this one's
    kept.replay()
    multiply(products[1])
    torch.cuda.synchronize()
    right(products[0])
    right(products[1])
