"""GPU parity of the training passes whose workgroups share a channel's slice: the checks of the other geometries, with
their tolerances, at the sizes where the split changes; then under graph replay and on two streams at once."""
import numpy as np
import pytest

import test_gpu_clipped_backward as clipped
import test_gpu_epilogue as epilogue
from pixienn_amd import workloads as wl
from util import F, assert_bit_exact, gpu, host

pytestmark = pytest.mark.gpu

# vectors of a slice: 4097 (the first that the small forms leave) in two members; three members of 2048; planes that end
# inside a share, in eight and in twelve; 64 members, the last of one wavefront, and 65 (three launches); members that are
# full, sixteen of 6144; more shares than the device runs at once; 512 channels of one member.  How they are split is held by
# tests/host/split_check.cpp.
VECTORS = [(1, 95, 16388), (4, 64, 6144), (7, 30, 10012), (3, 12, 32772), (1, 8, 532480), (1, 7, 532480), (4, 32, 98304),
           (3, 130, 32772), (4, 512, 4112)]
# odd planes (groups but for mish): five members, twelve, and sixteen that are full (but for the last value, which its vector shares)
ODD = [(8, 96, 10395), (32, 41, 5625), (1, 32, 393215)]


@pytest.fixture(scope="module")
def ops():
    from pixienn_amd import ops as o
    return o


@pytest.mark.parametrize("act", ["leaky", "mish"])
@pytest.mark.parametrize("shape", VECTORS + ODD, ids=str)
def test_shared_slices_backward(ops, oracle, monkeypatch, shape, act):
    for module in (epilogue, clipped):
        monkeypatch.setattr(module, "TRAIN_SHAPES", [shape])
    epilogue.test_bn_backward_matches_oracle(ops, oracle, act, False)
    clipped.test_bn_backward_clipped_matches_rescale_clip_then_backward(ops, oracle, act, False)


@pytest.mark.parametrize("act", ["logistic", "softplus"])
@pytest.mark.parametrize("shape", ODD, ids=str)
def test_shared_slices_of_odd_planes_before_an_exponential(ops, oracle, monkeypatch, shape, act):
    test_shared_slices_backward(ops, oracle, monkeypatch, shape, act)


class Layer:
    """A layer's tensors, and both passes over them with a workspace of its own."""

    def __init__(self, ops, torch, seed, shape):
        from pixienn_amd import capi
        lib = capi.load()
        N, C, H, W = shape
        self.ops = ops
        self.x, self.delta = gpu(wl.normal(seed, shape)), gpu(wl.normal(seed + 1, shape))
        scale, bias, rmean, rvar = wl.bn_params(seed + 2, C)
        self.scale, self.bias, self.rolling0 = gpu(scale), gpu(bias), (gpu(rmean), gpu(rvar))
        self.mean, self.var, self.rm, self.rv, self.su, self.bu = (torch.zeros(C, device="cuda") for _ in range(6))
        self.y, self.d = torch.empty_like(self.x), torch.empty_like(self.x)
        need = max(lib.pxh_bn_workspace_bytes(N, C, H * W), lib.pxh_bn_clipped_workspace_bytes(N, C, H * W))
        self.workspace = torch.zeros(need // 4 + 4, device="cuda")

    def run(self, clip):
        self.d.copy_(self.delta)
        self.rm.copy_(self.rolling0[0]); self.rv.copy_(self.rolling0[1])
        self.su.zero_(); self.bu.zero_()
        self.ops.bn_train_act_forward(self.x, self.y, self.mean, self.var, self.rm, self.rv, self.scale, self.bias, "leaky",
                                      workspace=self.workspace)
        self.ops.bn_act_backward_clipped(self.d, self.x, self.mean, self.var, self.scale, self.bias, self.su, self.bu, "leaky",
                                         1e6, clip, workspace=self.workspace)

    def results(self):
        return [host(t) for t in (self.y, self.mean, self.var, self.rm, self.rv, self.d, self.su, self.bu)]


@pytest.mark.parametrize("clip", [100.0, 3.0])      # nothing to clamp; some channels gone over again by the second launch
def test_shared_slices_in_a_replayed_graph(ops, clip):
    import torch
    layer = Layer(ops, torch, 9100, (4, 24, 104, 104))
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        layer.run(clip)
        stream.synchronize()
        want = layer.results()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            layer.run(clip)
        for _ in range(4):
            layer.y.zero_(); layer.d.zero_()
            graph.replay()
            stream.synchronize()
            for got, expected in zip(layer.results(), want):
                assert_bit_exact(got, expected, "replay")
            layer.run(clip)                         # eager work on the same workspace in between
            stream.synchronize()


def test_shared_slices_on_two_streams(ops):
    import torch
    layers = [Layer(ops, torch, 9200 + 10 * i, shape) for i, shape in enumerate([(4, 40, 104, 104), (8, 64, 152, 152)])]
    want = []
    for layer in layers:
        layer.run(3.0)
        torch.cuda.synchronize()
        want.append(layer.results())
    streams = [torch.cuda.Stream() for _ in layers]
    for _ in range(3):
        for layer, stream in zip(layers, streams):
            stream.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(stream):
                for _ in range(4):
                    layer.run(3.0)
        torch.cuda.synchronize()
        for layer, expected in zip(layers, want):
            for got, w in zip(layer.results(), expected):
                assert_bit_exact(got, w, "two streams")


# Slices that a workgroup of 1024 lanes holds: a plain call needs no workspace and never looks at the one it is given, so it
# leaves the same bits whatever that is, and a clipped call that changes nothing leaves them too.
@pytest.mark.parametrize("shape", [(9, 160, 3644), (1, 512, 24800), (4, 512, 4112)], ids=str)
def test_slices_of_one_workgroup_need_no_workspace(ops, shape):
    import torch
    N, C, HW = shape
    layer = Layer(ops, torch, 9300, (N, C, HW, 1))
    layer.run(100.0)                       # statistics to go by
    outcomes = []
    for workspace in (None, torch.zeros(4, device="cuda"), layer.workspace):
        d, su, bu = layer.delta.clone(), torch.ones(C, device="cuda"), torch.ones(C, device="cuda")
        ops.bn_act_backward(d, layer.x, layer.mean, layer.var, layer.scale, layer.bias, su, bu, "leaky", workspace=workspace)
        outcomes.append([host(t) for t in (d, su, bu)])
    d, su, bu = layer.delta.clone(), torch.ones(C, device="cuda"), torch.ones(C, device="cuda")
    ops.bn_act_backward_clipped(d, layer.x, layer.mean, layer.var, layer.scale, layer.bias, su, bu, "leaky", 1e6, 100.0,
                                workspace=layer.workspace)
    outcomes.append([host(t) for t in (d, su, bu)])
    for outcome in outcomes[1:]:
        for got, want in zip(outcome, outcomes[0]):
            assert_bit_exact(got, want, "workspace")


# A member that stops looking (never, within seconds) before the others' figures are there says so in everything it leaves:
# each value is the right one or a NaN, and none is the delta as it came.
@pytest.mark.parametrize("clip", [None, 100.0, 3.0])
def test_a_wait_that_gives_up_leaves_nothing_plausible(ops, clip):
    import torch
    from pixienn_amd import capi
    lib = capi.load()
    layer = Layer(ops, torch, 9400, (16, 6, 152, 152))
    layer.run(100.0)                       # statistics to go by
    norm = torch.zeros(1, device="cuda")

    def backward():
        layer.d.copy_(layer.delta); layer.su.zero_(); layer.bu.zero_(); norm.zero_()
        args = (layer.d, layer.x, layer.mean, layer.var, layer.scale, layer.bias, layer.su, layer.bu, "leaky")
        if clip is None:
            ops.bn_act_backward(*args, workspace=layer.workspace)
        else:
            ops.bn_act_backward_clipped(*args, 1e6, clip, norm, workspace=layer.workspace)
        return [host(t) for t in (layer.d, layer.su, layer.bu, norm)]

    want = backward()
    before = lib.pxh_debug_group_looks(0)
    try:
        got = backward()
    finally:
        lib.pxh_debug_group_looks(before)
    lost = [np.isnan(g) for g in got]
    for g, w, nan in zip(got, want, lost):
        assert_bit_exact(g[~nan], w[~nan], "what was left")
    # where the second launch has nothing else to do, it sees to it that all is lost where anything is
    if clip == 100.0:
        assert len({bool(n) for nan in lost for n in nan.reshape(-1)}) == 1
    for again, w in zip(backward(), want):
        assert_bit_exact(again, w, "the next call")


def test_streams_without_a_mask_have_the_whole_device():
    import torch
    from pixienn_amd import capi
    lib = capi.load()
    all_places = 2 * torch.cuda.get_device_properties(0).multi_processor_count
    for stream in (torch.cuda.default_stream(), torch.cuda.Stream()):
        assert lib.pxh_debug_group_places(stream.cuda_stream) == all_places
