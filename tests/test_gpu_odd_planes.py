"""GPU parity of the one-launch training passes on odd planes, whose vectors end with their plane: the checks of the other
geometries, with their tolerances, at the last size of each form and the first of the next, with one, two and three values
left in a plane's last vector, and on tensors off a 16-byte boundary; then a shortcut whose source is the output itself."""
import numpy as np
import pytest
import torch

import test_gpu_clipped_backward as clipped
import test_gpu_epilogue as epilogue
import test_gpu_epilogue_shortcut as shortcut
from util import F, assert_bit_exact, gpu, host

pytestmark = pytest.mark.gpu

# 64 values of a slice (one to a lane) and 65; vectors of a slice: 1, 64 and 65, 128 and 130, 256 and 259, 768 and 771, 1536 (up to 512 channels and beyond) and 1539, 2049, 3072 and
# 3075, 4096 and 4100 (few channels, which leave, and many), 6144 and 6148, 300 channels that are walked; then values of
# planes below four, the last of each form and the first of the next: 256, 1024, 2048, 4096, 6144 (few channels, which leave, and
# many), 8192, 16384, 24576; then more than 512 channels: 256 vectors and 260, 512 and 516, 1024 and 1028, and fewer: 512 and 514, 1024
# and 1028
SHAPES = [(1, 3, 4), (1, 5, 5), (7, 97, 9), (64, 97, 1), (13, 97, 5), (64, 97, 7), (65, 97, 7), (32, 97, 7), (13, 97, 17), (128, 96, 6), (37, 96, 25), (256, 97, 9), (257, 96, 9), (512, 96, 10),
          (384, 520, 13), (513, 96, 9), (683, 96, 11), (1024, 96, 9), (1025, 300, 11), (1024, 5, 14), (1025, 5, 15), (1025, 96, 15),
          (1536, 96, 15), (1537, 96, 14), (128, 97, 2), (129, 97, 2),
          (512, 5, 2), (513, 97, 2), (2048, 96, 1), (683, 97, 3), (2048, 97, 2), (2049, 97, 2), (2048, 5, 3), (3073, 5, 2), (3073, 96, 2),
          (4096, 96, 2), (2731, 96, 3), (8192, 96, 2), (5462, 96, 3), (8192, 96, 3), (8193, 96, 3),
          (64, 520, 13), (65, 520, 13), (128, 520, 13), (129, 520, 13), (256, 520, 13), (257, 520, 13), (256, 97, 7), (257, 97, 7), (256, 97, 13), (257, 97, 13)]


@pytest.fixture(scope="module")
def ops():
    from pixienn_amd import ops as o
    return o


@pytest.mark.parametrize("act", ["leaky", "mish"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_odd_planes(ops, oracle, monkeypatch, shape, act):
    for module in (epilogue, clipped, shortcut):
        monkeypatch.setattr(module, "TRAIN_SHAPES", [shape])
    epilogue.test_bn_train_forward_matches_oracle(ops, oracle, act)
    epilogue.test_bn_backward_matches_oracle(ops, oracle, act, False)
    epilogue.test_bn_backward_matches_oracle(ops, oracle, act, True)
    clipped.test_bn_backward_clipped_matches_rescale_clip_then_backward(ops, oracle, act, False)
    monkeypatch.setattr(shortcut, "EXTRA_SHAPES", [])
    shortcut.test_training_epilogue_with_shortcut_is_the_two_calls_to_the_bit(ops, act)


# three launches: a segment of 1024 values that ends one, two and three values behind its last whole vector, and one that
# holds a plane's last value alone; then slices of several members, and groups: two members, the last vector of a plane in another
# share than the one in front of it, channels that leave workgroups over, small planes and large ones
# (the pass behind the sums finishes the channels from planes of 256 values on, and up to 256 partial sums a channel: both
# sides, aligned and odd)
SPLIT = [(1, 5, 1025), (3, 7, 2051), (2, 9, 1022), (40, 3, 5003), (68, 3, 255), (68, 3, 257), (65, 4, 256), (1030, 2, 260), (1, 1, 4 * 1024 * 257),
         (1, 9, 16388), (3, 4, 5468),
         # one value a step, up to 64 values of a plane and 128 before an exponential, and vectors
         # few channels past 3072 vectors, which leave before or behind mish alone
         (96, 5, 125), (97, 5, 125), (193, 7, 63),
         (3000, 2, 5), (260, 2, 63), (250, 2, 65), (130, 2, 127), (130, 2, 129)]
GROUPS = [(1, 90, 16385), (2, 23, 25 * 1025), (3, 70, 10243), (8, 96, 10395), (500, 60, 45), (700, 23, 77), (2, 23, 160001)]


@pytest.mark.parametrize("act", ["leaky", "mish"])
@pytest.mark.parametrize("shape", SPLIT + GROUPS, ids=str)
def test_longer_slices(ops, oracle, monkeypatch, shape, act):
    for module in (epilogue, clipped):
        monkeypatch.setattr(module, "TRAIN_SHAPES", [shape])
    epilogue.test_bn_train_forward_matches_oracle(ops, oracle, act)
    epilogue.test_bn_backward_matches_oracle(ops, oracle, act, False)
    epilogue.test_bn_backward_matches_oracle(ops, oracle, act, True)
    clipped.test_bn_backward_clipped_matches_rescale_clip_then_backward(ops, oracle, act, False)


@pytest.mark.parametrize("shape", [(3, 20, 13, 13), (2, 5, 25, 41), (7, 3, 1, 5), (5, 3, 1, 3)], ids=str)
@pytest.mark.parametrize("threshold", [1e9, 1e-3])
def test_bias_backward(ops, shape, threshold):
    """d' = (rescaled delta) * the gradient in place, and its sums, against 64 bits: a handful of roundings a value."""
    (x, pre, delta), (_, _, _, _, _, updates) = layer(shape, 1)
    before = [host(t).astype(np.float64) for t in (delta, pre, updates)]
    ops.bias_act_backward_clipped(delta, pre, updates, "leaky", threshold, 0.0)
    norm = np.sqrt(np.sum(before[0] ** 2))
    want = before[0] * (threshold / norm if norm > threshold else 1.0) * np.where(before[1] > 0, 1.0, np.float64(F(0.1)))
    assert np.all(np.abs(host(delta) - want) <= 8 * 2.0 ** -24 * np.abs(want))
    total = before[2] + want.sum((0, 2, 3))
    room = 8 * 2.0 ** -24 * (np.abs(want).sum((0, 2, 3)) + np.abs(total))
    assert np.all(np.abs(host(updates) - total) <= room)


def layer(shape, offset, seed=3):
    """x, y, delta and the parameters of a layer, the tensors `offset` values off a 16-byte boundary."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    n = int(np.prod(shape))

    def tensor():
        place = torch.empty(n + 4, device="cuda")[offset:offset + n].view(shape)
        return place.copy_(torch.empty(n, device="cuda").normal_(generator=g).view(shape))

    return [tensor() for _ in range(3)], [torch.empty(shape[1], device="cuda").normal_(generator=g).abs_() + 0.5 for _ in range(6)]


@pytest.mark.parametrize("offset", [1, 2, 3])
@pytest.mark.parametrize("shape", [(6, 100, 4, 4), (40, 96, 13, 13)], ids=str)
def test_tensors_off_a_boundary(ops, shape, offset):
    """The same values as from tensors that begin on a word of their own: odd planes to the bit (one form), others within
    the rounding of sums in another order."""
    found = []
    for at in (offset, 0):
        (x, y, delta), (scale, bias, rm, rv, su, bu) = layer(shape, at)
        mean, var = torch.zeros_like(rm), torch.zeros_like(rm)
        source = layer(shape, at)[0][0].clone()
        ops.bn_train_act_forward(x, y, mean, var, rm, rv, scale, bias, "leaky")
        ops.bn_act_backward_clipped(delta, x, mean, var, scale, bias, su, bu, "leaky", 1e-3, 0.0)
        assert torch.equal(x, source)
        found.append([host(t) for t in (y, mean, var, rm, rv, su, bu, delta)])
    for a, b in zip(*found):
        if shape[2] % 2:
            assert_bit_exact(a, b)
        else:
            assert np.max(np.abs(a.astype(np.float64) - b)) <= 1e-5 * np.sqrt(np.mean(b.astype(np.float64) ** 2))


@pytest.mark.parametrize("act", ["leaky", "mish"])
@pytest.mark.parametrize("shape", [(3, 7, 45, 153), (2, 5, 96, 96), (64, 100, 5, 5)], ids=str)
def test_forward_in_place(ops, shape, act):
    """y may be x, also with a shortcut on top of it."""
    found = []
    for alias in (False, True):
        (x, y, source), (scale, bias, rm, rv, _, _) = layer(shape, 0)
        mean, var = torch.zeros_like(rm), torch.zeros_like(rm)
        out, riding = (x, x.clone()) if alias else (y, torch.empty_like(x))
        start = x.clone()
        ops.bn_train_act_forward(x, out, mean, var, rm, rv, scale, bias, act)
        at = start if not alias else riding
        ops.bn_train_act_shortcut_forward(at, riding if not alias else at, mean, var, rm, rv, scale, bias, act, source)
        found.append([host(t) for t in (out, riding, mean, var, rm, rv)])
    for a, b in zip(*found):
        assert_bit_exact(a, b)


@pytest.mark.parametrize("shape", [(64, 100, 5, 5), (33, 520, 13, 13), (40, 100, 19, 19), (3, 7, 45, 153)], ids=str)
def test_shortcut_source_is_the_output(ops, shape):
    found = []
    for alias in (False, True):
        (x, y, source), (scale, bias, rm, rv, _, _) = layer(shape, 0)
        mean, var = torch.zeros_like(rm), torch.zeros_like(rm)
        out = source if alias else y
        ops.bn_train_act_shortcut_forward(x, out, mean, var, rm, rv, scale, bias, "leaky", source)
        found.append(host(out))
    assert_bit_exact(*found)
