"""GPU parity of the one-launch training passes in their small forms (few lanes, two to eight steps each) and of odd planes: the checks of
the other geometries, with their tolerances, at the last size of each form and the first of the next, with fewer channels
than the other one-launch forms take and with more than the launch behind a clipped backward has workgroups; then the
accuracy of their sums against 64 bits."""
import numpy as np
import pytest

import test_gpu_clipped_backward as clipped
import test_gpu_epilogue as epilogue
import test_gpu_epilogue_shortcut as shortcut
import test_gpu_scalar_sums as sums

pytestmark = pytest.mark.gpu

# vectors of a slice: 1, 128 and 129, 256 and 257, 512 and 513 (where a smooth activation's backward leaves), 1024 and
# 1025, 2048, 2049 (256 channels, then 257, which leave), 4096 and 4097
VECTORS = [(1, 3, 4), (2, 5, 256), (3, 5, 172), (16, 270, 64), (1, 97, 1028), (2, 96, 1024), (27, 97, 76), (8, 7, 512),
           (25, 7, 164), (32, 264, 256), (3, 256, 2732), (3, 257, 2732), (4, 20, 4096), (1, 20, 16388)]
# odd planes: 1 channel of one value a plane, 256 values and 257, 1024 and 1025, 2048 and 2049, 4095 and 4097, 6143 and 6145
SCALARS = [(5, 1, 1), (256, 3, 1), (1, 270, 257), (8, 5, 127), (5, 5, 205), (2048, 4, 1), (3, 300, 683), (5, 97, 819),
           (17, 9, 241), (2, 100, 2049), (1, 9, 6143), (5, 97, 1229)]


@pytest.fixture(scope="module")
def ops():
    from pixienn_amd import ops as o
    return o


@pytest.mark.parametrize("act", ["leaky", "mish"])
@pytest.mark.parametrize("shape", VECTORS + SCALARS, ids=str)
def test_small_slices(ops, oracle, monkeypatch, shape, act):
    for module in (epilogue, clipped, shortcut):
        monkeypatch.setattr(module, "TRAIN_SHAPES", [shape])
    epilogue.test_bn_train_forward_matches_oracle(ops, oracle, act)
    epilogue.test_bn_backward_matches_oracle(ops, oracle, act, False)
    epilogue.test_bn_backward_matches_oracle(ops, oracle, act, True)
    clipped.test_bn_backward_clipped_matches_rescale_clip_then_backward(ops, oracle, act, False)
    # (plain and riding take the same form: no allowance for another order of the sums)
    monkeypatch.setattr(shortcut, "EXTRA_SHAPES", [])
    shortcut.test_training_epilogue_with_shortcut_is_the_two_calls_to_the_bit(ops, act)


def vector_error(values):
    """Error of the sum over each channel of `values` (N, C, HW) where the four values of a vector are added in fp32 and
    everything else exactly: what any form that takes 128 bits at a time starts from."""
    v = values.reshape(values.shape[0], values.shape[1], -1, 4)
    acc = ((v[..., 0] + v[..., 1]) + v[..., 2]) + v[..., 3]
    return (acc.astype(np.float64) - v.astype(np.float64).sum(3)).sum((0, 2))


@pytest.mark.parametrize("shape", [(2, 256, 100), (8, 256, 1600), (8, 256, 169), (16, 256, 361)], ids=str)
def test_sums_are_as_close_as_the_three_launches(monkeypatch, shape):
    if shape[2] % 4 == 0:
        monkeypatch.setattr(sums, "three_launch_error", vector_error)
    sums.test_sums_are_as_close_as_the_three_launches(shape)
