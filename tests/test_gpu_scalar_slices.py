"""GPU parity of the one-launch training passes on odd planes with more than 8192 values per channel (16 and 24
values per lane, one at a time): the checks of the other geometries, with their tolerances, at the first and the
last size of either form and at the first that falls back to three launches, and with enough channels for the
launch behind a clipped backward to walk them."""
import pytest

import test_gpu_clipped_backward as clipped
import test_gpu_epilogue as epilogue
import test_gpu_epilogue_shortcut as shortcut

pytestmark = pytest.mark.gpu

# batch * plane: 8193, 16384 (planes of two), 16385, 24575, 24577; then 300 channels of 13 x 13 and 19 x 19
SHAPES = [(3, 96, 2731), (8192, 96, 2), (5, 97, 3277), (25, 96, 983), (7, 96, 3511), (64, 300, 169), (46, 300, 361)]
# 16 values per lane on both sides of the channels from which an activation with an exponential goes back to three
# launches, and of those from which the form with a shortcut runs two workgroups to a compute unit
MANY = [(49, 256, 169), (49, 257, 169), (64, 512, 169), (64, 513, 169), (64, 1024, 169)]


@pytest.fixture(scope="module")
def ops():
    from pixienn_amd import ops as o
    return o


CASES = [(s, a) for s in SHAPES for a in ("leaky", "mish")] + [(s, a) for s in MANY for a in ("leaky", "mish", "logistic")]


@pytest.mark.parametrize("shape,act", CASES, ids=str)
def test_scalar_slices(ops, oracle, monkeypatch, shape, act):
    for module in (epilogue, clipped, shortcut):
        monkeypatch.setattr(module, "TRAIN_SHAPES", [shape])
    epilogue.test_bn_train_forward_matches_oracle(ops, oracle, act)
    epilogue.test_bn_backward_matches_oracle(ops, oracle, act, False)
    epilogue.test_bn_backward_matches_oracle(ops, oracle, act, True)
    clipped.test_bn_backward_clipped_matches_rescale_clip_then_backward(ops, oracle, act, False)
    # (plain and riding take the same form: no allowance for another order of the sums)
    monkeypatch.setattr(shortcut, "EXTRA_SHAPES", [])
    shortcut.test_training_epilogue_with_shortcut_is_the_two_calls_to_the_bit(ops, act)


# partial sums with 4, 4, 8 and 16 segments to a workgroup, ragged and 128-bit, the last workgroup of a channel short
@pytest.mark.parametrize("shape", [(1, 5, 4100), (3, 90, 10245), (24, 80, 4099), (24, 80, 8200)])
def test_split_of_a_channel(ops, oracle, monkeypatch, shape):
    for module in (epilogue, clipped):
        monkeypatch.setattr(module, "TRAIN_SHAPES", [shape])
    epilogue.test_bn_train_forward_matches_oracle(ops, oracle, "leaky")
    epilogue.test_bn_backward_matches_oracle(ops, oracle, "mish", False)
    clipped.test_bn_backward_clipped_matches_rescale_clip_then_backward(ops, oracle, "leaky", False)
