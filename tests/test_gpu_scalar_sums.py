"""Accuracy of the sums in the training passes on odd planes and on planes of fewer values than a vector: every value is rounded
to fp32 once, as a term, and added in doubles, whatever form takes the slice.  What the passes leave is then the rounded value of
the same sums in 64 bits: half a unit in the last place, and the rounding of the doubles themselves."""
import numpy as np
import pytest

from util import F, gpu, host

pytestmark = pytest.mark.gpu

# one value a step: up to 64, 1024, 2048, 6144, 8192, 16384 and 24576 values; then vectors in one launch, in several, and in groups
SHAPES = [(50, 97, 1), (300, 5, 3), (513, 97, 2), (1023, 70, 2), (2048, 96, 3), (2731, 96, 3), (8000, 96, 3),
          (64, 256, 169), (46, 256, 361), (200, 256, 63), (3, 7, 2051), (40, 3, 5003), (68, 3, 257), (2, 23, 25625),
          (3000, 3, 5), (260, 3, 63), (250, 3, 65), (130, 3, 129)]


def check(got, want, terms, what):
    """`terms`: sum of the magnitudes that were added (in the result's scale)."""
    error = np.abs(np.asarray(got, np.float64) - want)
    bound = 2.0 ** -24 * np.abs(want) * (1.0 + 1e-6) + 1e-13 * terms + 2.0 ** -149
    assert (error <= bound).all(), (what, float(np.max(error / bound)))


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_terms_are_added_in_doubles(shape):
    from pixienn_amd import ops
    N, C, HW = shape
    rng = np.random.Generator(np.random.Philox(key=N * HW))
    x, delta = (rng.standard_normal((N, C, HW)).astype(F) for _ in range(2))
    count = N * HW
    zero, one = np.zeros(C, F), np.ones(C, F)

    def wide(a):
        return a.astype(np.float64).sum((0, 2))

    # forward: relative to the channel's first value
    shift = x[0:1, :, 0:1]
    d = x - shift
    square = d * d
    gx = gpu(x.reshape(N, C, HW, 1))
    mean, var = gpu(zero), gpu(zero)
    ops.bn_train_act_forward(gx, gpu(np.zeros((N, C, HW, 1), F)), mean, var, gpu(zero), gpu(one), gpu(one), gpu(zero), "linear")
    m = wide(d) / count
    check(host(mean), shift.reshape(C).astype(np.float64) + m, wide(np.abs(d)) / count + np.abs(shift.reshape(C)), "mean")
    check(host(var), (wide(square) - wide(d) * m) / count, 2.0 * wide(square) / count, "variance")

    # backward: plain, with the norm, and clamped throughout
    denom = 1.0 + float(F(1e-5))
    centre = rng.standard_normal(C).astype(F) * F(0.25)
    for mode in ("plain", "norm", "clamped"):
        su, bu, norm = gpu(zero), gpu(zero), gpu(np.zeros(1, F))
        args = [gpu(delta.reshape(N, C, HW, 1)), gx, gpu(centre), gpu(one), gpu(one), gpu(zero), su, bu, "linear"]
        if mode == "plain":
            ops.bn_act_backward(*args)
        else:
            ops.bn_act_backward_clipped(*args, 1e9, 0.5 if mode == "clamped" else 0.0, norm)
        t = np.clip(delta, F(-0.5), F(0.5)) if mode == "clamped" else delta
        product = t * (x - centre.reshape(1, C, 1))
        check(host(bu), wide(t), wide(np.abs(t)), mode + " bias")
        check(host(su), wide(product) / denom, wide(np.abs(product)), mode + " scale")
        if mode != "plain":
            total = np.sqrt(np.sum(wide(delta * delta)))
            check(host(norm), total, total, mode + " norm")


# A looser bound that other geometries are held to as well (test_gpu_small_slices.py): no further from 64 bits than partial sums
# in fp32.  The inputs are centred, so that the rounding of the results to fp32 is far below the error of the sums.
def three_launch_error(values):
    """Error of the sum over each channel of `values` (N, C, HW) where a lane adds its share of a plane's segment of 1024 values
    (every 64th) in fp32 and carries on in doubles: launches that take one value a step."""
    n, c, hw = values.shape
    error = np.zeros(c)
    for s0 in range(0, hw, 1024):
        part = values[:, :, s0:s0 + 1024]
        steps = -(-part.shape[2] // 64)
        lanes = np.zeros((n, c, steps * 64), F)
        lanes[:, :, :part.shape[2]] = part
        lanes = lanes.reshape(n, c, steps, 64)
        acc = np.zeros((n, c, 64), F)
        for k in range(steps):
            acc += lanes[:, :, k]
        error += (acc.astype(np.float64) - lanes.astype(np.float64).sum(2)).sum((0, 2))
    return error


# (the root mean square of 256 channels' errors is known to one part in 22: 1.1 is two of those)
MARGIN = 1.1


def rms(v):
    return float(np.sqrt(np.mean(np.square(v))))


@pytest.mark.parametrize("shape", [(64, 256, 169), (46, 256, 361), (4000, 256, 3), (200, 256, 63)], ids=str)
def test_sums_are_as_close_as_the_three_launches(shape):
    from pixienn_amd import ops
    N, C, HW = shape
    rng = np.random.Generator(np.random.Philox(key=N * HW))
    x = rng.standard_normal((N, C, HW))
    x = (x - x.mean((0, 2), keepdims=True)).astype(F)
    count = N * HW
    if count <= 16384:
        mean, var = gpu(np.zeros(C, F)), gpu(np.zeros(C, F))
        gx = gpu(x.reshape(N, C, HW, 1))
        ops.bn_train_act_forward(gx, gpu(np.zeros((N, C, HW, 1), F)), mean, var, gpu(np.zeros(C, F)), gpu(np.ones(C, F)),
                                 gpu(np.ones(C, F)), gpu(np.zeros(C, F)), "linear")
        d = x - x[0:1, :, 0:1]
        exact = x[0, :, 0].astype(np.float64) + d.astype(np.float64).sum((0, 2)) / count
        got = rms(host(mean) - exact) * count
        assert got <= MARGIN * rms(three_launch_error(d)) + 1e-10 * count, "forward"
    # the two sums of the backward: of the delta, and of the delta times x - mean (here 0, exactly)
    delta = rng.standard_normal((N, C, HW))
    for _ in range(2):
        delta -= delta.mean((0, 2), keepdims=True)
        delta -= (delta * x).sum((0, 2), keepdims=True) / (x.astype(np.float64) ** 2).sum((0, 2), keepdims=True) * x
    delta = delta.astype(F)
    zero, one = np.zeros(C, F), np.ones(C, F)
    su, bu = gpu(zero), gpu(zero)
    ops.bn_act_backward(gpu(delta.reshape(N, C, HW, 1)), gpu(x.reshape(N, C, HW, 1)), gpu(zero), gpu(one), gpu(one),
                        gpu(zero), su, bu, "linear")
    product = delta * x
    for name, got, values in (("bias", host(bu).astype(np.float64), delta),
                              ("scale", host(su).astype(np.float64) * (1.0 + float(F(1e-5))), product)):
        error = rms(got - values.astype(np.float64).sum((0, 2)))
        assert error <= MARGIN * rms(three_launch_error(values)) + 1e-10 * count, name
