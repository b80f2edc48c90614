"""Accuracy of the sums in the one-launch training passes on odd planes with more than 8192 values per channel: no
further from 64 bits than the order of the three-launch passes, which the same shapes take with fewer channels.  There
a lane adds its share of one plane's segment of 1024 values in fp32 (every 64th value) and carries on in doubles; that
order is formed here in numpy.  The inputs are centred, so that the rounding of the results to fp32 is far below the
error of the sums."""
import numpy as np
import pytest

from util import F, gpu, host

pytestmark = pytest.mark.gpu


def three_launch_error(values):
    """Error of the sum over each channel of `values` (N, C, HW) in the three-launch order."""
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
