"""The gradients of the activations with an exponential, over their whole range and its edges, against 64 bits."""
import numpy as np
import pytest
import torch

from pixienn_amd import ops

pytestmark = pytest.mark.gpu

EDGES = np.array([0.0, 20.0, -4.4, -20.0, -64.0, -87.0, -88.9, -104.0, -110.0, -200.0, -1e30, 20.5, 88.9, 200.0, 1e30])


def _exact(act, x):
    with np.errstate(over="ignore", invalid="ignore"):
        s = np.where(x > -700, 1.0 / (1.0 + np.exp(-np.maximum(x, -700.0))), 0.0)
        if act == "logistic":
            return s * (1.0 - s)
        if act == "swish":
            return np.where(x < -700, 0.0, s + np.maximum(x, -700.0) * s * (1.0 - s))
        if act == "softplus":
            return s
        t = np.tanh(np.log1p(np.exp(np.minimum(np.maximum(x, -700.0), 40.0))))
        return np.where(x > 40, 1.0, t + np.maximum(x, -700.0) * (1.0 - t * t) * s)


# in units of 2^-24.  A logistic is formed from an exponential good to 1.5 units in its last place, a rounded sum and a
# quotient good to one: 4 of its value, 5 with its complement's rounding.  swish multiplies by x and adds three terms of up
# to 1.3 (each rounded): 6 + 2 |x| s.  mish takes tanh(softplus) from u = float(1 + exp(x)): a unit of u moves it by as much
# again, and 1 - t^2, rounded to 2^-24, is multiplied by x.
def _bound(act, x, s):
    unit = 2.0 ** -24
    if act == "swish":
        return unit * (6.0 + 4.0 * np.abs(x) * s)
    if act == "mish":
        return unit * (6.0 + 4.0 * np.minimum(np.abs(x), 20.0))
    return unit * 5.0 * np.maximum(s, 2.0 ** -126)


@pytest.mark.parametrize("act", ["logistic", "swish", "mish", "softplus"])
def test_gradient_over_the_whole_range(act):
    x = np.concatenate([np.linspace(-120.0, 120.0, 100001), np.linspace(-25.0, 25.0, 100003), EDGES,
                        np.nextafter(np.float32(EDGES), np.float32(-np.inf)), np.nextafter(np.float32(EDGES), np.float32(np.inf))])
    x = x.astype(np.float32)
    d = torch.ones(x.size, device="cuda")
    got = ops.gradient(act, torch.from_numpy(x).cuda(), d).cpu().numpy().astype(np.float64)
    xd = x.astype(np.float64)
    s = np.where(xd > -700, 1.0 / (1.0 + np.exp(-np.clip(xd, -700.0, 700.0))), 0.0)
    err = np.abs(got - _exact(act, xd))
    # (exponentials below the smallest normal float have fewer digits)
    bad = err > _bound(act, xd, s) + 2.0 ** -126 * np.maximum(1.0, np.abs(xd)) * (xd < -80)
    assert not bad.any(), (act, x[bad][:5], got[bad][:5], err[bad][:5])


@pytest.mark.parametrize("act,want", [("logistic", (0.0, 0.0)), ("softplus", (1.0, 0.0)), ("mish", (1.0, np.nan)),
                                      ("swish", (np.nan, np.nan))])
def test_gradient_of_infinities_and_nan(act, want):
    x = torch.tensor([np.inf, -np.inf, np.nan], device="cuda")
    got = ops.gradient(act, x, torch.ones(3, device="cuda")).cpu().numpy()
    assert np.array_equal(got[:2], np.float32(want), equal_nan=True) and np.isnan(got[2]), got
