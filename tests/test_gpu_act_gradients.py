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


# in units of 2^-24.  An exponential is good to one unit in its last place, 2; a logistic s from it, with a rounded sum and a
# quotient good to one, to 4 of its value, 5 with its complement's rounding.
# swish adds x * s and s * (1 - x * s): 4 + 1 of |x| s and 4 + 0.5 + 1 of s below -14, where the second factor rounds to 1 and
# nothing cancels, and half a unit of the sum: 6 (1 + |x|) s.  Above, terms of up to 1.3 (each rounded) and 4 |x| s.
# mish takes t = tanh(softplus) from u = float(1 + exp(x)), whose rounding is half a unit in its last place, 1, and moves t by
# no more; the quotient adds 5 of t.  1 - t^2 is then off by 2 t (1 + 5 t) + 1, times |x| s, s and the products' roundings by 7 of
# |x| s, and the sum by one of t: 1 + 6 t + |x| s (2 t (1 + 5 t) + 8).  Below -20 t is the exponential itself, and so is s:
# 6 (1 + |x|) s.  Above 0 the terms are of the order of 1 and |x|.
def _bound(act, x, s):
    unit, size = 2.0 ** -24, np.abs(x)
    tail = 6.0 * (1.0 + size) * s
    if act == "swish":
        return unit * np.where(x < -14.0, tail, 6.0 + 4.0 * size * s)
    if act == "mish":
        t = np.tanh(np.log1p(np.exp(np.clip(x, -700.0, 40.0))))
        middle = 1.0 + 6.0 * t + size * s * (2.0 * t * (1.0 + 5.0 * t) + 8.0)
        return unit * np.where(x < -20.0, tail, np.where(x < 0.0, middle, 6.0 + 4.0 * np.minimum(size, 20.0)))
    return unit * 5.0 * s


# (exponentials below the smallest normal float, from -87 on, have fewer digits: a unit of the smallest subnormal for each term)
def _fewer_digits(x):
    return 2.0 ** -149 * 4.0 * (1.0 + np.minimum(np.abs(x), 200.0)) * (x < -87.0)


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
    bound = _bound(act, xd, s) + _fewer_digits(xd)
    # in the tail a gradient of 0 or of the wrong sign is beyond the bound
    if act in ("swish", "mish"):
        tail = (xd < -20.0) & (xd > -87.0)
        assert tail.sum() > 10000 and np.all(bound[tail] < 1e-5 * np.abs(_exact(act, xd[tail])))
    bad = err > bound
    assert not bad.any(), (act, x[bad][:5], got[bad][:5], err[bad][:5])


@pytest.mark.parametrize("act,want", [("logistic", (0.0, 0.0)), ("softplus", (1.0, 0.0)), ("mish", (1.0, np.nan)),
                                      ("swish", (np.nan, np.nan))])
def test_gradient_of_infinities_and_nan(act, want):
    x = torch.tensor([np.inf, -np.inf, np.nan], device="cuda")
    got = ops.gradient(act, x, torch.ones(3, device="cuda")).cpu().numpy()
    assert np.array_equal(got[:2], np.float32(want), equal_nan=True) and np.isnan(got[2]), got
