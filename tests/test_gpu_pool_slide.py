"""Bit-exact parity of the max-pools whose windows move by one cell: rows and columns that end inside a run of four, planes
of fewer cells than a vector, several planes to a tile, strips, no padding, windows wider than the plane; with ties, NaN, -inf
and tensors off a 16-byte boundary, and indexes that name no cell of their window."""
import numpy as np
import pytest
import torch

import test_gpu_layers as layers
from pixienn_amd import workloads as wl
from util import F, assert_bit_exact, gpu, host

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from pixienn_amd import ops as o
    return o


# batch, channels, height, width, window, padding
CASES = [(1, 1, 1, 1, 3, 2), (3, 1, 1, 3, 3, 2), (1, 5, 2, 2, 5, 4), (1, 3, 13, 13, 13, 12), (1, 2, 12, 12, 13, 12), (2, 1, 40, 9, 9, 8),
         (2, 1, 9, 8, 9, 8), (37, 61, 19, 19, 5, 4), (1, 1300, 13, 13, 3, 2), (2, 3, 17, 18, 5, 0), (1, 4, 30, 30, 13, 0), (2, 3, 61, 47, 3, 1),
         (1, 2, 91, 130, 9, 8), (1, 2, 300, 301, 3, 2), (1, 2, 67, 95, 5, 4), (5, 7, 14, 15, 2, 1),
         # tiles of 256 outputs (a value to a lane) and 272, of 528 and more: one plane, and several small ones
         (1, 3, 16, 16, 3, 2), (1, 3, 16, 17, 5, 4), (1, 3, 22, 24, 9, 8), (1, 2, 26, 23, 5, 4), (2, 2100, 13, 13, 9, 8), (1, 4100, 12, 12, 13, 12),
         (1, 1, 1, 1, 2, 1), (3, 5, 1, 2, 2, 1), (2, 3, 3, 1, 2, 1), (1, 4, 13, 13, 2, 1), (7, 11, 26, 23, 2, 1), (1, 1, 8, 8, 2, 1)]


@pytest.mark.parametrize("case", CASES, ids=str)
def test_slide(ops, oracle, case):
    n, c, h, w, k, p = case
    x = wl.normal(2100 + h * w, (n, c, h, w))
    layers.run_maxpool(ops, oracle, x, k, 1, p, 2200)
    layers.run_maxpool(ops, oracle, np.round(x).astype(F) * F(-0.0 if k == 3 else 1.0), k, 1, p, 2201)
    if h * w > 30:
        flat = x.reshape(-1)
        flat[::97] = -np.inf
        x[:, :, : h // 2] = -np.inf
        layers.run_maxpool(ops, oracle, x, k, 1, p, 2202)
        flat[5::89] = np.nan
        layers.run_maxpool(ops, oracle, x, k, 1, p, 2203)


@pytest.mark.parametrize("k", [2, 3, 5, 13])
def test_off_a_boundary(ops, k):
    """Tensors that begin one value behind a 16-byte boundary: the results of those that begin on one."""
    found = []
    for at in (0, 1):
        def tensor(seed, kind=F):
            values = wl.normal(seed, (3, 7, 19, 21)).astype(kind)
            place = torch.zeros(values.size + 4, device="cuda", dtype=torch.float32 if kind is F else torch.int32)
            return place[at:at + values.size].view(values.shape).copy_(torch.from_numpy(values))
        x, y, delta, grad, index = tensor(1), tensor(2), tensor(3), tensor(4), tensor(5, np.int32)
        ops.maxpool_forward(x, y, index, k, 1, k - 1)
        ops.maxpool_backward(delta, index, grad, k, 1, k - 1)
        found.append([host(t) for t in (y, index, grad)])
    for a, b in zip(*found):
        assert_bit_exact(a, b)


@pytest.mark.parametrize("k,shape", [(3, (2, 3, 7, 6)), (5, (1, 3, 19, 19)), (9, (1, 1, 40, 60)), (13, (2, 2, 14, 13))])
def test_foreign_indexes(ops, k, shape):
    """Indexes drawn from the whole tensor and beyond: only those that name a cell of their own window count."""
    n, c, h, w = shape
    rng = np.random.Generator(np.random.Philox(key=k))
    cells = n * c * h * w
    index = rng.integers(-3, cells + 3, cells).astype(np.int32)
    own = np.arange(cells, dtype=np.int64)
    near = rng.random(cells) < 0.7
    index[near] = (own + rng.integers(-k, k, cells) + w * rng.integers(-k, k, cells))[near]
    delta, grad = wl.normal(1, shape), wl.normal(2, shape)
    want = grad.reshape(-1).copy()
    origin = -((k - 1) // 2)
    for o in range(cells):
        at = int(index[o])
        if not 0 <= at < cells or at // (h * w) != o // (h * w):
            continue
        ty, tx = at // w % h - o // w % h - origin, at % w - o % w - origin
        if 0 <= ty < k and 0 <= tx < k:
            want[at] = want[at] + delta.reshape(-1)[o]
    got = gpu(grad)
    ops.maxpool_backward(gpu(delta), gpu(index.reshape(shape)), got, k, 1, k - 1)
    assert_bit_exact(host(got).reshape(-1), want)
