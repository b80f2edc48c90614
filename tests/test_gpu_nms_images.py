"""Suppression image by image at the sizes where its shares change: images that end inside sixteen places, a word of 64 and
the last word there is; batches with 16, 8, 4, 2 and 1 lanes to an image, and more images than lanes; records that are equal
but for their place in the list; more conflicting words than a lane keeps; images without records, and none at all."""
import numpy as np
import pytest

from test_gpu_nms import run, same
from util import random_detections

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from pixienn_amd import ops as o
    return o


def of_sizes(oracle, seed, sizes, classes, clusters, equal=False):
    """Images of `sizes` records around `clusters` centres, shuffled; `equal`: only a few probabilities and orders."""
    rng = np.random.Generator(np.random.Philox(key=seed))
    parts = []
    for image, n in enumerate(sizes):
        rec = random_detections(oracle, seed + image, max(n, 1), 1, classes, clusters)[:n]
        rec["batch"] = image
        parts.append(rec)
    rec = np.concatenate(parts)
    rec = rec[rng.permutation(len(rec))]
    rec["order"] = np.arange(len(rec))
    if equal:
        rec["prob"] = np.round(rec["prob"] * 4) / 4
        rec["order"] = 7
    return rec


EDGES = [1, 15, 16, 17, 0, 31, 33, 63, 64, 65, 127, 129, 1008, 1009, 1023, 1024, 1025]


@pytest.mark.parametrize("clusters", [2, 40])
@pytest.mark.parametrize("size", [n for n in EDGES if n])
def test_one_image(ops, oracle, size, clusters):
    rec = of_sizes(oracle, 50 + size, [size], 5, clusters)
    same(run(ops, rec, 1, 5, 0.45, 3000), oracle.nms(rec, 0.45), size)


@pytest.mark.parametrize("batch", [2, 4, 5, 8, 9, 16, 17, 32, 33, 64, 65, 150])
def test_batches(ops, oracle, batch):
    sizes = [EDGES[(7 * i + batch) % 12] for i in range(batch)]
    rec = of_sizes(oracle, 90 + batch, sizes, 4, 6)
    for capacity in (len(rec) + 600, 20000):
        same(run(ops, rec, batch, 4, 0.45, capacity), oracle.nms(rec, 0.45), (batch, capacity))


def test_all_edges_at_once(ops, oracle):
    rec = of_sizes(oracle, 7, EDGES, 3, 9)
    same(run(ops, rec, len(EDGES), 3, 0.3, len(rec)), oracle.nms(rec, 0.3), "edges")


@pytest.mark.parametrize("sizes", [[100], [600, 64, 300], [40] * 20])
def test_equal_keys_keep_input_order(ops, oracle, sizes):
    rec = of_sizes(oracle, 11 + len(sizes), sizes, 3, 12, equal=True)
    # told apart by their class and box; the list's order decides
    same(run(ops, rec, len(sizes), 3, 0.45, 4000), oracle.nms(rec, 0.45), sizes)


def test_no_records(ops, oracle):
    rec = of_sizes(oracle, 3, [4], 3, 2)[:0]
    assert len(run(ops, rec, 9, 3, 0.45, 3000)) == 0


@pytest.mark.parametrize("sizes", [[1 + 7 * i % 90 for i in range(300)], [500 - i for i in range(40)]], ids=["many", "long"])
def test_more_quarters_of_blocks_than_workgroups(ops, oracle, sizes):
    rec = of_sizes(oracle, 21, sizes, 4, 8)
    assert 4 * sum(-(-n // 64) for n in sizes) > 1024
    same(run(ops, rec, len(sizes), 4, 0.45, len(rec) + 9000), oracle.nms(rec, 0.45), len(sizes))
