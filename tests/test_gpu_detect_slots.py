"""GPU parity of the thresholded compaction at the number of passing slots where a workgroup changes over, at class counts
around a wavefront, and where the records run out of room."""
import numpy as np
import pytest

from pixienn_amd import workloads as wl
from util import F, assert_bit_exact, assert_close, gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from pixienn_amd import ops as o
    return o


def decoded_head(seed, N, A, K, W, slots):
    """A decoded head in which the first `slots` of a shuffle of the first 512 slots, and every 97th behind, pass 0.5."""
    rng = np.random.default_rng(seed)
    v = rng.uniform(0.0, 0.45, (N, A, K + 5, W * W)).astype(F)
    v[:, :, 4] = 0.1
    objectness = v[:, :, 4].reshape(-1).copy()
    passing = np.concatenate([rng.permutation(512)[:slots], np.arange(512, N * A * W * W, 97)])
    objectness[passing] = 0.9
    v[:, :, 4] = objectness.reshape(N, A, W * W)
    hot = rng.uniform(size=v[:, :, 5:].shape) < 0.1
    v[:, :, 5:][hot] = 0.8
    v[:, :, 5, ::2] = 0.9        # the first and the last class too
    v[:, :, -1, ::3] = 0.9
    return v.reshape(N, A * (K + 5), W, W)


@pytest.mark.parametrize("classes", [1, 64, 65, 80, 129, 300])
@pytest.mark.parametrize("slots", [0, 1, 8, 32, 33, 512])
def test_passing_slots_of_a_workgroup(ops, oracle, classes, slots):
    N, A, W = 2, 3, 20
    masks, anchors = [0, 1, 2], wl.YOLOV3_ANCHORS[:6]
    head = decoded_head(classes * 1000 + slots, N, A, classes, W, slots)
    cfg, keep = oracle.yolo_cfg(N, W, W, classes, masks, anchors, 640, 640)
    for capacity in (1 << 18, 40):
        want, found_w = oracle.yolo_detections(cfg, head, 0.5, 1 << 18)
        got, found_g = ops.yolo_detections(gpu(head), N, masks, anchors, classes, W, W, 640, 640, 0.5, capacity)
        assert found_g == found_w > 0 and len(got) == min(found_w, capacity)
        if capacity < found_w:
            assert len(set(got["order"])) == capacity and set(got["order"]) <= set(want["order"])
            want = want[np.isin(want["order"], got["order"])]
        for k in ("order", "batch", "class_index"):
            assert np.array_equal(got[k], want[k]), k
        assert_bit_exact(got["prob"], want["prob"], "probabilities")
        for k in ("x", "y", "w", "h"):
            assert_close(got[k], want[k], 1e-5, 1.0, k)
