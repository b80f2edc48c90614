"""GPU parity of the device-resident tensor tables (pxh_tensor_table_*): Adam, SGD, fill and
rescale + clip over all tensors of a table in one launch (two for rescale + clip) must leave every
tensor exactly as the single-tensor entry points do -- which the other tests hold to the CPU checker --
bit for bit, for tensors of every size class, more tensors than the by-value tables hold, empty
tensors and one that is not 16-byte aligned."""
import numpy as np
import pytest

from pixienn_amd import workloads as wl
from test_gpu_yolo_adam import MULTI_SIZES, _multi_tensors
from util import F, assert_bit_exact, gpu, host

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from pixienn_amd import ops as o
    return o


def test_adam_table_gives_every_tensor_what_the_single_call_gives(ops):
    flags = [i % 3 == 0 for i in range(len(MULTI_SIZES))]
    _, gw = _multi_tensors(6000, 0.02)
    _, gd = _multi_tensors(6100, 1e-3)
    _, gm = _multi_tensors(6200, 1e-4)
    _, gv = _multi_tensors(6300, 1e-4)
    gv = [t.abs_() for t in gv]
    single = [[t.clone() for t in group] for group in (gw, gd, gm, gv)]
    table = ops.TensorTable([gw, gd, gm, gv], flags)
    assert table.count == sum(1 for n in MULTI_SIZES if n)
    for step in (1, 2, 3):
        table.adam_update(16, step, 1e-3, 0.9, 0.999, 1e-8, 5e-4)
        for i, n in enumerate(MULTI_SIZES):
            if n:
                ops.adam_update(single[0][i], single[1][i], single[2][i], single[3][i], 16, step, 1e-3, 0.9, 0.999, 1e-8,
                                5e-4, flags[i])
        for i, n in enumerate(MULTI_SIZES):      # a fresh gradient on both sides
            if n:
                g = gpu(wl.normal(6400 + 10 * step + i, n, std=1e-3))
                gd[i] += g; single[1][i] += g
    for name, many, one in zip("wdmv", (gw, gd, gm, gv), single):
        for i, n in enumerate(MULTI_SIZES):
            assert_bit_exact(host(many[i]), host(one[i]), "adam table %s[%d] n=%d" % (name, i, n))
    assert all(float(t.abs().max()) > 0 for t, n in zip(gw, MULTI_SIZES) if n)
    # an Adam table serves the operations that need fewer buffers: SGD on (w, d), fill and norms on w
    table.sgd_update(16, 1e-3, 0.9, 5e-4)
    for i, n in enumerate(MULTI_SIZES):
        if n:
            ops.sgd_update(single[0][i], single[1][i], 16, 1e-3, 0.9, 5e-4, flags[i])
    for i, n in enumerate(MULTI_SIZES):
        assert_bit_exact(host(gw[i]), host(single[0][i]), "sgd through the adam table w[%d]" % i)
        assert_bit_exact(host(gd[i]), host(single[1][i]), "sgd through the adam table d[%d]" % i)
    table.close()


def test_sgd_table_gives_every_tensor_what_the_single_call_gives(ops):
    flags = [i % 2 == 0 for i in range(len(MULTI_SIZES))]
    _, gw = _multi_tensors(6600, 0.02)
    _, gd = _multi_tensors(6700, 0.5)
    single = [[t.clone() for t in group] for group in (gw, gd)]
    table = ops.TensorTable([gw, gd], flags)
    for step in range(2):
        table.sgd_update(16, 1e-3, 0.9, 5e-4)
        for i, n in enumerate(MULTI_SIZES):
            if n:
                ops.sgd_update(single[0][i], single[1][i], 16, 1e-3, 0.9, 5e-4, flags[i])
    for name, many, one in zip("wd", (gw, gd), single):
        for i, n in enumerate(MULTI_SIZES):
            assert_bit_exact(host(many[i]), host(one[i]), "sgd table %s[%d] n=%d" % (name, i, n))


def test_fill_table_writes_every_tensor_and_nothing_else(ops):
    import torch
    bufs = [torch.full((n + 8,), 7.0, device="cuda") for n in MULTI_SIZES]
    views = [b[4:4 + n] for b, n in zip(bufs, MULTI_SIZES)]
    views[5] = bufs[5][5:5 + MULTI_SIZES[5]]            # one view off the 16-byte grid
    table = ops.TensorTable([views])
    table.fill(-0.5)
    for b, v in zip(bufs, views):
        assert bool((v == -0.5).all())
        assert int((b == 7.0).sum()) == 8


@pytest.mark.parametrize("threshold,clip", [(0.5, 0.0), (0.0, 0.01), (3.0, 0.02), (1e9, 1e9), (0.0, 0.0)])
def test_rescale_clip_table_leaves_every_tensor_as_the_single_call_does(ops, threshold, clip):
    import torch
    _, many = _multi_tensors(6800, 0.02)
    for i, t in enumerate(many):
        t *= float(1 + i % 5)
    one = [t.clone() for t in many]
    table = ops.TensorTable([many])
    norms = torch.full((table.count,), -1.0, device="cuda")
    table.rescale_clip(threshold, clip, norms)
    want_norms = []
    for t in one:
        if t.numel():
            norm = torch.full((1,), -1.0, device="cuda")
            ops.rescale_clip(t, threshold, clip, norm)
            want_norms.append(float(norm))      # empty tensors have no place in the table
    for i, (a_, b_) in enumerate(zip(many, one)):
        assert_bit_exact(host(a_), host(b_), "rescale table tensor %d n=%d" % (i, MULTI_SIZES[i]))
    if threshold > 0.0 or clip > 0.0:
        assert host(norms).tolist() == want_norms
    # a second call on the same table (its partial sums are reused) and the no-op
    before = [t.clone() for t in many]
    table.rescale_clip(0.0, 0.0)
    for a_, b_ in zip(many, before):
        assert_bit_exact(host(a_), host(b_), "no-op")
    table.rescale_clip(threshold, clip)
    for t in one:
        if t.numel():
            ops.rescale_clip(t, threshold, clip)
    for i, (a_, b_) in enumerate(zip(many, one)):
        assert_bit_exact(host(a_), host(b_), "second rescale, tensor %d" % i)


# Shares of the launch behind the norms: one to a workgroup below 2048, two, four from 4096 on; a last workgroup that is not
# full, workgroups that end one tensor and begin others.
@pytest.mark.parametrize("big", [2, 3, 6])
def test_rescale_clip_table_by_shares(ops, big):
    import torch
    sizes = [5, 1027]
    for k in range(big):
        sizes += [3 << 20 | 4 * k, 4096, 9 + k, 3 * 4096 + 4]
    g = torch.Generator(device="cuda")
    g.manual_seed(6900 + big)
    many = [torch.empty(n, device="cuda").normal_(0.0, 0.01 * (1 + i % 7), generator=g) for i, n in enumerate(sizes)]
    one = [t.clone() for t in many]
    table = ops.TensorTable([many])
    norms = torch.zeros(table.count, device="cuda")
    for threshold, clip in ((1e9, 1e9), (40.0, 0.0), (30.0, 0.05)):
        table.rescale_clip(threshold, clip, norms)
        want = []
        for t in one:
            norm = torch.zeros(1, device="cuda")
            ops.rescale_clip(t, threshold, clip, norm)
            want.append(float(norm))
        assert host(norms).tolist() == want
        for i, (a_, b_) in enumerate(zip(many, one)):
            assert torch.equal(a_, b_), "tensor %d of %d values" % (i, sizes[i])


def test_table_of_a_whole_model_and_edge_cases(ops):
    import torch
    from pixienn_amd import capi
    # YOLOv3's 222 parameter tensors (scaled down 16x in length): one launch reaches every one
    sizes = [max(1, n // 16) for n, decayed in wl.yolov3_parameter_tensors(608)]
    assert len(sizes) > 200
    w = [torch.full((n,), float(i % 7), device="cuda") for i, n in enumerate(sizes)]
    d = [torch.ones(n, device="cuda") for n in sizes]
    table = ops.TensorTable([w, d])
    table.sgd_update(1, 0.5, 0.0)
    for i, t in enumerate(w):
        assert float(t.min()) == float(t.max()) == i % 7 + 0.5, i
    assert all(float(g.abs().max()) == 0.0 for g in d)      # momentum 0 clears the update buffer
    # an empty table is a no-op; wrong uses are rejected before anything is launched
    empty = ops.TensorTable([[]])
    empty.fill(1.0)
    assert empty.count == 0
    one = ops.TensorTable([[w[0]]])
    with pytest.raises(capi.PxError, match="buffers per tensor"):
        one.sgd_update(1, 0.5, 0.0)
    with pytest.raises(capi.PxError, match="buffers per tensor"):
        one.adam_update(1, 1, 1e-3)
    with pytest.raises(capi.PxError):
        table.sgd_update(0, 0.5, 0.0)
    with pytest.raises(capi.PxError):
        ops.TensorTable([[w[0]], [d[0]], [d[0]]])       # 3 buffers per tensor is no operation's shape
