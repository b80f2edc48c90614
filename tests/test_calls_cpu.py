"""The native calls of the C ABI against the ctypes binding: what they cover, what they leave to it, and that both refuse
the same.  No device: every call here ends at an argument check."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from pixienn_amd import capi, ops


def test_every_native_call_has_the_arguments_of_the_binding():
    capi.load()
    assert capi.native
    for name, (_, tensors) in capi.native.items():
        types = capi.SIGNATURES[name]
        assert len(tensors) == len(types), name
        assert all(t is ctypes.c_void_p for t, is_tensor in zip(types, tensors) if is_tensor), name
        assert types[-1] is ctypes.c_void_p and not tensors[-1], name      # the stream


def test_a_call_is_made_or_left_and_refused_alike():
    capi.load()
    axpy = capi.native["pxh_axpy"][0]
    null = (4, 1.0, None, None, None)
    assert axpy(*null) == capi.call_raw("pxh_axpy", *null) != 0
    cpu = torch.zeros(4)
    for args in [(4, 1.0, cpu, cpu, None), (4, 1, None, None, None), (-1, 1.0, None, None, None), (4, 1.0, 64, None, None),
                 (np.int64(4), 1.0, None, None, None), (2 ** 70, 1.0, None, None, None), (4, 1.0, None, None, -2 ** 70),
                 (4, 1.0, None, None), ("4", 1.0, None, None, None)]:
        assert axpy(*args) is None, args
    route = capi.native["pxh_route_forward"][0]
    assert route(None, None, 2 ** 31, 1, 1, 0, None) is None                # an int, not whatever is left of it


@pytest.mark.parametrize("bad,message", [(torch.zeros(1, 2, 2, 2), "must live on the GPU"), (np.zeros((1, 2, 2, 2)), "torch.Tensor expected"),
                                         (7, "torch.Tensor expected")])
def test_what_is_no_tensor_of_the_device_is_named(bad, message):
    good = torch.zeros(1, 2, 2, 2)
    for f in (lambda: ops.bias_act_forward(bad, good, good, "leaky"), lambda: ops.axpy(1.0, bad, good),
              lambda: ops.bn_act_backward(bad, *[good] * 7, "leaky"), lambda: ops.route_forward(bad, good, 0),
              lambda: ops.rescale_clip(bad), lambda: ops.sgd_update(bad, good, 1, 0.1, 0.9)):
        with pytest.raises(capi.PxError, match=message):
            f()


def child(source):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    proc = subprocess.run([sys.executable, "-c", source], cwd=root, capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0, proc.stderr


def test_the_binding_loads_without_torch():
    child("""
import sys
from pixienn_amd import capi
assert capi.load().pxh_abi_version() == 2 and capi.call_raw("pxh_axpy", 4, 1.0, None, None, None) != 0
assert "torch" not in sys.modules and not capi.native
from pixienn_amd import ops
try:
    ops.axpy(1.0, 7, 7)
except capi.PxError as e:
    assert "torch.Tensor expected" in str(e)
ops.torch.zeros(1)
capi.bind_calls()
assert "pxh_axpy" in capi.native
""")


def test_a_missing_extension_is_named_by_the_first_call_that_wants_it():
    child("""
import sys, torch
sys.modules["pixienn_amd._calls"] = None
from pixienn_amd import capi, ops
assert capi.load().pxh_abi_version() == 2 and not capi.native
try:
    ops.axpy(1.0, torch.zeros(4), torch.zeros(4))
except capi.PxError as e:
    assert "not built" in str(e)
else:
    raise SystemExit("no error")
""")
