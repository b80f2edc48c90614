"""Which stream nms_to_host waits for, without a GPU: the copies of the survivors and their count go to the
current stream of the TENSORS' device, so that is the one that has to be synchronised, whatever the current
device is.  torch is stood in for by a few lines in which a copy that does not block lands when its device's
stream is synchronised, and not before."""
import numpy as np
import pytest

from pixienn_amd import ops


class Device:
    def __init__(self, type, index):
        self.type, self.index = type, index


class Machine:
    """Two devices, device 0 current; `torch` for nms_to_host."""
    int32 = "int32"

    def __init__(self):
        self.cuda = self
        self.devices = [Device("cuda", 0), Device("cuda", 1)]
        self.at = 0
        self.queued = {0: [], 1: []}

    def install(self, monkeypatch):
        monkeypatch.setattr(ops, "torch", self)
        monkeypatch.setattr(ops, "_current_device", lambda: self.at)

    def current_stream(self, device=None):
        if device is not None and device.type != "cuda":
            raise ValueError("expected a cuda device")
        return Stream(self, self.at if device is None else device.index)

    def empty(self, shape, dtype, pin_memory):
        assert pin_memory
        return Tensor(self, np.full(shape, -77, np.int32), Device("cpu", 0))


class Stream:
    def __init__(self, machine, index):
        self.machine, self.index = machine, index

    def synchronize(self):
        for copy in self.machine.queued[self.index]:
            copy()
        self.machine.queued[self.index].clear()


class Tensor:
    def __init__(self, machine, values, device):
        self.machine, self.values, self.device = machine, values, device
        self.shape, self.dtype = values.shape, values.dtype
        self.is_cuda = device.type == "cuda"

    def copy_(self, source, non_blocking):
        assert non_blocking

        def land():
            self.values[...] = source.values
        if source.is_cuda:
            self.machine.queued[source.device.index].append(land)
        else:
            land()

    def __getitem__(self, at):
        v = self.values[at]
        return Tensor(self.machine, v, self.device) if isinstance(v, np.ndarray) else v

    def cpu(self):
        if self.is_cuda:
            Stream(self.machine, self.device.index).synchronize()
        return Tensor(self.machine, self.values.copy(), Device("cpu", 0))

    def numpy(self):
        assert not self.is_cuda
        return self.values


@pytest.mark.parametrize("where", [0, 1, "cpu"])
@pytest.mark.parametrize("found", [0, 3, 5000])
def test_survivors_are_read_after_the_copies(monkeypatch, where, found):
    machine = Machine()
    device = Device("cpu", 0) if where == "cpu" else machine.devices[where]
    rows = np.arange(6000 * 8, dtype=np.int32).reshape(6000, 8)
    machine.install(monkeypatch)
    got = ops.nms_to_host(Tensor(machine, rows, device), Tensor(machine, np.array([found], np.int32), device))
    assert got.tobytes() == rows[:found].tobytes()


def test_count_and_records_on_two_devices(monkeypatch):
    machine = Machine()
    rows = np.arange(64, dtype=np.int32).reshape(8, 8)
    machine.install(monkeypatch)
    got = ops.nms_to_host(Tensor(machine, rows, machine.devices[0]),
                          Tensor(machine, np.array([2], np.int32), machine.devices[1]))
    assert got.tobytes() == rows[:2].tobytes()


def test_launches_of_the_current_device_end_before_the_copies(monkeypatch):
    """Records on device 1 that a launch on device 0's stream writes."""
    machine = Machine()
    rows = np.zeros((8, 8), np.int32)
    machine.queued[0].append(lambda: rows.fill(5))
    machine.install(monkeypatch)
    got = ops.nms_to_host(Tensor(machine, rows, machine.devices[1]),
                          Tensor(machine, np.array([8], np.int32), machine.devices[1]))
    assert got.tobytes() == np.full((8, 8), 5, np.int32).tobytes()
