"""When the products' weight operands are rebuilt: after a write, and not for
having been read."""
import numpy as np
import pytest

from cpde_amd import hip
from test_gpu_rows import workload

pytestmark = pytest.mark.gpu


class Forward:
    def __init__(self, device, neurons):
        self.wl = wl = workload(2, 1, neurons, 9, 0, seed=31)
        self.net = hip.Net(device, wl.neurons, wl.linear, wl.init)
        self.plan = hip.Plan(self.net, wl.schema, wl.size, False)
        self.data = hip.Buffer.of(device, np.ascontiguousarray(wl.inputs.transpose(0, 2, 1), np.float32))
        self.rows = np.arange(wl.rows, dtype=np.int32)
        self.out = hip.Buffer(device, 4 * wl.rows * wl.size)
        self.plan.activate(self.data, wl.size, self.rows, 0, wl.size)
        self.run()

    def run(self):
        self.plan.forward()
        self.plan.output(self.out, self.wl.size, self.rows, 0, self.wl.size)

    def outputs(self):
        return self.out.download(np.float32, self.wl.rows * self.wl.size)

    def close(self):
        for b in (self.data, self.out):
            b.free()
        self.plan.destroy()
        self.net.destroy()


def rebuilds(device, body):
    device.trace(True)
    body()
    report = device.trace_report()
    device.trace(False)
    return report.get('other', (0,))[0]


def test_operands_are_rebuilt_after_a_write_alone(device):
    f = Forward(device, [2, 128, 128, 1])
    first = f.outputs()
    for t in range(3):
        assert np.array_equal(f.net.state(t, 0), f.wl.init[t])
    assert rebuilds(device, f.run) == 0
    f.net.set_state(1, 0, np.zeros_like(f.wl.init[1]))
    assert rebuilds(device, f.run) == 1
    assert not np.array_equal(f.outputs(), first)
    assert rebuilds(device, f.run) == 0
    f.net.set_state(1, 0, f.wl.init[1])
    f.run()
    assert np.array_equal(f.outputs(), first)
    # refused while a capture is open, which records nothing of it
    device.capture_begin()
    for refused in (lambda: f.net.state(1, 0), lambda: f.net.set_state(1, 0, np.zeros_like(f.wl.init[1]))):
        with pytest.raises(hip.CpdeError) as e:
            refused()
        assert e.value.code == hip.EINVAL
    f.run()
    replay = device.capture_end()
    replay.launch()
    assert np.array_equal(f.outputs(), first)
    replay.destroy()
    for bad in ((3, 0), (0, 4), (-1, 0)):
        v = np.zeros(1024, np.float32)
        for call in (hip.load().cpde_net_read, hip.load().cpde_net_write):
            assert call(f.net.handle, *bad, v.ctypes.data) == hip.EINVAL
        with pytest.raises(hip.CpdeError):
            f.net.state(*bad)
    f.close()


@pytest.mark.parametrize('width', [128, 40])
def test_replayed_forwards_see_weights_written_through_a_held_pointer(device, width):
    f = Forward(device, [2, width, width, 1])
    first = f.outputs()
    pointer, count = f.net.state_ptr(1, 0)
    f.run()
    device.capture_begin()
    f.run()
    replay = device.capture_end()
    for _ in range(2):
        device.upload_ptr(pointer, np.zeros(count, np.float32))
        replay.launch()
        assert not np.array_equal(f.outputs(), first)
        device.upload_ptr(pointer, np.ascontiguousarray(f.wl.init[1], np.float32))
        replay.launch()
        assert np.array_equal(f.outputs(), first)
    replay.destroy()

    # recorded before the pointer went out
    g = Forward(device, [2, width, width, 1])
    device.capture_begin()
    g.run()
    replay = device.capture_end()
    pointer, count = g.net.state_ptr(1, 0)
    for _ in range(2):
        device.upload_ptr(pointer, np.zeros(count, np.float32))
        replay.launch()
        assert not np.array_equal(g.outputs(), first)
        device.upload_ptr(pointer, np.ascontiguousarray(f.wl.init[1], np.float32))
        replay.launch()
        assert np.array_equal(g.outputs(), first)
    replay.destroy()
    f.close()
    g.close()
