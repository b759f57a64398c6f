"""The stacks of forwards that write their outputs alone (plans without a
backward): whoever asks for one, whenever, finds what a plan that writes every
stack leaves in it, bit for bit."""
import numpy as np
import pytest

from cpde_amd import hip
from test_gpu_rows import workload

pytestmark = pytest.mark.gpu

POINTS = 9001   # more workgroups than CUs at every width here


class Values:
    """A network, a plan without a backward and data in a buffer of its own."""

    def __init__(self, device, neurons, order=1, seed=53, backward=False, net=None):
        self.device, self.wl = device, workload(2, order, neurons, POINTS, 0, seed=seed)
        wl = self.wl
        self.net = net or hip.Net(device, neurons, wl.linear, wl.init)
        self.own = net is None
        self.plan = hip.Plan(self.net, wl.schema, POINTS, backward)
        self.data = hip.Buffer.of(device, self.stack(0.0))
        self.rows = np.arange(wl.rows, dtype=np.int32)
        self.out = hip.Buffer(device, 4 * wl.rows * POINTS)

    def stack(self, shift):
        """The data of the points moved by `shift`."""
        x = self.wl.inputs.transpose(0, 2, 1).copy()
        x[0] += np.float32(shift)
        return np.ascontiguousarray(x, np.float32)

    def activate(self):
        self.plan.activate(self.data, POINTS, self.rows, 0, POINTS)

    def forward(self, shift=None):
        if shift is not None:
            self.device.upload_ptr(self.data.ptr, self.stack(shift))
        self.activate()
        self.plan.forward()
        return self

    def output(self):
        self.plan.output(self.out, POINTS, self.rows, 0, POINTS)
        return self.out.download(np.float32, self.wl.rows * POINTS)

    def stacks(self):
        return [self.plan.stack(layer, kind) for layer in range(1, len(self.net.neurons) - 1) for kind in (1, 3)]

    def close(self):
        for b in (self.data, self.out):
            b.free()
        self.plan.destroy()
        if self.own:
            self.net.destroy()


def same(got, want):
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


def expected(device, neurons, shift, **kw):
    """Stacks and outputs of a plan that keeps everything."""
    v = Values(device, neurons, backward=True, **kw)
    v.forward(shift)
    result = v.stacks(), v.output()
    v.close()
    return result


WIDTHS = [[2, 128, 130, 1], [2, 40, 24, 1]]   # split products, fp32 products


@pytest.mark.parametrize('neurons', WIDTHS)
def test_recorded_forwards_write_stacks(device, neurons):
    """A recording made before anyone asked for a stack, replayed afterwards on new data."""
    want, outputs = expected(device, neurons, 0.25)
    v = Values(device, neurons)
    v.forward(0.0)
    device.capture_begin()
    v.forward()
    replay = device.capture_end()
    pointer = v.plan.stack_ptr(1, 1)
    device.upload_ptr(v.data.ptr, v.stack(0.25))
    replay.launch()
    got = device.download_ptr(pointer, np.float32, want[0].size).reshape(want[0].shape)
    same([got, v.output()], [want[0], outputs])
    same(v.stacks(), want)
    replay.destroy()
    v.close()


@pytest.mark.parametrize('neurons', WIDTHS)
def test_stacks_after_a_replay_are_the_recorded_plans(device, neurons):
    """Another plan's forward before the replay, and its pointer after it."""
    want, outputs = expected(device, neurons, 0.25)
    v = Values(device, neurons)
    other = Values(device, neurons, seed=59, net=v.net)
    v.forward(0.0)
    device.capture_begin()
    v.forward()
    replay = device.capture_end()
    other.forward()
    device.upload_ptr(v.data.ptr, v.stack(0.25))
    replay.launch()
    same([other.plan.stack(1, 1)], want[:1])
    same([v.output()], [outputs])
    replay.destroy()
    other.close()
    v.close()


@pytest.mark.parametrize('neurons', WIDTHS)
def test_stacks_after_a_discarded_recording(device, neurons):
    want, _ = expected(device, neurons, 0.25)
    v = Values(device, neurons)
    v.forward(0.25)
    device.capture_begin()
    v.forward()
    device.capture_end(keep=False)
    same(v.stacks(), want)
    v.close()
