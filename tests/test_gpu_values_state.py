"""The stacks of forwards that write their outputs alone (plans without a
backward): whoever asks for one, whenever, finds what a plan that writes every
stack leaves in it, bit for bit."""
import numpy as np
import pytest

from cpde_amd import hip
from test_gpu_rows import workload

pytestmark = pytest.mark.gpu

POINTS = 9001


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


@pytest.mark.parametrize('order', [1, 6])   # several points per workgroup, one
@pytest.mark.parametrize('held', [False, True])
@pytest.mark.parametrize('neurons', WIDTHS + [[2, 130, 1]])
def test_stacks_are_those_of_the_forward(device, neurons, held, order):
    """Other weights and another chunk in the meantime, through the weights'
    pointer of before the forward (held) or of after it; the outputs stay."""
    want, outputs = expected(device, neurons, 0.25, order=order)
    v = Values(device, neurons, order)
    pointers = [v.net.state_ptr(t, 0)[0] for t in range(len(neurons) - 1)] if held else None
    v.forward(0.25)
    for t, w in enumerate(v.wl.init):
        device.upload_ptr(pointers[t] if held else v.net.state_ptr(t, 0)[0], np.float32(0.5) * w)
    device.upload_ptr(v.data.ptr, v.stack(0.5))
    v.activate()
    same(v.stacks(), want)
    same([v.output()], [outputs])
    for t, w in enumerate(v.wl.init):
        v.net.set_state(t, 0, w)
    v.plan.forward()   # the chunk that was activated, every stack
    same(v.stacks(), expected(device, neurons, 0.5, order=order)[0])
    v.close()


@pytest.mark.parametrize('neurons', WIDTHS)
def test_stacks_after_an_update(device, neurons):
    """An RPROP update and an Adam update behind a forward, and weights of the
    updated network in the next one."""
    want, outputs = expected(device, neurons, 0.25)
    runs = []
    for backward in (False, True):
        v = Values(device, neurons, backward=backward)
        for t in range(len(neurons) - 1):
            v.net.set_state(t, v.net.active(t), np.ones_like(v.wl.init[t]))
        v.forward(0.25)
        v.net.rprop()
        v.net.adam(1, 1e-2)
        if not backward:
            same(v.stacks(), want)
            same([v.output()], [outputs])
        runs.append([v.forward().output()] + v.stacks())
        v.close()
    same(*runs)


@pytest.mark.parametrize('neurons', WIDTHS)
def test_bound_sets_and_the_arena_keep_their_own(device, neurons):
    """A forward into a bound set, one in the arena before and after: each place
    holds its own forward's stacks."""
    in_set, set_outputs = expected(device, neurons, 0.25)
    in_arena, outputs = expected(device, neurons, 0.5)
    v = Values(device, neurons)
    kept = hip.vp()
    hip.check(hip.load().cpde_stacks_create(v.plan.handle, hip.ctypes.byref(kept)))
    bind = hip.load().cpde_plan_bind
    v.forward(0.5)
    hip.check(bind(v.plan.handle, kept))
    v.forward(0.25)
    for t, w in enumerate(v.wl.init):
        v.net.set_state(t, 0, 0.5 * w)
    same(v.stacks(), in_set)
    same([v.output()], [set_outputs])
    hip.check(bind(v.plan.handle, None))
    same(v.stacks(), in_arena)
    same([v.output()], [outputs])
    hip.check(bind(v.plan.handle, kept))
    same(v.stacks(), in_set)
    hip.check(bind(v.plan.handle, None))
    hip.check(hip.load().cpde_stacks_destroy(kept))
    v.close()


@pytest.mark.parametrize('neurons', WIDTHS)
@pytest.mark.parametrize('keep', [True, False])
def test_stacks_asked_for_inside_a_capture(device, neurons, keep):
    """Of a forward before the capture, in a recording that runs none."""
    want, outputs = expected(device, neurons, 0.25)
    v = Values(device, neurons)
    v.forward(0.25)
    v.output()   # its rows are on the device before the capture
    device.capture_begin()
    pointer = v.plan.stack_ptr(1, 1)
    v.plan.output(v.out, POINTS, v.rows, 0, POINTS)
    replay = device.capture_end(keep)
    got = device.download_ptr(pointer, np.float32, want[0].size).reshape(want[0].shape)
    same([got] + v.stacks(), [want[0]] + want)
    same([v.output()], [outputs])
    if replay:
        replay.launch()
        same(v.stacks(), want)
        replay.destroy()
    v.close()


def test_backward_of_another_plan_reads_the_arena(device):
    """A backward plan's adjoints of a forward that another plan ran."""
    neurons = [2, 40, 24, 1]
    adjoint = np.random.default_rng(3).standard_normal((POINTS, 3, 1)).astype(np.float32)
    got = []
    for plain in (False, True):
        v = Values(device, neurons)
        other = Values(device, neurons, net=v.net, backward=True)
        other.activate()
        (other if plain else v).forward(0.0)
        device.upload_ptr(other.plan.stack_ptr(3, 2), adjoint)
        other.plan.backward()
        got.append([v.net.gradient(t) for t in range(3)])
        other.close()
        v.close()
    same(*got)


def test_operands_after_a_rejected_update(device):
    """Stacks of an older forward asked for between an update's issue and its
    rejection: the next forward runs on the weights that stand."""
    neurons = [2, 128, 130, 1]
    v = Values(device, neurons)
    T = len(neurons) - 1
    v.forward(0.25)
    for t, w in enumerate(v.wl.init):
        v.net.set_state(t, 0, 0.5 * w)
    kept = hip.vp()
    hip.check(hip.load().cpde_stacks_create(v.plan.handle, hip.ctypes.byref(kept)))
    hip.check(hip.load().cpde_plan_bind(v.plan.handle, kept))
    want = v.forward(0.25).output()   # the operands are current
    hip.check(hip.load().cpde_plan_bind(v.plan.handle, None))
    for t in range(T):
        v.net.set_state(t, v.net.active(t), np.full_like(v.wl.init[t], np.inf))
    device.costs_begin(1)
    v.net.issue_update(1, inspect='full')
    v.plan.stack_ptr(1, 1)
    assert not v.net.resolve_update(1)[2]
    v.plan.forward()
    same([v.output()], [want])
    hip.check(hip.load().cpde_stacks_destroy(kept))
    v.close()
