"""Stacks of recorded one-pass epochs over more workgroups than fit on the device
together: a stack's pointer taken after the recording shows what separate
launches leave, on every replay."""
import numpy as np
import pytest

from cpde_amd import hip
from test_gpu_rows import workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('variables,order,neurons,points', [
    (2, 5, [2, 64, 40, 1], 1031),     # one point per workgroup
    (1, 3, [1, 33, 64, 64, 1], 8301),  # several
])
def test_recorded_long_epochs_write_their_stacks(device, variables, order, neurons, points):
    wl = workload(variables, order, neurons, points, 0, seed=61)
    moved = workload(variables, order, neurons, points, 0, seed=67)
    hidden = [(layer, kind) for layer in range(1, len(neurons) - 1) for kind in (1, 2, 3)]

    def load(run, w):
        run.data.upload(np.ascontiguousarray(w.inputs.transpose(0, 2, 1), np.float32))
        run._loaded = None

    run = hip.MatchingRun(device, wl)
    run.step()
    run._loaded = None
    device.capture_begin()
    run.step()
    replay = device.capture_end()
    recorded = run.loss(), run.gradients()
    pointers = [run.plan.stack_ptr(*s) for s in hidden]
    load(run, moved)
    replay.launch()
    got = [device.download_ptr(p, np.float32, points * wl.rows * neurons[layer]) for p, (layer, _) in zip(pointers, hidden)]
    replay.destroy()
    run.close()

    separate = hip.MatchingRun(device, wl, one_pass=False)
    separate.step()
    loss, grads = separate.loss(), separate.gradients()
    assert abs(recorded[0] / loss - 1) < 1e-12
    for a, b in zip(recorded[1], grads):
        assert np.array_equal(a, b)
    load(separate, moved)
    separate.step()
    for a, (layer, kind) in zip(got, hidden):
        assert np.array_equal(a, separate.plan.stack(layer, kind).ravel()), (layer, kind)
    separate.close()
