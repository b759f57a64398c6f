"""Forwards of plans without a backward write no layer's stacks: their outputs
are those of a plan that keeps everything, bit for bit, and the stacks appear
when they are asked for."""
import numpy as np
import pytest

from cpde_amd import hip, workloads as W
from test_gpu_rows import workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('variables,order,neurons,points,chunk', [
    (2, 0, [2, 128, 130, 1], 65, 33),   # split products, one row, a ragged chunk
    (3, 2, [3, 40, 24, 1], 29, 0),      # fp32 products, several points per workgroup
    (2, 6, [2, 64, 1], 5, 0),           # one hidden layer
])
def test_outputs_and_stacks_without_a_backward(device, variables, order, neurons, points, chunk):
    wl = workload(variables, order, neurons, points, chunk, seed=41)
    print(f'[case] values neurons={neurons} rows={wl.rows} points={points} chunk={chunk}', flush=True)
    width = chunk or points
    rows = np.arange(wl.rows, dtype=np.int32)
    data = hip.Buffer.of(device, np.ascontiguousarray(wl.inputs.transpose(0, 2, 1), np.float32))
    got = []
    for backward in (False, True):
        net = hip.Net(device, wl.neurons, wl.linear, wl.init)
        plan = hip.Plan(net, wl.schema, width, backward)
        out = hip.Buffer(device, 4 * wl.rows * points)
        for repeat in range(2):   # the second pass follows the first look at a stack
            for offset in range(0, points, width):
                valid = min(width, points - offset)
                plan.activate(data, points, rows, offset, valid)
                plan.forward()
                plan.output(out, points, rows, offset, valid)
            outputs = out.download(np.float32, wl.rows * points)
            stacks = [plan.stack(layer, kind)[:valid] for layer in range(1, len(neurons) - 1) for kind in (1, 3)]
            got.append([outputs] + stacks)
        out.free()
        plan.destroy(); net.destroy()
    data.free()
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b)
