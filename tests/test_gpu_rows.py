"""Plans outside the fused kernels (more than 64 rows, layers wider than 256):
the epoch of the generated row kernels and their products against the oracle,
and against the table-driven compositions on the same plan (the products'
precision is pinned by test_gpu_product_accuracy.py)."""
import numpy as np
import pytest

from cpde_amd import hip, workloads as W
from helpers import oracle_epoch, rel_l2

pytestmark = pytest.mark.gpu

# (variables, order, neurons, points, chunk): the largest schema that takes row
# kernels (126 rows), the first widths past the fused kernels, one row, one
# point, elements that do not fill a workgroup, a ragged last chunk
SHAPES = [
    (3, 6, [3, 20, 12, 1], 37, 0),
    (4, 5, [4, 9, 7, 1], 11, 0),
    (2, 2, [2, 264, 257, 1], 29, 13),
    (1, 0, [1, 300, 1], 5, 0),
    (2, 6, [2, 288, 31, 1], 1, 0),
    (3, 6, [3, 17, 65, 1], 6, 0),
]


def workload(variables, order, neurons, points, chunk, seed=17):
    schema = W.full_schema(variables, order)
    rng = np.random.default_rng(seed)
    pts = rng.uniform(0, 1, (points, variables))
    freq, coef, phase = W.fourier_modes(variables, 4, 2, seed)
    target = W.fourier_target(pts, schema, freq, coef, phase)
    return W.MatchingWorkload('rows', neurons, pts, schema, target, 1.0 / (target ** 2).mean(axis=1),
                              W.xavier_weights(neurons, seed), chunk=chunk)


def epoch(device, wl):
    run = hip.MatchingRun(device, wl)
    try:
        run.step()
        device.synchronize()
        return run.loss(), run.gradients()
    finally:
        run.close()


@pytest.mark.parametrize('variables,order,neurons,points,chunk', SHAPES)
def test_row_kernel_epoch_matches_oracle(device, monkeypatch, variables, order, neurons, points, chunk):
    wl = workload(variables, order, neurons, points, chunk)
    print(f'[case] rows={wl.rows} neurons={neurons} points={points} chunk={chunk}', flush=True)
    loss, grads = epoch(device, wl)
    want_loss, want, _ = oracle_epoch(wl)
    assert abs(loss / want_loss - 1) < 1e-5
    for t, (g, w) in enumerate(zip(grads, want)):
        assert rel_l2(g, w) < 1e-4, t
    monkeypatch.setenv('CPDE_FUSED', '0')   # the table-driven compositions
    table_loss, table = epoch(device, wl)
    assert abs(loss / table_loss - 1) < 1e-5
    for t, (g, w) in enumerate(zip(grads, table)):
        assert rel_l2(g, w) < 1e-4, t


@pytest.mark.parametrize('outputs', [1, 3, 8, 9])   # up to 8 the output adjoint forms dE/dy itself
def test_output_adjoint_of_row_kernels(device, monkeypatch, outputs):
    """Gradients from given dE/dz of the output layer, against the table-driven
    path, whose products run on their own."""
    neurons, points = [2, 270, outputs], 7
    print(f'[case] output adjoint, {outputs} outputs', flush=True)
    schema = W.full_schema(2, 3)
    init = W.xavier_weights(neurons, 5)
    pts = np.random.default_rng(5).random((points, 2), dtype=np.float32)
    stack = np.ascontiguousarray(W.input_stack(pts, schema).transpose(0, 2, 1), np.float32)
    adjoint = np.random.default_rng(6).standard_normal(points * len(schema) * outputs).astype(np.float32)
    got = []
    for fused in ('2', '0'):
        monkeypatch.setenv('CPDE_FUSED', fused)
        net = hip.Net(device, neurons, W.linear_flags(neurons), init)
        plan = hip.Plan(net, schema, points, True)
        data = hip.Buffer.of(device, stack)
        plan.activate(data, points, np.arange(len(schema), dtype=np.int32), 0, points)
        plan.forward()
        device.upload_ptr(plan.stack_ptr(2, 2), adjoint)
        plan.backward(False)
        got.append([net.gradient(t) for t in range(2)])
        data.free()
        plan.destroy(); net.destroy()
    for t in range(2):
        assert rel_l2(got[0][t], got[1][t]) < 1e-5, t
