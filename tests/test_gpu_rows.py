"""Plans outside the fused kernels (more than 64 rows, layers wider than 256):
the epoch of the generated row kernels and their products against the oracle,
and against the table-driven compositions on the same plan."""
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
