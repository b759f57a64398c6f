"""Weight gradients of thin transitions (a side of at most 16) outside the
network kernels: four adjacent entries of the wide side a lane where the
narrow side is at most 4, the scalar form elsewhere, against the oracle."""
import pytest

from cpde_amd import hip
from helpers import oracle_epoch, rel_l2
from test_gpu_rows import workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('variables,order,neurons,points', [
    (1, 1, [1, 260, 4, 1], 700),     # one input; a transition of 4 neurons; 65 lanes a column
    (4, 2, [4, 1028, 1], 83),        # four inputs; more than one round of the wide side
    (3, 6, [3, 12, 16, 1], 41),      # 84 rows, short columns of 12
    (2, 0, [2, 262, 5, 1], 333),     # a wide side off the float4s, a narrow one past 4: the scalar form
])
def test_thin_transitions(device, variables, order, neurons, points):
    wl = workload(variables, order, neurons, points, 0, seed=43)
    print(f'[case] thin neurons={neurons} rows={wl.rows} points={points}', flush=True)
    run = hip.MatchingRun(device, wl)
    run.step()
    device.synchronize()
    loss, grads = run.loss(), run.gradients()
    run.close()
    want_loss, want, _ = oracle_epoch(wl)
    assert abs(loss / want_loss - 1) < 1e-5
    for t, (g, w) in enumerate(zip(grads, want)):
        assert rel_l2(g, w) < 1e-4, t
