"""Two points per workgroup in one LDS tile at the most that it holds: a narrow
layer beside a wide one, whose compositions leave lanes idle, and a single
hidden layer of 56 rows, which has no product and no operand planes.

Against float64: a gradient sums K products of 24-bit values in fp32, off by
about sqrt(K) 2^-24 of their norm (3e-5 for 230,000 columns in one chain; the
kernels' chains are at most a few thousand long, 4e-6)."""
import pytest

import exact
from cpde_amd import hip
from helpers import rel_l2
from test_gpu_rows import workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('variables,order,neurons,points', [
    (2, 6, [2, 80, 256, 1], 4133),
    (2, 6, [2, 128, 240, 1], 4133),
    (3, 5, [3, 256, 1], 4101),
])
def test_two_points_in_one_tile(device, variables, order, neurons, points):
    wl = workload(variables, order, neurons, points, 0, seed=47)
    print(f'[case] two points in one tile neurons={neurons} rows={wl.rows}', flush=True)
    run = hip.MatchingRun(device, wl)
    run.step()
    device.synchronize()
    loss, grads = run.loss(), run.gradients()
    run.close()
    want_loss, want = exact.epoch(wl)
    assert abs(loss / want_loss - 1) < 4e-6
    for t, (g, w) in enumerate(zip(grads, want)):
        print(f'[result] transition {t} float64 {rel_l2(g, w):.2e}', flush=True)
        assert rel_l2(g, w) < 4e-6, t
