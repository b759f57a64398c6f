"""Epochs of networks whose layers differ in width, on split and on fp32
products of layers of 128 and more, against float64."""
import pytest

import exact
from cpde_amd import hip
from helpers import rel_l2
from test_gpu_rows import workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('variables,order,neurons,points', [
    (2, 6, [2, 256, 64, 1], 4133),         # fp32, two points per workgroup at 64 rows of columns
    (2, 2, [2, 128, 256, 128, 1], 5003),   # fp32, 16-column tiles paired over 128 neurons
    (2, 3, [2, 128, 64, 32, 1], 729),      # fp32, eight waves
    (2, 6, [2, 256, 128, 1], 729),         # fp32, one point
    (1, 4, [1, 250, 20, 20, 1], 333),      # fp32, masked tiles
    (2, 2, [2, 192, 256, 1], 5003),        # split
    (2, 2, [2, 128, 50, 128, 1], 2003),    # split
])
def test_mixed_widths(device, variables, order, neurons, points):
    wl = workload(variables, order, neurons, points, 0, seed=79)
    print(f'[case] mixed products {neurons} rows={wl.rows} points={points}', flush=True)
    got = []
    for one_pass in (True, False):
        run = hip.MatchingRun(device, wl, one_pass=one_pass)
        run.step()
        got.append((run.loss(), run.gradients()))
        run.close()
    loss, want = exact.epoch(wl)
    for (l, grads) in got:
        assert abs(l / loss - 1) < 4e-6
        for t, (g, w) in enumerate(zip(grads, want)):
            print(f'[result] transition {t} float64 {rel_l2(g, w):.2e}', flush=True)
            # chains of a few thousand columns: sqrt(4,000) 2^-24 of the terms' norm
            assert rel_l2(g, w) < 4e-6, t
