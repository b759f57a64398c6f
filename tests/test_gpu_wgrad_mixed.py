"""Weight gradients of layers of several widths: which transitions take split
tiles, and in one launch or two, against float64 and with every partial in its
place (a second, accumulating epoch doubles the gradient to rounding)."""
import numpy as np
import pytest

import exact
from cpde_amd import hip
from helpers import rel_l2
from test_gpu_rows import workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('order,neurons,points', [
    (1, [2, 256, 256, 64, 1], 30011),      # a 256 tile, and direct tiles in another launch
    (1, [2, 200, 100, 50, 1], 30011),      # the same, masked
    (1, [2, 96, 96, 64, 1], 60013),        # masked 128 tiles beside direct ones
    (1, [2, 128, 128, 64, 1], 60013),      # whole ones: direct all
    (1, [2, 256, 70, 66, 1], 60013),       # 256 and 128 tiles
    (1, [2, 130, 130, 1], 700),            # too few columns for a 256 tile
    (0, [2, 512, 512, 264, 1], 20001),     # outside the network kernels: 256 tiles all the same
    (0, [2, 512, 512, 1], 700),
])
def test_mixed_widths(device, order, neurons, points):
    wl = workload(2, order, neurons, points, 0, seed=73)
    print(f'[case] mixed widths {neurons} rows={wl.rows}', flush=True)
    run = hip.MatchingRun(device, wl)
    run.step()
    loss, grads = run.loss(), run.gradients()
    cost = (run.target, run.samples, run.target_rows, run.weights, run.weight_samples, 0, points, 0, True)
    run.plan.epoch_matching(*cost, True)
    twice = run.gradients()
    run.close()
    want_loss, want = exact.epoch(wl, step=4096)
    assert abs(loss / want_loss - 1) < 4e-6
    for t, (g, w, s) in enumerate(zip(grads, want, twice)):
        print(f'[result] transition {t} float64 {rel_l2(g, w):.2e}', flush=True)
        # chains of a few thousand columns: sqrt(4,000) 2^-24 of the terms' norm
        assert rel_l2(g, w) < 4e-6, t
        assert rel_l2(s, 2.0 * g.astype(np.float64)) < 2.0 ** -23, t
