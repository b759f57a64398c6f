"""The weight gradient's split tiles (bf16 matrix instructions at fp32 accuracy)
at the edges of their tiles and splits: each epoch against the oracle, and
against the same plan on the direct tiles (CPDE_WGRAD_SPLIT=0).

Tolerance between the two: both sum the same fp32 products; a sum of K columns
in fp32 partial sums is off by at most about sqrt(K) 2^-24 of its terms' norm in
one chain, 3e-5 at the longest case here, and its chains are a split's, 5e-6 at
most.  Against the oracle, whose serial fp32 sums err
by up to K 2^-24 (2e-2 at 264,006 columns), the repository's gradient bar, 1e-3."""
import numpy as np
import pytest

from cpde_amd import hip, workloads as W
from helpers import oracle_epoch, rel_l2
from test_gpu_rows import workload

pytestmark = pytest.mark.gpu


def epoch(device, wl, static=False):
    run = hip.MatchingRun(device, wl, static_scratch=static)
    try:
        run.step()
        device.synchronize()
        return run.loss(), run.gradients()
    finally:
        run.close()


# (variables, order, neurons, points, chunk)
@pytest.mark.parametrize('variables,order,neurons,points,chunk', [
    (2, 2, [2, 65, 65, 1], 44001, 0),       # 128 tiles, one column past 64, scalar loads
    (2, 1, [2, 128, 68, 1], 44001, 0),      # 128 tiles, two a CU, a ragged last split
    (2, 2, [2, 132, 129, 1], 21763, 0),     # 256 tiles, odd width, a last split of 18 columns
    (2, 2, [2, 260, 300, 100, 1], 701, 350),  # several 256 tiles, mixed with wider than them, chunks
    (1, 0, [1, 288, 288, 1], 33, 0),        # one row, one step and one column
])
def test_split_tiles(device, monkeypatch, variables, order, neurons, points, chunk):
    wl = workload(variables, order, neurons, points, chunk, seed=23)
    print(f'[case] split tiles neurons={neurons} rows={wl.rows} points={points} chunk={chunk}', flush=True)
    loss, grads = epoch(device, wl)
    monkeypatch.setenv('CPDE_WGRAD_SPLIT', '0')
    direct_loss, direct = epoch(device, wl)
    assert loss == direct_loss
    want_loss, want, _ = oracle_epoch(wl)
    assert abs(loss / want_loss - 1) < 1e-4
    # the same sums in another order: equal bits would be the direct tiles twice
    assert any(not np.array_equal(g, d) for g, d in zip(grads, direct))
    for t, (g, d, w) in enumerate(zip(grads, direct, want)):
        print(f'[result] transition {t} direct {rel_l2(g, d):.2e} oracle {rel_l2(g, w):.2e}', flush=True)
        assert rel_l2(g, d) < 5e-6, t
        assert rel_l2(g, w) < 1e-3, t


def test_static_scratch_keeps_its_plans(device):
    """256-wide layers over one-pass chunks: the split tiles' partials exceed the
    static scratch, so both epochs take the direct tiles, bit for bit."""
    wl = workload(2, 2, [2, 256, 256, 1], 700, 0, seed=5)
    loss, grads = epoch(device, wl)
    static_loss, static = epoch(device, wl, static=True)
    assert loss == static_loss
    for g, s in zip(grads, static):
        assert np.array_equal(g, s)
