"""The network kernels' products on split bf16 operands (networks of wide
layers) at the edges of their tiles: widths off the 16-neuron blocks and the
32-k steps, a narrow layer beside a wide one, row counts around the column
tiles, one and several points per workgroup, one LDS tile and two.

Against the oracle, which sums in fp32 in one chain and is itself off by up to
about 5e-5 here (the repository's gradient bar is 1e-3): values in the wrong place
show, a loss of precision need not.  test_gpu_product_accuracy.py pins that."""
import numpy as np
import pytest

from cpde_amd import hip, workloads as W
from helpers import oracle_epoch, rel_l2
from test_gpu_rows import workload

pytestmark = pytest.mark.gpu


def steps(device, wl, one_pass):
    run = hip.MatchingRun(device, wl, one_pass=one_pass)
    try:
        run.step()
        device.synchronize()
        return run.loss(), run.gradients()
    finally:
        run.close()


# (variables, order, neurons, points, chunk)
@pytest.mark.parametrize('variables,order,neurons,points,chunk', [
    (2, 6, [2, 128, 128, 1], 3, 0),          # 28 rows, one point per workgroup
    (2, 2, [2, 130, 129, 131, 1], 37, 0),    # off every block and step
    (1, 0, [1, 128, 20, 1], 77, 16),         # one row; a narrow layer (fewer blocks than waves)
    (3, 4, [3, 20, 136, 17, 1], 19, 0),      # 35 rows on 48 columns
    (2, 5, [2, 144, 256, 1], 4133, 0),       # a long grid: two points, one LDS tile, a lone last point
    (3, 3, [3, 200, 160, 2, 1], 41, 0),      # 20 rows; a two-neuron layer
])
def test_split_products(device, variables, order, neurons, points, chunk):
    wl = workload(variables, order, neurons, points, chunk, seed=29)
    print(f'[case] split products neurons={neurons} rows={wl.rows} points={points} chunk={chunk}', flush=True)
    loss, grads = steps(device, wl, True)
    separate_loss, separate = steps(device, wl, False)
    assert abs(loss / separate_loss - 1) < 1e-12
    want_loss, want, _ = oracle_epoch(wl)
    assert abs(loss / want_loss - 1) < 1e-5
    for t, (g, s, w) in enumerate(zip(grads, separate, want)):
        print(f'[result] transition {t} oracle {rel_l2(g, w):.2e}', flush=True)
        assert np.array_equal(g, s), t
        assert rel_l2(g, w) < 1e-4, t


@pytest.mark.parametrize('variables,order,neurons,points,chunk', [
    (2, 5, [2, 64, 40, 1], 1031, 0),     # 21 rows: one point per workgroup, a few past the resident grid
    (1, 3, [1, 33, 64, 64, 1], 8301, 8250),  # four rows: several points, a ragged second chunk
    (2, 0, [2, 20, 1], 33001, 0),        # one hidden layer, one row
])
def test_long_one_pass_of_narrow_layers(device, variables, order, neurons, points, chunk):
    """One-pass epochs over more workgroups than fit on the device together:
    loss and gradients of separate launches; and once a stack's pointer is out,
    every stack as separate launches leave it."""
    wl = workload(variables, order, neurons, points, chunk, seed=37)
    print(f'[case] long one pass neurons={neurons} rows={wl.rows} points={points}', flush=True)
    got = []
    for one_pass in (True, False):
        run = hip.MatchingRun(device, wl, one_pass=one_pass)
        run.step()
        device.synchronize()
        got.append((run.loss(), run.gradients()))
        # deferred, the chunks' reductions finish their staged cost records together
        hip.check(hip.load().cpde_gradients_defer(device.handle, 1))
        run.step()
        assert run.loss() == got[-1][0]
        hip.check(hip.load().cpde_gradients_defer(device.handle, 0))
        for a, b in zip(run.gradients(), got[-1][1]):
            assert np.array_equal(a, b)
        run.plan.stack_ptr(1, 1)
        run.step()
        device.synchronize()
        last = points % (chunk or points) or points   # points of the chunk the stacks hold
        got[-1] += ([run.plan.stack(layer, kind)[:last] for layer in range(1, len(neurons) - 1) for kind in (1, 2, 3)],)
        run.close()
    assert abs(got[0][0] / got[1][0] - 1) < 1e-12
    for a, b in zip(got[0][1] + got[0][2], got[1][1] + got[1][2]):
        assert np.array_equal(a, b)


def test_forward_sees_weights_written_through_a_held_pointer(device):
    """A program that keeps a weights pointer and writes through it again: each
    separate forward runs on what it wrote, on split operands too."""
    for width in (128, 40):
        wl = workload(2, 1, [2, width, width, 1], 9, 0, seed=31)
        net = hip.Net(device, wl.neurons, wl.linear, wl.init)
        plan = hip.Plan(net, wl.schema, wl.size, False)
        data = hip.Buffer.of(device, np.ascontiguousarray(wl.inputs.transpose(0, 2, 1), np.float32))
        rows = np.arange(wl.rows, dtype=np.int32)
        out = hip.Buffer(device, 4 * wl.rows * wl.size)
        plan.activate(data, wl.size, rows, 0, wl.size)

        def outputs():
            plan.forward()
            plan.output(out, wl.size, rows, 0, wl.size)
            return out.download(np.float32, wl.rows * wl.size)

        pointer, count = net.state_ptr(1, 0)
        first = outputs()
        device.upload_ptr(pointer, np.zeros(count, np.float32))
        zero = outputs()
        device.upload_ptr(pointer, np.ascontiguousarray(wl.init[1], np.float32))
        assert np.array_equal(outputs(), first)
        assert not np.array_equal(zero, first)
        for b in (data, out):
            b.free()
        plan.destroy(); net.destroy()
