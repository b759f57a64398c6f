"""Each product on split bf16 operands against float64, from the fp32 operands
that the kernels themselves read: its error relative to the norm of the terms.

Three bf16 planes hold an operand exactly; three of nine partial products are
left out, 2^-26 of a term in the mean; the sums are fp32.  Bars are in units of
2^-24 of the terms' norm.  The fp32 matrix instruction, a chain of K roundings,
is off by 3.4 to 4.3 units (rms) and 23 to 45 (most) on the long products here;
split ones (K / 32 roundings) are held to 2 and 16.  Without the third plane, or
without one of the six partial products, a product is off by 100 and more.
Sums of up to three terms are held to what K fused fp32 multiply-adds give, K
units of the terms' absolute sum."""
import numpy as np
import pytest

from cpde_amd import hip, workloads as W

pytestmark = pytest.mark.gpu

UNIT = 2.0 ** -24


class Layers:
    """A network on random weights and points, forward and (from a random output
    adjoint) backward, and its stacks as float64."""

    def __init__(self, device, neurons, order, points, bias=True, seed=71):
        rng = np.random.default_rng(seed)
        self.neurons = neurons
        self.schema = W.full_schema(neurons[0], order)
        self.weights = [rng.standard_normal((n, m)).astype(np.float32) * np.float32(n ** -0.5)
                        for n, m in zip(neurons, neurons[1:])]
        self.bias = [(rng.standard_normal(m) if bias else np.zeros(m)).astype(np.float32) for m in neurons[1:]]
        self.net = hip.Net(device, neurons, W.linear_flags(neurons),
                           [np.concatenate([w.ravel(), b]) for w, b in zip(self.weights, self.bias)])
        self.plan = hip.Plan(self.net, self.schema, points, True)
        self.x = rng.standard_normal((points, neurons[0])).astype(np.float32)
        stack = np.ascontiguousarray(W.input_stack(self.x, self.schema).transpose(0, 2, 1), np.float32)
        data = hip.Buffer.of(device, stack)
        self.plan.activate(data, points, np.arange(len(self.schema), dtype=np.int32), 0, points)
        self.plan.forward()
        last = len(neurons) - 1
        self.adjoint = rng.standard_normal((points, len(self.schema), neurons[-1])).astype(np.float32)
        device.upload_ptr(self.plan.stack_ptr(last, 2), self.adjoint)
        self.plan.backward()
        data.free()

    def stack(self, layer, kind):
        return self.plan.unscaled_stack(layer, kind).astype(np.float64)

    def product(self, t, values, transposed=False):
        """Float64 W values (+ bias on the value row), or W^T values, and the
        norm and absolute sum of each entry's terms."""
        w = self.weights[t].astype(np.float64)
        w = w.T if transposed else w
        z, square, total = values @ w, values ** 2 @ w ** 2, np.abs(values) @ np.abs(w)
        if not transposed:
            b = self.bias[t].astype(np.float64)
            z[:, 0] += b
            square[:, 0] += b ** 2
            total[:, 0] += np.abs(b)
        return z, np.sqrt(square), total

    def close(self):
        self.plan.destroy()
        self.net.destroy()


def check(label, error, rms=2.0, most=16.0):
    error = np.abs(error) / UNIT
    got = np.sqrt((error ** 2).mean()), error.max()
    print(f'[result] {label}: rms {got[0]:.2f}, most {got[1]:.2f} of 2^-24', flush=True)
    assert got[0] < rms and got[1] < most, (label, got)


@pytest.mark.parametrize('neurons', [[1, 128, 128, 1], [1, 200, 130, 1], [1, 128, 40, 136, 1]])
def test_network_products(device, neurons):
    """Through derivative rows: y' = u z' and dE/dz' = u dE/dy' (order 1), each
    one rounding away from the product, 1 more unit of the value at most."""
    n = Layers(device, neurons, 1, 700)
    for t in range(1, len(neurons) - 2):
        z, norm, _ = n.product(t, n.stack(t, 1))
        u, y = n.stack(t + 1, 3)[:, 0], n.stack(t + 1, 1)[:, 1]
        check(f'{neurons} forward {t}', (y - u * z[:, 1]) / (u * norm[:, 1]))
        g, norm, _ = n.product(t, n.stack(t + 1, 2), transposed=True)
        u, got = n.stack(t, 3)[:, 0], n.stack(t, 2)[:, 1]
        check(f'{neurons} backward {t}', (got - u * g[:, 1]) / (u * norm[:, 1]))
    n.close()


@pytest.mark.parametrize('narrow', [1, 2, 3])
def test_short_network_products(device, narrow):
    n = Layers(device, [1, 128, 128, narrow, 130, 1], 1, 700)
    z, _, total = n.product(3, n.stack(3, 1))
    u, y = n.stack(4, 3)[:, 0], n.stack(4, 1)[:, 1]
    check('forward', (y - u * z[:, 1]) / (u * total[:, 1]), most=narrow + 1.0)
    g, _, total = n.product(2, n.stack(3, 2), transposed=True)
    u, got = n.stack(2, 3)[:, 0], n.stack(2, 2)[:, 1]
    check('backward', (got - u * g[:, 1]) / (u * total[:, 1]), most=narrow + 1.0)
    n.close()


@pytest.mark.parametrize('neurons', [[2, 300, 264, 1], [2, 261, 70, 259, 9, 1]])
def test_layer_products(device, neurons):
    """Plans outside the network kernels keep z; dE/dz = sigma'(z) dE/dy at order
    0, where sigma' is off by up to four units of a value that reaches four norms."""
    n = Layers(device, neurons, 0, 900)
    for t in range(1, len(neurons) - 2):
        z, norm, _ = n.product(t, n.stack(t, 1))
        check(f'{neurons} forward {t}', (n.stack(t + 1, 0) - z) / norm)
        g, norm, _ = n.product(t, n.stack(t + 1, 2), transposed=True)
        s = 1 / (1 + np.exp(-n.stack(t, 0)))
        check(f'{neurons} backward {t}', (n.stack(t, 2) - s * (1 - s) * g) / (s * (1 - s) * norm), rms=4.0, most=32.0)
    n.close()


@pytest.mark.parametrize('variables,neurons', [(1, [1, 260, 1]), (2, [2, 261, 1]), (3, [3, 300, 1]), (2, [2, 300, 3, 264, 1])])
def test_short_layer_products(device, variables, neurons):
    """The input transition, and a layer of three neurons."""
    n = Layers(device, neurons, 0, 900, bias=False)
    x = n.x.astype(np.float64)[:, None, :]
    z, _, total = n.product(0, x)
    check('input', (n.stack(1, 0) - z) / total, most=variables * 1.001)
    if len(neurons) > 3:
        z, _, total = n.product(2, n.stack(2, 1))
        check('forward', (n.stack(3, 0) - z) / total, most=3.001)
    n.close()


@pytest.mark.parametrize('neurons,order,points', [
    ([2, 128, 96, 1], 2, 6000),     # 128 x 128 tiles
    ([2, 256, 200, 1], 2, 6000),    # 256 x 256 tiles
    ([2, 300, 280, 1], 0, 700),
    ([2, 300, 280, 1], 0, 3),       # three columns
    ([2, 200, 256, 1], 0, 1),
])
def test_weight_gradients(device, neurons, order, points):
    """dW = sum over K columns of dE/dz y^T, in chains of 32-column steps: a chain
    of J steps of random terms is off by about 0.4 sqrt(J) units of its norm."""
    n = Layers(device, neurons, order, points)
    for t in range(1, len(neurons) - 2):
        y = n.stack(t, 1).reshape(-1, neurons[t])
        g = n.stack(t + 1, 2).reshape(-1, neurons[t + 1])
        want, norm, total = y.T @ g, np.sqrt((y ** 2).T @ g ** 2), np.abs(y).T @ np.abs(g)
        got = n.net.gradient(t)[:want.size].reshape(want.shape)
        if len(y) <= 3:
            check(f'{neurons} {len(y)} columns', (got - want) / total, most=len(y) * 1.001 + 2e-3)
        else:
            growth = 1 + 0.4 * np.sqrt(len(y) / 32)
            check(f'{neurons} {len(y)} columns', (got - want) / norm, rms=growth, most=8 * growth)
    n.close()
