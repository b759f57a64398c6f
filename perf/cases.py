"""The work this framework is measured by.

A case is one call, or one step of a training loop, as a program that uses the
framework makes it, on inputs made from a seed:

  * ``epoch``     forward, matching cost and weight gradient over every chunk;
  * ``loss``      the same, and the loss read back (what an optimiser of the
                  caller's own asks for);
  * ``rprop``     an epoch with its RPROP update;
  * ``adam``      an epoch followed by an Adam update;
  * ``evaluate``  derivative outputs of new points: activation, forward, copy out;
  * ``poisson``   a training call of the protocol server: the Poisson problem on
                  a disk (two expression costs, a cost graph, RPROP), then the
                  trained weights read back.

The first five go through the binding of the C ABI, the last through the wire
protocol.  A network takes ``variables`` inputs through ``hidden`` sigmoid layers of
``neurons`` neurons to one output, on all mixed partials through ``order``.
"""
import math
import random

import numpy as np
import torch

from cpde_amd import hip, wire, workloads
from cpde_amd.build import SERVER

MODES, MAX_FREQUENCY = 8, 3      # of the Fourier sums that the networks fit
ADAM_RATE = 1e-3


def _case(name, call, variables, order, neurons, hidden, points, chunk=0, per_sample=False, epochs=0):
    return {'name': name, 'call': call, 'variables': variables, 'order': order, 'neurons': neurons, 'hidden': hidden,
            'points': points, 'chunk': chunk, 'per_sample': per_sample, 'epochs': epochs}


def listed():
    return [
        # the smallest fit: a small network on a few dozen points, one training
        # epoch; latency and launches are all of it
        _case('fit_tiny', 'rprop', 2, 6, 32, 2, 40),
        # the published benchmark shape (2->128^4->1 on 27 x 27 points) at the
        # order a second-order PDE needs, one training epoch
        _case('fit_order2', 'rprop', 2, 2, 128, 4, 729),
        # the headline: the same shape at order 6 in the published scope
        # (forward, cost, weight gradient)
        _case('fit_order6', 'epoch', 2, 6, 128, 4, 729),
        # a network and a point set of no round size, weights per sample (a
        # quadrature), the loss back on the host each time
        _case('fit_odd_width', 'loss', 2, 3, 50, 3, 5003, per_sample=True),
        # a narrow network on a full batch of collocation points, Adam
        _case('fit_narrow', 'adam', 2, 2, 64, 3, 16384),
        # the physics-informed workload: training epochs of the Poisson problem
        # (4096 interior points, 256 on the boundary) through the server
        _case('poisson_train', 'poisson', 2, 2, 64, 3, 4352, epochs=50),
        # all mixed partials through order 4 in three variables, full batch, Adam
        _case('fit_3d_order4', 'adam', 3, 4, 128, 5, 32768),
        # sixth order in three variables (84 rows): one loss and gradient
        _case('fit_3d_order6', 'loss', 3, 6, 64, 3, 2000),
        # a wide network in chunks
        _case('fit_wide', 'epoch', 2, 2, 512, 3, 4096, chunk=2048),
        # the largest: 2->256^4->1 at order 6 on 512 x 512 points in chunks
        _case('fit_large', 'epoch', 2, 6, 256, 4, 262144, chunk=65536),
        # a trained network looked at on a fine grid: values alone
        _case('evaluate_values', 'evaluate', 2, 0, 128, 4, 65536),
        # and with the derivatives through order 2 in three variables
        _case('evaluate_3d_order2', 'evaluate', 3, 2, 128, 5, 32768),
    ]


def _spread(rng, low, high):
    """A whole number between low and high, even over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng: random.Random):
    call = rng.choice(['epoch', 'epoch', 'loss', 'rprop', 'adam', 'evaluate', 'evaluate', 'poisson'])
    if call == 'poisson':
        c = _case('', call, 2, 2, rng.choice([32, 48, 64, 96]), rng.randint(2, 4), 0, epochs=50)
        c['points'] = 16 * _spread(rng, 8, 256) + 256
        del c['name']
        return c
    variables = rng.choice([1, 2, 2, 2, 3, 3])
    order = rng.randint(0, 6)
    rows = math.comb(variables + order, order)
    # (the most that the fused kernels take at this many rows, or a wider network)
    wide = rng.random() < 0.2
    neurons = _spread(rng, 288, 512) if wide else _spread(rng, 16, 256 if rows <= 32 else 192)
    grain = rng.choice([1, 2, 16, 32])     # odd widths among the round ones
    neurons = max(grain, neurons // grain * grain)
    c = _case('', call, variables, order, neurons, rng.randint(2, 5), _spread(rng, 32, 262144),
              per_sample=rng.random() < 0.25)
    while work(c)['flops'] > 1e12:         # no more than a large listed case
        c['points'] = max(32, c['points'] // 2)
    if c['points'] > 1000 and rng.random() < 0.3:
        c['chunk'] = c['points'] // rng.randint(2, 4) + 1
    del c['name']
    return c


# ----------------------------------------------------------------------------- sizes
def _network(case):
    return [case['variables']] + [case['neurons']] * case['hidden'] + [1]


def _schema(case):
    return workloads.full_schema(case['variables'], case['order'])


def _disk(case):
    """Radii, angles and boundary points of a Poisson case."""
    interior = case['points'] - 256
    radial = 64 if interior == 4096 else 16
    return radial, interior // radial, 256


def work(case):
    neurons = _network(case)
    pairs = list(zip(neurons, neurons[1:]))
    macs = sum(a * b for a, b in pairs)
    inner = sum(a * b for a, b in pairs[1:])
    params = sum(b * (a + 1) for a, b in pairs)
    if case['call'] == 'poisson':
        columns = 5 * (case['points'] - 256) + 256
        epoch = 2.0 * columns * (2 * macs + inner)
        # points, source and quadrature weights in, every weight read and written
        return {'bytes': case['epochs'] * (4.0 * 2 * columns + 16.0 * case['points'] + 28.0 * params),
                'flops': case['epochs'] * epoch}
    rows, points, v = len(_schema(case)), case['points'], case['variables']
    columns = float(rows) * points
    if case['call'] == 'evaluate':
        return {'bytes': 4.0 * (columns * (v + 1) + params), 'flops': 2.0 * columns * macs}
    # inputs, targets and (per sample) their weights, the weights, the gradient;
    # with an update, its state read and written
    bytes_ = 4.0 * (columns * (v + 1 + (1 if case['per_sample'] else 0)) + 2 * params)
    if case['call'] in ('rprop', 'adam'):
        bytes_ += 24.0 * params
    return {'bytes': bytes_, 'flops': 2.0 * columns * (2 * macs + inner)}


def tolerance(case):
    if case['call'] == 'poisson':
        # RPROP acts on the gradients' signs: over the epochs of a call, an
        # entry near zero may take another turn
        return {'rel': 2e-3, 'max': 0.2}
    if case['call'] in ('rprop', 'adam'):
        # a first update moves every weight by one step along its gradient's
        # sign: an entry near zero may take the other turn
        return {'rel': 1e-3, 'max': 0.2}
    # against 64 bits: outputs 1e-7 to 1.5e-5 (values that cancel), gradients
    # 1e-7 to 1e-6, and up to 2e-5 where they sum over millions of rows
    if case['call'] == 'evaluate':
        return {'rel': 6e-5, 'max': 1e-3}
    return {'rel': 1e-4 if work(case)['flops'] > 1e11 else 1e-5, 'max': 1e-3}


# ----------------------------------------------------------------------------- inputs
def _inputs(case, seed):
    """Points in the unit cube, a Fourier sum and its derivatives on them, the
    cost's weights, and the network's initial weights."""
    rng = np.random.default_rng(seed)
    v, order, n = case['variables'], case['order'], case['points']
    schema = _schema(case)
    points = rng.random((n, v), dtype=np.float32)
    frequency = rng.integers(1, MAX_FREQUENCY + 1, size=(MODES, v)).astype(np.float64)
    amplitude = rng.standard_normal(MODES)
    phase = rng.uniform(0, 2 * np.pi, size=(MODES, v))
    x = torch.from_numpy(points).cuda().double()
    f, p = torch.from_numpy(frequency).cuda(), torch.from_numpy(phase).cuda()
    factor = [[f[:, i, None] ** a * torch.sin(f[:, i, None] * x[None, :, i] + p[:, i, None] + a * math.pi / 2)
               for a in range(order + 1)] for i in range(v)]
    amp = torch.from_numpy(amplitude).cuda()[:, None]
    target = torch.empty(len(schema), n, dtype=torch.float32, device='cuda')
    for r, row in enumerate(schema):
        term = amp
        for i in range(v):
            term = term * factor[i][int(row[1 + i])]
        target[r] = term.sum(0)
    scale = 1.0 / target.double().var(dim=1, unbiased=False).clamp_min(1e-6).cpu().numpy()
    weights = scale.astype(np.float32)
    if case['per_sample']:
        weights = (scale[:, None] * rng.uniform(0.5, 1.5, (1, n))).astype(np.float32)
    init = workloads.xavier_weights(_network(case), seed)
    for w, fan_out in zip(init, _network(case)[1:]):
        w[-fan_out:] = rng.uniform(-0.1, 0.1, fan_out)
    return schema, points, target.cpu().numpy(), weights, init


class _View:
    """Device memory of the framework, as torch sees it without a copy; `owner`
    lives as long as a tensor of it does."""

    def __init__(self, owner, pointer, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {'data': (pointer.value, False), 'shape': tuple(shape), 'typestr': '<f4',
                                         'version': 2}


def _view(owner, pointer, *shape):
    return torch.as_tensor(_View(owner, pointer, shape), device='cuda')


class _Owner:
    """Framework objects, released when the last state and output of theirs is gone."""

    def __init__(self, *release):
        self.release = release

    def __del__(self):
        for f in self.release:
            f()


_shared = {}


def _device():
    """The program's device handle, opened once."""
    if 'device' not in _shared:
        _shared['device'] = hip.Device(0)
    return _shared['device']


def _session():
    """The program's server process, started once."""
    if 'session' not in _shared:
        _shared['session'] = wire.Session(SERVER)
    return _shared['session']


class _Fit:
    """A network, a plan and data for a matching cost."""

    def __init__(self, case, seed):
        schema, points, target, weights, init = _inputs(case, seed)
        neurons = _network(case)
        wl = workloads.MatchingWorkload('case', neurons, points, schema, target, weights, init, chunk=case['chunk'])
        self.call = case['call']
        self.run_ = hip.MatchingRun(_device(), wl)
        self.steps = 0
        owner = _Owner(self.run_.close)
        self.weights, self.gradients = [], [[], []]
        for t in range(len(neurons) - 1):
            for buffer, views in ((0, self.weights), (1, self.gradients[0]), (2, self.gradients[1])):
                pointer, count = self.run_.net.state_ptr(t, buffer)
                views.append(_view(owner, pointer, count))

    def active_gradients(self):
        net = self.run_.net
        return [self.gradients[net.active(t) - 1][t] for t in range(len(self.weights))]

    def run(self):
        run = self.run_
        if self.call == 'rprop':
            run.step(update=True)
            return {'weights': self.weights}
        run.step()
        if self.call == 'adam':
            self.steps += 1
            run.net.adam(self.steps, ADAM_RATE)
            return {'gradients': self.active_gradients(), 'weights': self.weights}
        if self.call == 'loss':
            return {'gradients': self.active_gradients(), 'loss': run.loss()}
        return {'gradients': self.active_gradients()}


class _Evaluation:
    """A network, a forward plan, points and the buffer of their outputs."""

    def __init__(self, case, seed):
        schema, points, _, _, init = _inputs(dict(case, per_sample=False), seed)
        neurons = _network(case)
        device = _device()
        self.rows, self.points = len(schema), len(points)
        self.net = hip.Net(device, neurons, workloads.linear_flags(neurons), init)
        self.width = min(case['chunk'] or self.points, self.points)
        self.plan = hip.Plan(self.net, schema, self.width, backward=False)
        stack = workloads.input_stack(points, schema).transpose(0, 2, 1)
        self.data = hip.Buffer.of(device, np.ascontiguousarray(stack, np.float32))
        self.out = hip.Buffer(device, 4 * self.rows * self.points)
        self.index = np.arange(self.rows, dtype=np.int32)
        owner = _Owner(self.data.free, self.out.free, self.plan.destroy, self.net.destroy)
        self.view = _view(owner, self.out.ptr, self.rows, self.points)

    def run(self):
        for offset in range(0, self.points, self.width):
            valid = min(self.width, self.points - offset)
            self.plan.activate(self.data, self.points, self.index, offset, valid)
            self.plan.forward()
            self.plan.output(self.out, self.points, self.index, offset, valid)
        return {'outputs': self.view}


class _Poisson:
    """The Poisson problem's data, costs and network in the server."""

    def __init__(self, case, seed):
        radial, angular, boundary = _disk(case)
        self.session = _session()
        wl = workloads.PoissonWorkload(tuple(_network(case)), radial, angular, boundary, seed)
        wl.f = workloads.gaussian_source(wl.interior, seed=seed)
        self.ids = wl.upload(self.session)
        self.graph = wl.graph()
        self.epochs = case['epochs']

    def run(self):
        s, net = self.session, self.ids['net']
        result = s.train(net, self.ids['costs'], self.epochs, method=0, log=self.epochs, graph=self.graph)
        _, layers = wire.decode_state(s.snapshot(net))
        return {'reports': [e['values'] for e in result['events'] if 'values' in e],
                'weights': [layer['buffers'][0] for layer in layers]}

    def __del__(self):
        if hasattr(self, 'ids') and not self.session.closed:
            for cost in self.ids['costs']:
                self.session.close_object(2, cost)
            self.session.close_object(1, self.ids['net'])
            for data in (self.ids['interior'], self.ids['boundary']):
                self.session.close_object(0, data)


def prepare(case, seed):
    return {'evaluate': _Evaluation, 'poisson': _Poisson}.get(case['call'], _Fit)(case, seed)


def run(state):
    return state.run()


# ----------------------------------------------------------------------------- 64 bits
def _sigmoid_jet(z, index):
    """Derivatives of sigmoid(z) from those of z, as Taylor coefficients by
    multi-index (y' = (y - y^2) z', order by order)."""
    keys = sorted(index, key=sum)
    zero = keys[0]
    y = {zero: torch.sigmoid(z[zero])}
    u = {zero: y[zero] * (1 - y[zero])}
    for a in keys[1:]:
        i = next(k for k, c in enumerate(a) if c)
        total = 0
        for b in u:
            rest = tuple(p - q for p, q in zip(a, b))
            if min(rest) >= 0 and rest[i] > 0:
                total = total + rest[i] * u[b] * z[rest]
        y[a] = total / a[i]
        square = 0
        for b in list(y):
            rest = tuple(p - q for p, q in zip(a, b))
            if min(rest) >= 0 and rest in y:
                square = square + y[b] * y[rest]
        u[a] = y[a] - square
    return y


def _outputs(blocks, neurons, keys, x):
    """Derivative rows (rows, points) of the network's output at points x."""
    scale = [math.prod(math.factorial(c) for c in k) for k in keys]
    zero = (0,) * x.shape[1]
    rows = []
    for k in keys:
        if sum(k) == 0:
            rows.append(x)
        elif sum(k) == 1:
            rows.append(x.new_tensor(k).expand_as(x))
        else:
            rows.append(torch.zeros_like(x))
    for t, (a, b) in enumerate(zip(neurons, neurons[1:])):
        weight, bias = blocks[t][:a * b].view(a, b), blocks[t][a * b:]
        z = dict(zip(keys, torch.stack(rows) @ weight))
        z[zero] = z[zero] + bias
        if t + 2 < len(neurons):
            z = _sigmoid_jet(z, keys)
        rows = [z[k] for k in keys]
    return torch.stack([r[:, 0] * s for r, s in zip(rows, scale)])


def exact(case, seed):
    if case['call'] in ('poisson', 'rprop'):
        return None   # weights moved along gradients' signs: no measure of rounding
    schema, points, target, weights, init = _inputs(case, seed)
    neurons = _network(case)
    keys = [tuple(int(c) for c in row[1:]) for row in schema]
    blocks = [torch.from_numpy(w).cuda().double().requires_grad_(case['call'] != 'evaluate') for w in init]
    x = torch.from_numpy(points).cuda().double()
    t = torch.from_numpy(target).cuda().double()
    w = torch.from_numpy(weights).cuda().double()
    w = w if w.dim() == 2 else w[:, None].expand(-1, len(points))
    # points at a time, so that the products of the jets (one for each pair of
    # rows b <= a, kept for the backward) fit in memory
    pairs = math.comb(2 * case['variables'] + case['order'], case['order'])
    step = max(64, int(4e10 / (64 * pairs * max(neurons) * len(neurons))))
    loss, rows = 0.0, []
    for i in range(0, len(points), step):
        u = _outputs(blocks, neurons, keys, x[i:i + step])
        if case['call'] == 'evaluate':
            rows.append(u)
            continue
        part = (w[:, i:i + step] * (u - t[:, i:i + step]) ** 2).sum()
        part.backward()
        loss += float(part.detach())
    if case['call'] == 'evaluate':
        return {'outputs': torch.cat(rows, 1)}
    gradients = [b.grad for b in blocks]
    if case['call'] == 'adam':
        return {'gradients': gradients, 'weights': None}
    return {'gradients': gradients, 'loss': loss} if case['call'] == 'loss' else {'gradients': gradients}
