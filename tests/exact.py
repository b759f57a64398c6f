"""Networks and matching costs in float64 (torch, autograd), on the Taylor
coefficients of every row: what the fp32 kernels are rounded from.  A network's
sigmoid layers take y' = u z', u = y - y y, coefficient by coefficient of the
truncated series; schemas hold every multi-index below one of theirs."""
import math

import numpy as np
import torch


def _sigmoid(z, keys):
    y, u = {}, {}
    for a in sorted(keys, key=sum):
        if sum(a) == 0:
            y[a] = torch.sigmoid(z[a])
            u[a] = y[a] * torch.sigmoid(-z[a])
            continue
        i = next(k for k, c in enumerate(a) if c)
        pairs = [(b, tuple(p - q for p, q in zip(a, b))) for b in y]
        y[a] = sum(rest[i] * u[b] * z[rest] for b, rest in pairs if min(rest) >= 0 and rest[i] > 0) / a[i]
        u[a] = y[a] - sum(y[b] * y[rest] for b, rest in pairs + [(a, (0,) * len(a))] if rest in y)
    return y


def outputs(neurons, schema, blocks, points):
    """Rows (rows, points, outputs) of the network's derivatives at `points`;
    `blocks` are float64 tensors in the library's layout, W[o + n_out * i] then b."""
    keys = [tuple(int(c) for c in row[1:]) for row in schema]
    factorial = [math.prod(math.factorial(c) for c in k) for k in keys]
    rows = [points if sum(k) == 0 else points.new_tensor(k).expand_as(points) if sum(k) == 1 else torch.zeros_like(points)
            for k in keys]
    for t, (n, m) in enumerate(zip(neurons, neurons[1:])):
        w, bias = blocks[t][:n * m].view(n, m), blocks[t][n * m:]
        z = {k: r @ w + (bias if sum(k) == 0 else 0) for k, r in zip(keys, rows)}
        if t + 2 < len(neurons):
            z = _sigmoid(z, keys)
        rows = [z[k] for k in keys]
    return torch.stack([r * f for r, f in zip(rows, factorial)])


def epoch(wl, device='cuda', step=512):
    """Loss and gradient blocks of a single-output MatchingWorkload of a full
    (or closed) schema with weights per row."""
    blocks = [torch.as_tensor(np.asarray(b), dtype=torch.float64, device=device).requires_grad_() for b in wl.init]
    x = torch.as_tensor(np.asarray(wl.points), dtype=torch.float32, device=device).double()
    target = torch.as_tensor(np.asarray(wl.target, np.float32), device=device).double()
    weights = torch.as_tensor(np.asarray(wl.weight_block(), np.float32), device=device).double().reshape(wl.rows, -1)
    loss = 0.0
    for i in range(0, len(x), step):
        y = outputs(wl.neurons, wl.schema, blocks, x[i:i + step])[..., 0]
        part = (weights * (y - target[:, i:i + step]) ** 2).sum()
        part.backward()
        loss += float(part.detach())
    return loss, [b.grad.cpu().numpy() for b in blocks]
