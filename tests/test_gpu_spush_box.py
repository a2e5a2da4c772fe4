"""The streaming push and its reverse with the sums of neighbouring particles formed in LDS, against the same particles
in a random order (whose workgroups cover too many nodes for that: one atomic per contribution)."""
import numpy as np
import pytest
import torch

import g3d_autograd as ga

pytestmark = pytest.mark.gpu


# rows that begin in mid-box (boxes across the periodic edge in x), a row shorter than a workgroup (boxes as wide as
# the grid), one particle more than whole workgroups, fewer than one workgroup
@pytest.mark.parametrize("nx,ny,count", [(128, 64, 16384), (32, 256, 8193), (512, 32, 16000), (96, 80, 100)])
def test_boxed_sums_against_single_atomics(nx, ny, count):
    r = np.random.default_rng(nx + count)
    dx, dy, h = 0.5, 0.7, 0.25
    hc = ga.HalfCell(nx, ny, dx, dy, 0.0, h, 2, 5.0, 5.0, 5.0, 0.9, 1 / dx)
    k = np.arange(count) + nx // 2
    if count < 128:
        k *= 37                         # far apart: a list in its own order without a box
    x = dx * (0.5 * k % nx + r.uniform(-0.6, 0.6, count))
    y = dy * ((0.5 * k) // nx % ny + r.uniform(-0.6, 0.6, count))
    zeta = 2 * h + h * r.uniform(-0.2, 1.2, count)
    cols = [x, y, zeta, r.uniform(0, 4, count)] + [0.3 * r.standard_normal(count) for _ in range(3)]
    cols[6][::11] = 30.0                # trapped: a second deposit
    fixed = [-np.ones(count), -np.ones(count), 1e-2 * np.ones(count)]
    alive = np.where(zeta < 2 * h, 0, 6).astype(np.int32)
    F = [torch.from_numpy(0.5 * r.standard_normal(6 * nx * ny)).cuda() for _ in range(2)]
    bars = [r.standard_normal(count) for _ in range(7)]
    bJ = torch.from_numpy(r.standard_normal(5 * nx * ny)).cuda()

    def run(order):
        t = [torch.from_numpy(c[order].copy()).cuda() for c in cols + fixed + [alive] + bars]
        leaves = [f.clone().requires_grad_() for f in F] + [c.requires_grad_() for c in t[:7]]
        out = ga.StreamPush.apply(hc, *leaves, *t[7:11])
        grads = torch.autograd.grad(out, leaves, t[11:] + [bJ])
        back = np.argsort(order)
        one = [c.detach().cpu().numpy()[back] for c in list(out[:7]) + list(grads[2:])]
        return one, [c.detach().cpu().numpy() for c in (out[7].reshape(5, -1), *[g.reshape(6, -1) for g in grads[:2]])]

    one, planes = run(np.arange(count))
    one2, planes2 = run(r.permutation(count))
    for a, b in zip(one, one2):
        assert np.array_equal(a, b)     # a particle's own results do not depend on its neighbours
    # a node's sum has some 40 terms at most, each no larger than a few of the plane's largest sum: 40 x 40 roundings
    for a, b in zip(planes, planes2):
        for u, v in zip(a, b):
            assert np.abs(u - v).max() <= 1e-12 * max(np.abs(v).max(), 1e-300)
