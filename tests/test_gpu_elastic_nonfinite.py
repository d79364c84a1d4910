"""GPU: non-finite values in the hex8 elasticity brick kernels stay where they belong.

A collapsed layer of cells makes the rows of its own vertices non-finite and no other row; an Inf in the
state of one vertex makes the residual of a corner node of the brick (one cell) the infinity that the
matrix gives, not the NaN of a cell outside the brick that the vertex would also belong to.
"""
import numpy as np
import pytest
import torch

import tianxin_amd as txa
from tianxin_amd import synth
from test_gpu_parity import Case, dev

pytestmark = pytest.mark.gpu
TRANSIENT = dict(transient=True, alpha=4.0, gamma2=16.0, rho=1.5, rayleigh=(0.01, 0.001))
SHEAR = np.array([[1.0, 0.25, 0.125], [0.375, 1.25, 0.25], [0.125, 0.375, 0.875]])   # exact on an integer lattice


def mesh(engine, n, affine, collapsed=None):
    """n cells per axis; collapsed: (axis, layer) of zero thickness."""
    X = synth.brick_coords(*n, hi=n, jitter=0.0 if affine else 0.15, seed=7) @ SHEAR
    if collapsed:
        axis, layer = collapsed
        L = X.reshape(n[2] + 1, n[1] + 1, n[0] + 1, 3)
        lo, hi = ([slice(None)] * 3 for _ in range(2))
        lo[2 - axis], hi[2 - axis] = layer, layer + 1
        if affine:   # the planes above keep their distances
            L[tuple(hi[:2 - axis] + [slice(layer + 1, None)] + hi[3 - axis:])] -= (L[tuple(hi)] - L[tuple(lo)]).reshape(-1, 3)[0]
        else:
            L[tuple(hi)] = L[tuple(lo)]
    c = Case(engine, txa.HEX8, *n, 3, X=X)
    assert bool(c.m.affine) == affine
    return c


def assemble(c, x, kw):
    f = torch.zeros(c.ndofs, device="cuda", dtype=torch.float64)
    v = torch.zeros(c.nnz, device="cuda", dtype=torch.float64)
    st = dict(xdot=dev(synth.uniform(3, c.ndofs, -1, 1)), xddot=dev(synth.uniform(4, c.ndofs, -1, 1))) if kw else {}
    c.m.assemble(physics=txa.ELASTICITY, coef=dev(synth.lognormal(5, c.el.shape[0], 0.3)), x=dev(x), f=f, vals=v, nu=0.3,
                 src=(0.5, -1.0, 0.25), **st, **kw)
    torch.cuda.synchronize()
    return f.cpu().numpy(), v.cpu().numpy()


@pytest.mark.parametrize("kw", [{}, TRANSIENT])
@pytest.mark.parametrize("affine", [True, False])
@pytest.mark.parametrize("axis,layer", [(0, 0), (1, 0), (2, 0), (0, 5)])
def test_collapsed_layer(engine, axis, layer, affine, kw):
    n = (6, 5, 4)
    c = mesh(engine, n, affine, (axis, layer))
    f, v = assemble(c, synth.uniform(2, c.ndofs, -1, 1), kw)
    pt = np.arange(c.ndofs // 3)
    at = (pt % (n[0] + 1), pt // (n[0] + 1) % (n[1] + 1), pt // ((n[0] + 1) * (n[1] + 1)))[axis]
    bad = np.zeros(c.ndofs, bool)
    bad[c.m.point_lids()[(at == layer) | (at == layer + 1)].ravel()] = True
    assert np.array_equal(~np.isfinite(f), bad)
    row = np.repeat(np.arange(c.ndofs), np.diff(c.rp))
    # an entry is summed over the cells that both vertices have in common: non-finite where the layer is among them
    assert np.array_equal(~np.isfinite(v), bad[row] & bad[c.col])
    c.m.destroy()


@pytest.mark.parametrize("kw", [{}, TRANSIENT])
@pytest.mark.parametrize("affine", [True, False])
def test_infinite_state(engine, affine, kw):
    n = (3, 4, 2)
    c = mesh(engine, n, affine)
    lids = c.m.point_lids().reshape(n[2] + 1, n[1] + 1, n[0] + 1, 3)
    x0 = synth.uniform(2, c.ndofs, -1, 1)
    _, K = assemble(c, x0, {})   # the steady matrix: its sign is the sign of dR/du
    for corner in range(8):
        p = [(corner >> d & 1) * n[d] for d in range(3)]
        for axis in range(3):   # the vertex across the corner's cell face normal to this axis
            q = [p[d] if d == axis else p[d] + (1 if p[d] == 0 else -1) for d in range(3)]
            a, b = lids[p[2], p[1], p[0]], lids[q[2], q[1], q[0]]
            x = x0.copy()
            x[b[0]] = np.inf
            f, _ = assemble(c, x, kw)
            for i in range(3):
                k = K[c.rp[a[i]]:c.rp[a[i] + 1]][c.col[c.rp[a[i]]:c.rp[a[i] + 1]] == b[0]][0]
                assert k != 0.0 and f[a[i]] == np.sign(k) * np.inf
    c.m.destroy()
