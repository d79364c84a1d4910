"""GPU: an infinite coefficient of one tet gives infinite, not undefined, entries.

One tet of a brick has the coefficient Inf: every matrix entry and residual that sums it is Inf or NaN, the diagonal
entries of its vertices +Inf (a sum of squares times the coefficient), everything else finite and unchanged.
"""
import numpy as np
import pytest
import torch

import tianxin_amd as txa
from tianxin_amd import synth
from test_gpu_parity import Case, dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [txa.FP64, txa.FP32])
def test_infinite_coefficient(engine, precision):
    n = (5, 4, 3)
    c = Case(engine, txa.TET4, *n, 1, jitter=0.1, seed=3)
    coef = synth.lognormal(5, c.el.shape[0], 0.3)
    x = dev(synth.uniform(6, c.ndofs, -1, 1))
    tet = 6 * 23 + 2
    out = []
    for k in (coef[tet], np.inf):
        coef[tet] = k
        f = torch.zeros(c.ndofs, device="cuda", dtype=torch.float64)
        v = torch.zeros(c.nnz, device="cuda", dtype=torch.float64)
        g = torch.zeros(c.ndofs, device="cuda", dtype=torch.float64)
        kw = dict(physics=txa.DIFFUSION, precision=precision, coef=dev(coef), x=x, src=(1.0,))
        c.m.assemble(f=f, vals=v, **kw)
        c.m.assemble(f=g, **kw)
        torch.cuda.synchronize()
        out.append((f.cpu().numpy(), v.cpu().numpy(), g.cpu().numpy()))
    (f0, v0, _), (f1, v1, g1) = out
    lids = c.el[tet]
    row = np.repeat(np.arange(c.ndofs), np.diff(c.rp))
    hit = np.isin(row, lids) & np.isin(c.col, lids)
    assert np.all(v1[hit & (row == c.col)] == np.inf)
    assert not np.isfinite(v1[hit]).any() and not np.isfinite(f1[lids]).any() and not np.isfinite(g1[lids]).any()
    # cells are the unit of work: entries of the tet's cell may be undefined, no other
    cell = np.unique(c.el[6 * 23:6 * 24])
    far = ~(np.isin(row, cell) & np.isin(c.col, cell))
    assert np.array_equal(v1[far], v0[far])
    rest = np.setdiff1d(np.arange(c.ndofs), cell)
    assert np.array_equal(f1[rest], f0[rest]) and np.array_equal(g1[rest], f0[rest])
    c.m.destroy()
