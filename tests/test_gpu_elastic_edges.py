"""GPU: elasticity bricks one cell wide with general cells, accumulating and allocation-free hex27 FP64 calls.

Every vertex of a brick of 1, 1 x 4 x 3 and 5 x 1 x 2 cells is moved (the jittered bricks of the other tests
move interior vertices, which these do not have): R and J against the oracle (1e-12 normwise, only the order of
FP64 sums and the fused products differ).  hex27 FP64: accumulate adds the staged rows behind the line kernel's
point table, and the static workspace of the allocation-free call holds that table; both exactly txa_assemble's.
"""
import numpy as np
import pytest
import torch

import tianxin_amd as txa
from tianxin_amd import synth
from test_gpu_parity import Case, dev, rel_err, run_both

pytestmark = pytest.mark.gpu
TRANSIENT = dict(transient=True, alpha=2000.0, gamma2=4.0e6, rho=1.4, rayleigh=(0.01, 0.001), src=(0.5, -1.0, 0.25))


def moved(n, seed):
    X = synth.brick_coords(*n)
    return X + (np.random.default_rng(seed).random(X.shape) - 0.5) * (0.3 / np.array(n))


@pytest.mark.parametrize("kw", [dict(src=(0.0, 0.0, -1.0)), TRANSIENT])
@pytest.mark.parametrize("topo", [txa.HEX8, txa.HEX27])
@pytest.mark.parametrize("n", [(1, 1, 1), (1, 4, 3), (5, 1, 2)])
def test_one_cell_wide(engine, n, topo, kw):
    c = Case(engine, topo, *n, 3, X=moved(n, 11))
    assert not c.m.affine
    f, v, fr, vr = run_both(engine, c, txa.ELASTICITY, seed=12, **dict(kw, nu=0.3))
    assert rel_err(f, fr) <= 1e-12 and rel_err(v, vr) <= 1e-12
    c.m.destroy()


def outputs(c):
    return (torch.full((c.ndofs,), np.nan, device="cuda", dtype=torch.float64),
            torch.full((c.nnz,), np.nan, device="cuda", dtype=torch.float64))


@pytest.mark.parametrize("transient", [False, True])
@pytest.mark.parametrize("n", [(1, 1, 1), (3, 2, 4)])
def test_hex27_fp64_accumulate_and_noalloc(engine, n, transient):
    c = Case(engine, txa.HEX27, *n, 3, X=moved(n, 13))
    st = [dev(synth.uniform(62 + i, c.ndofs, -1, 1)) for i in range(3)]
    kw = dict(physics=txa.ELASTICITY, coef=dev(synth.lognormal(61, c.el.shape[0], 0.4)), x=st[0], nu=0.3, src=(0.5, -1.0, 0.25))
    if transient:
        kw.update(TRANSIENT, xdot=st[1], xddot=st[2])
    f1, v1 = outputs(c)
    c.m.assemble(f=f1, vals=v1, **kw)
    f2, v2 = torch.zeros_like(f1), torch.zeros_like(v1)
    for _ in range(2):
        c.m.assemble(f=f2, vals=v2, accumulate=True, **kw)
    f3, v3 = outputs(c)
    c.m.assemble_noalloc(f=f3, vals=v3, **kw)
    f4, v4 = torch.zeros_like(f1), torch.zeros_like(v1)
    c.m.assemble_noalloc(f=f4, vals=v4, accumulate=True, **kw)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(f1).all()) and bool(torch.isfinite(v1).all())
    assert torch.equal(f2, 2 * f1) and torch.equal(v2, 2 * v1)
    assert torch.equal(f3, f1) and torch.equal(v3, v1)
    assert torch.equal(f4, f1) and torch.equal(v4, v1)
    c.m.destroy()
