"""GPU: the hex27 elasticity line kernel on bricks (calls that want the matrix), FP64.

One to three cells per axis (lines with no, one and two inner cells; every class of nodes on and off the
boundary) and a longer line (several workgroups per line), steady and transient calls, cells of negative
determinant.  R and J against the oracle (1e-12 normwise: only the order of FP64 sums
and the fused products differ), two calls equal bit for bit, one call without f.
"""
import numpy as np
import pytest
import torch

import oracle as O
import tianxin_amd as txa
from tianxin_amd import synth
from test_gpu_parity import Case, dev, rel_err

pytestmark = pytest.mark.gpu
TRANSIENT = dict(transient=True, alpha=2000.0, gamma2=4.0e6, rho=1.4, rayleigh=(0.01, 0.001), src=(0.5, -1.0, 0.25))


@pytest.mark.parametrize("kw", [dict(src=(0.0, 0.0, -1.0)), TRANSIENT])
@pytest.mark.parametrize("nx,ny,nz,mirror", [(1, 1, 1, False), (2, 1, 3, False), (3, 2, 1, True), (2, 3, 2, False),
                                             (13, 1, 2, False)])
def test_brick(engine, nx, ny, nz, mirror, kw):
    X = synth.brick_coords(nx, ny, nz, jitter=0.15, seed=nx + ny) * np.array([-1.0 if mirror else 1.0, 1.0, 1.0])
    c = Case(engine, txa.HEX27, nx, ny, nz, 3, X=X)
    coef = synth.lognormal(61, c.el.shape[0], 0.4)
    st = [synth.uniform(62 + i, c.ndofs, -1, 1) for i in range(3)]
    x, xd, xdd = (st if kw.get("transient") else (st[0], None, None))
    fr, vr = c.oracle(txa.ELASTICITY, coef, nu=0.3, rho=kw.get("rho", 1.0), src=kw["src"],
                      rayleigh=kw.get("rayleigh", (0.0, 0.0))).evaluate(
        x, xd, xdd, alpha=kw.get("alpha", 0.0), beta=1.0, gamma2=kw.get("gamma2", 0.0),
        transient=kw.get("transient", False), mode=O.MODE_EXPLICIT)
    outs = []
    for want_f in (True, True, False):
        f = torch.full((c.ndofs,), np.nan, device="cuda", dtype=torch.float64) if want_f else None
        v = torch.full((c.nnz,), np.nan, device="cuda", dtype=torch.float64)
        c.m.assemble(physics=txa.ELASTICITY, coef=dev(coef), x=dev(x), xdot=None if xd is None else dev(xd),
                     xddot=None if xdd is None else dev(xdd), f=f, vals=v, nu=0.3, **kw)
        torch.cuda.synchronize()
        outs.append((None if f is None else f.cpu().numpy(), v.cpu().numpy()))
    (f0, v0), (f1, v1) = outs[:2]
    assert rel_err(f0, fr) <= 1e-12 and rel_err(v0, vr) <= 1e-12
    assert np.array_equal(f0, f1) and np.array_equal(v0, v1) and np.array_equal(v0, outs[2][1])
    c.m.destroy()
