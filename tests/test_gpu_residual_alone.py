"""GPU: f of a residual-only call against f of the full call.

Diffusion on bricks (the residual kernel against the row-owner kernel, small and wide tiles): bit for bit in
steady and transient calls, every cell kind and both precisions.  hex27 elasticity, FP64, on bricks: the full
call's f comes from the line kernel, f alone from the element kernel and gather (which need no point table:
the sizes that fit a fixed workspace stay what they were), in another order of sums: each entry is a sum of at most 8 cells x
27 points x 81 products, so rounding grows to about 1.1e-16 sqrt(17496) = 1.5e-14; 1e-13 normwise allowed.
"""
import numpy as np
import pytest
import torch

import oracle as O
import tianxin_amd as txa
from tianxin_amd import synth
from test_gpu_parity import Case, dev, rel_err

pytestmark = pytest.mark.gpu
TRANSIENT = dict(transient=True, alpha=2000.0, gamma2=4.0e6, rho=1.4, rayleigh=(0.01, 0.001))


def both(c, **kw):
    out = []
    for want in (True, False):
        f = torch.full((c.ndofs,), np.nan, device="cuda", dtype=torch.float64)
        v = torch.full((c.nnz,), np.nan, device="cuda", dtype=torch.float64) if want else None
        c.m.assemble(f=f, vals=v, **kw)
        torch.cuda.synchronize()
        out.append(f.cpu().numpy())
    return out


# (topology, cells, jitter): one tile and several of each shape, one and several slabs
@pytest.mark.parametrize("topo,n,jitter", [(txa.HEX8, (14, 6, 3), 0.0), (txa.HEX8, (40, 33, 17), 0.0), (txa.HEX8, (14, 6, 3), 0.1),
                                           (txa.HEX8, (62, 34, 21), 0.1), (txa.TET4, (14, 6, 3), 0.1),
                                           (txa.TET4, (62, 34, 21), 0.1)])
@pytest.mark.parametrize("precision", [txa.FP64, txa.FP32])
@pytest.mark.parametrize("transient", [False, True])
def test_diffusion_bitwise(engine, topo, n, jitter, precision, transient):
    c = Case(engine, topo, *n, 1, jitter=jitter, seed=n[0])
    x, xd = (dev(synth.uniform(32 + i, c.ndofs, -1, 1)) for i in range(2))
    full, alone = both(c, physics=txa.DIFFUSION, precision=precision, coef=dev(synth.lognormal(31, c.el.shape[0], 0.5)), x=x,
                       xdot=xd if transient else None, transient=transient, alpha=3.0 if transient else 0.0, rho=1.3,
                       src=(0.7, 0.0, 0.0))
    assert np.isfinite(full).all() and np.array_equal(alone, full)
    c.m.destroy()


@pytest.mark.parametrize("kw", [dict(src=(0.0, 0.0, -1.0)), dict(src=(0.5, -1.0, 0.25), **TRANSIENT)])
@pytest.mark.parametrize("n", [(1, 1, 1), (3, 2, 4), (7, 5, 6)])
def test_hex27_elasticity_fp64(engine, n, kw):
    c = Case(engine, txa.HEX27, *n, 3, jitter=0.1, seed=n[0])
    coef = synth.lognormal(61, c.el.shape[0], 0.4)
    st = [synth.uniform(62 + i, c.ndofs, -1, 1) for i in range(3)]
    x, xd, xdd = (st if kw.get("transient") else (st[0], None, None))
    full, alone = both(c, physics=txa.ELASTICITY, coef=dev(coef), x=dev(x), xdot=None if xd is None else dev(xd),
                       xddot=None if xdd is None else dev(xdd), nu=0.3, **kw)
    fr, _ = c.oracle(txa.ELASTICITY, coef, nu=0.3, rho=kw.get("rho", 1.0), src=kw["src"],
                     rayleigh=kw.get("rayleigh", (0.0, 0.0))).evaluate(
        x, xd, xdd, alpha=kw.get("alpha", 0.0), beta=1.0, gamma2=kw.get("gamma2", 0.0),
        transient=kw.get("transient", False), mode=O.MODE_EXPLICIT)
    assert rel_err(alone, fr) <= 1e-12 and rel_err(full, fr) <= 1e-12
    assert rel_err(alone, full) <= 1e-13
    c.m.destroy()
