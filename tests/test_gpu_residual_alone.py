"""GPU: f of a residual-only call against f of the full call.

Diffusion on bricks (the residual kernel against the row-owner kernel, small and wide tiles): bit for bit in
steady and transient calls, every cell kind and both precisions.
"""
import numpy as np
import pytest
import torch

import tianxin_amd as txa
from tianxin_amd import synth
from test_gpu_parity import Case, dev

pytestmark = pytest.mark.gpu


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
