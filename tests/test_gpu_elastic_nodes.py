"""GPU: the hex8 elasticity node kernels on general cells, FP64 (bricks and uploads).

Sizes at the edges of the brick kernel's 4 x 4 node tiles (one to nine nodes along x and y) and of
the upload kernel's two nodes per wave and eight instances at a time (an odd node count; every
cell listed twice, sixteen instances per node), cells of negative determinant, steady and transient calls.  R and J
against the oracle (1e-12 normwise: only the order of FP64 sums and the fused products differ), f
alone equal to the full call's, two calls equal bit for bit.
"""
import numpy as np
import pytest
import torch

import oracle as O
import tianxin_amd as txa
from tianxin_amd import synth
from test_gpu_parity import Case, dev, rel_err, run_both

pytestmark = pytest.mark.gpu
TRANSIENT = dict(transient=True, alpha=2000.0, gamma2=4.0e6, rho=1.4, rayleigh=(0.01, 0.001), src=(0.5, -1.0, 0.25))


def check(m, ndofs, nnz, coef, x, xd, xdd, fr, vr, **kw):
    outs = []
    for want in (True, True, False):
        f = torch.full((ndofs,), np.nan, device="cuda", dtype=torch.float64)
        v = torch.full((nnz,), np.nan, device="cuda", dtype=torch.float64) if want else None
        m.assemble(physics=txa.ELASTICITY, coef=dev(coef), x=dev(x), xdot=None if xd is None else dev(xd),
                   xddot=None if xdd is None else dev(xdd), f=f, vals=v, nu=0.3, **kw)
        torch.cuda.synchronize()
        outs.append((f.cpu().numpy(), None if v is None else v.cpu().numpy()))
    (f0, v0), (f1, v1), (f2, _) = outs
    assert rel_err(f0, fr) <= 1e-12 and rel_err(v0, vr) <= 1e-12
    assert np.array_equal(f0, f1) and np.array_equal(v0, v1) and np.array_equal(f0, f2)


@pytest.mark.parametrize("kw", [dict(src=(0.0, 0.0, -1.0)), TRANSIENT])
@pytest.mark.parametrize("nx,ny,nz", [(2, 2, 2), (3, 4, 2), (4, 3, 3), (7, 8, 2), (8, 2, 5)])
def test_brick_general_cells(engine, nx, ny, nz, kw):
    c = Case(engine, txa.HEX8, nx, ny, nz, 3, jitter=0.2, seed=nx + ny)
    assert not c.m.affine
    coef = synth.lognormal(41, c.el.shape[0], 0.4)
    st = [synth.uniform(42 + i, c.ndofs, -1, 1) for i in range(3)]
    x, xd, xdd = (st if kw.get("transient") else (st[0], None, None))
    fr, vr = c.oracle(txa.ELASTICITY, coef, nu=0.3, rho=kw.get("rho", 1.0), src=kw["src"],
                      rayleigh=kw.get("rayleigh", (0.0, 0.0))).evaluate(
        x, xd, xdd, alpha=kw.get("alpha", 0.0), beta=1.0, gamma2=kw.get("gamma2", 0.0),
        transient=kw.get("transient", False), mode=O.MODE_EXPLICIT)
    check(c.m, c.ndofs, c.nnz, coef, x, xd, xdd, fr, vr, **kw)
    c.m.destroy()


def test_brick_mirrored_cells(engine):
    # a left-handed lattice: every determinant negative, the measure positive
    n = 5
    X = synth.brick_coords(n, n, n, jitter=0.1, seed=3) * np.array([-1.0, 1.0, 1.0])
    c = Case(engine, txa.HEX8, n, n, n, 3, X=X)
    f, v, fr, vr = run_both(engine, c, txa.ELASTICITY, **TRANSIENT)
    assert rel_err(f, fr) <= 1e-12 and rel_err(v, vr) <= 1e-12
    c.m.destroy()


@pytest.mark.parametrize("kw", [dict(src=(0.0, 0.0, -1.0)), TRANSIENT])
@pytest.mark.parametrize("mesh", ["one", "odd", "shuffled", "twice"])
def test_upload(engine, mesh, kw):
    n = {"one": (1, 1, 1), "odd": (2, 4, 6), "shuffled": (5, 4, 7), "twice": (3, 3, 4)}[mesh]
    conn, _, _ = O.brick_mesh(O.HEX8, *n)
    X = synth.brick_coords(*n, jitter=0.2, seed=9)
    if mesh == "shuffled":
        conn = conn[np.random.default_rng(4).permutation(conn.shape[0])]
    if mesh == "twice":   # two materials in the same cells: up to sixteen instances per node
        conn = np.concatenate([conn, conn])
    m = engine.upload(txa.HEX8, conn, X)
    ndofs, nnz = m.build_dofmap(3), m.build_graph()
    _, owned, el = O.dofmap(conn, 3)
    rp, col = O.graph(el, owned.size)
    coef = synth.lognormal(51, conn.shape[0], 0.4)
    st = [synth.uniform(52 + i, ndofs, -1, 1) for i in range(3)]
    x, xd, xdd = (st if kw.get("transient") else (st[0], None, None))
    A = O.Assembler(O.HEX8, txa.ELASTICITY, conn, X, el, coef, rp, col, nu=0.3, rho=kw.get("rho", 1.0), src=kw["src"],
                    rayleigh=kw.get("rayleigh", (0.0, 0.0)))
    fr, vr = A.evaluate(x, xd, xdd, alpha=kw.get("alpha", 0.0), beta=1.0, gamma2=kw.get("gamma2", 0.0),
                        transient=kw.get("transient", False), mode=O.MODE_EXPLICIT)
    check(m, ndofs, nnz, coef, x, xd, xdd, fr, vr, **kw)
    m.destroy()
