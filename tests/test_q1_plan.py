"""The slab plan of one-field bricks stays inside the launch limits (host code, no GPU).

Slabs run along the grid's z dimension, which holds 65,536 workgroups: thin bricks of tens of millions of
layers must take taller slabs.  Every plan covers the mesh with slabs of at least one layer.
"""
import os
import subprocess

import pytest

import tianxin_amd as txa
from tianxin_amd.build import CSRC, HERE, HIPCC

GRID_Z = 65536


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "q1_plan_test")
    cpp = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "q1_plan_test.cpp")
    subprocess.run([HIPCC, "-O1", "-std=c++17", "-I" + CSRC, "-I" + os.path.join(HERE, "..", "include"), cpp, "-L" + HERE, "-ltxa",
                    "-Wl,-rpath," + HERE, "-o", exe], check=True)

    def run(meshes):
        args = [str(int(v)) for m in meshes for v in m]
        out = subprocess.run([exe, *args], check=True, stdout=subprocess.PIPE, text=True).stdout
        return [tuple(int(v) for v in line.split()) for line in out.split("\n") if line]

    return run


def test_slabs_fit_the_grid(plan):
    nz = [1, 2, 7, 33, 1000, 65535, 65536, 10 ** 6, 33_600_000, 10 ** 8, 5 * 10 ** 8]
    xy = [(1, 1), (14, 6), (15, 7), (31, 7), (200, 3)]
    meshes = [(t, a, x, y, z, 256) for t, a in [(txa.HEX8, 1), (txa.HEX8, 0), (txa.TET4, 0)] for x, y in xy for z in nz
              if (x + 1) * (y + 1) * (z + 1) < 2 ** 31]   # 32-bit LIDs
    for (t, a, x, y, z, _), (small, zc, zc_f) in zip(meshes, plan(meshes)):
        for h in (zc, zc_f):
            assert 1 <= h <= z + 1 and -(-(z + 1) // h) <= GRID_Z, (t, a, x, y, z, zc, zc_f)
