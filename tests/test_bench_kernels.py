"""CPU: the kernels that bench.py reports and summarises exist in the library, by the names a profiler gives them."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import bench
from tianxin_amd.build import LIB


def test_reported_kernels_are_instances_of_the_library():
    syms = subprocess.run(["nm", "-C", LIB], check=True, stdout=subprocess.PIPE, text=True).stdout
    names = [line.split(" ", 2)[2] for line in syms.splitlines() if " txa::" in line or " void txa::" in line]
    names = [n for n in names if "k_" in n and "__device_stub__" not in n]
    assert names
    for k in (bench.FP32_KERNEL, bench.FP64_KERNEL, bench.FP32_KERNEL_GENERAL, *bench.Q2_KERNELS.values(),
              *bench.Q2_GATHER.values(), *bench.Q2_COUNTED.values(), *bench.ELASTIC_KERNELS, "k_dirichlet",
              "k_patch<1, double, false, true, false>", "k_patch<1, float, false, true, true>"):
        hit = {n for n in names if bench._match(n, k)}
        assert len(hit) == 1 if "<" in k else hit, f"{k}: {len(hit)} instances"


def test_match_takes_whole_arguments():
    n = "void txa::(anonymous namespace)::k_a<txa::(anonymous namespace)::Tile<16, 128>, 17, float>(txa::P const*, int)"
    assert bench._match(n, "k_a<Tile<16, 128>, 17, float>") and bench._match(n, "k_a")
    assert not bench._match(n, "k_a<Tile<16, 128>, 1, float>") and not bench._match(n, "k_a<Tile<16, 128>, 17>")
    assert not bench._match(n, "a") and not bench._match(n, "k_")
