// Prints the slab plan of one-field bricks, one line per mesh: vertex layers per slab of the row-owner
// kernel and of the residual kernel.  Host code only.  Arguments: topology, affine, nx, ny, nz, CUs, repeated.
#include <cstdio>
#include <cstdlib>

#include "txa.h"
#include "txa_internal.hpp"

int main(int argc, char **argv) {
  for (int i = 1; i + 5 < argc; i += 6) {
    txa::Mesh m;
    m.topo = std::atoi(argv[i]);
    m.affine = std::atoi(argv[i + 1]) != 0;
    m.nx = std::atoi(argv[i + 2]);
    m.ny = std::atoi(argv[i + 3]);
    m.nz = std::atoi(argv[i + 4]);
    const txa::Q1Plan p = txa::q1_plan(m, std::atoi(argv[i + 5]));
    std::printf("%d %d %d\n", p.small ? 1 : 0, p.zc, p.zc_f);
  }
  return 0;
}
