// Linear elasticity, element-centric: hex8 (Q1) and hex27 (Q2), three fields.
//
// Replaces, for the displacement equation set, the chain
//   GatherSolution_Tpetra (+ seeds) -> DOFGradient -> stress -> Integrator_GradBasisDotVector,
//   Integrator_BasisTimesScalar (body force, inertia) -> ScatterResidual_Tpetra<Jacobian>
// (disc-fe/src/evaluators/Panzer_GatherSolution_Tpetra_impl.hpp:549-650,
//  Panzer_DOFGradient_impl.hpp:60-160, Panzer_Integrator_GradBasisDotVector_impl.hpp:225-294,
//  Panzer_Integrator_BasisTimesScalar_impl.hpp:215-296,
//  Panzer_ScatterResidual_Tpetra_impl.hpp:446-520), with the Sacado-FAD element
// Jacobian replaced by the explicit tangent
//   J_e = beta K + alpha (a_R M + b_R K) + gamma2 M,   R_e = K u + C v + M a - F.
//
// One workgroup per element (grid-stride).  The reference element is the
// tensor product of 1D Gauss rules and Lagrange bases (tables in LDS), so no
// per-point tables are read from memory.  Geometry (J, det J, J^-1) is FP64 at
// every quadrature point.  The element stiffness is assembled from the
// gradient Gram matrix
//   T[(k,a),(l,b)] = sum_q w_q |det J_q| dN_a/dx_k dN_b/dx_l        (3 NB x 3 NB),
//   K[(a,i),(b,j)] = lambda T[(i,a),(j,b)] + mu T[(j,a),(i,b)] + delta_ij mu sum_k T[(k,a),(k,b)],
// i.e. B^T D B for isotropic D written as one symmetric product G^T W G.  T is
// computed on the matrix cores: T = A^T G with A = w det J G in FP64
// (v_mfma_f64_16x16x4f64) or FP32 (v_mfma_f32_16x16x4f32), or as T = O^T O with
// O = sqrt(w |det J|) G by bf16 MFMA (v_mfma_f32_16x16x32_bf16) on a three-way split of
// each FP32 operand (x = x0 + x1 + x2, every x_s in bf16) keeping the six cross products
// of order <= 2^-16, accumulated in FP32.
//
// hex8 in FP64 (parallelepiped bricks in every precision) and hex27 bricks in FP64 with the matrix
// skip both phases: the node and line kernels below form rows directly and need no element blocks.
//
// Assembly into the CRS is two-phase.  The element kernel writes each element's
// Jacobian block (FP32, FP64 in FP64 mode) and residual (FP64) to a workspace,
// coalesced; a node-centric gather then sums, for every node, the blocks of the
// elements around it into the node's three CRS rows in FP64, in a fixed element
// order, and writes each row once.  No global-memory atomics (the gather's LDS adds
// run in one wave's program order): results are bitwise reproducible.
// The row position of every (node, neighbour) pair comes from a per-node table
// built with the graph.
#include <map>
#include <type_traits>

#include "txa_internal.hpp"

namespace txa {
namespace {

constexpr int MODE_F64 = 0, MODE_F32 = 1, MODE_SPLIT = 2;

struct ElasticParams {
  int nq;
  int64_t nelem;
  int64_t e0, e1;               // elements [e0, e1) of this launch
  int nconn;
  const int64_t *conn;          // the first 8 entries of an element are its vertices
  const double *X, *Y, *Z;
  const int32_t *elem_lid;      // [E][3 NB]: node-major, field-minor
  const double *coef;           // Young's modulus per element
  double nu, rho, src[3], ra, rb;
  const double *x, *xdot, *xddot;
  double alpha, beta, gamma2;
  int transient;
  void *jbuf;        // element Jacobian blocks [E][NB][block_stride(NB)], node-major: node a holds the
                     // rows of DOFs (a, 0), (a, 1), (a, 2), each over the Gram columns j NB + b = DOF
                     // (b, j), then zero padding (FP32, FP64 in FP64 mode); null: none
  double *rbuf;      // element residuals [E][ND]; null: none
};

// Entries per node in the workspace block: the node's three rows (9 NB entries), padded for
// hex27 to 256 so every node's rows start on a 1 KiB boundary (FP32) and the gather reads
// whole cache lines; hex8's 72 entries stay unpadded.
__host__ __device__ constexpr int block_stride(int NB) { return NB == 27 ? 256 : 9 * NB; }

// lattice offsets of the element's nodes: shards vertex order (hex8), Q2 order (hex27)
__device__ const int8_t kHexV[8][3] = {{0, 0, 0}, {1, 0, 0}, {1, 1, 0}, {0, 1, 0},
                                       {0, 0, 1}, {1, 0, 1}, {1, 1, 1}, {0, 1, 1}};
__device__ const int8_t kQ2[27][3] = {
    {0, 0, 0}, {2, 0, 0}, {2, 2, 0}, {0, 2, 0}, {0, 0, 2}, {2, 0, 2}, {2, 2, 2}, {0, 2, 2},
    {1, 0, 0}, {2, 1, 0}, {1, 2, 0}, {0, 1, 0}, {1, 0, 2}, {2, 1, 2}, {1, 2, 2}, {0, 1, 2},
    {0, 0, 1}, {2, 0, 1}, {2, 2, 1}, {0, 2, 1},
    {1, 0, 1}, {2, 1, 1}, {1, 2, 1}, {0, 1, 1}, {1, 1, 0}, {1, 1, 2}, {1, 1, 1}};

typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef double v4d __attribute__((ext_vector_type(4)));

// bf16 with round-to-nearest-even, returned as its bit pattern and its value
__device__ __forceinline__ short bf16_rne(float x, float &v) {
  const __bf16 h = static_cast<__bf16>(x);   // v_cvt_pk_bf16_f32
  const short s = __builtin_bit_cast(short, h);
  v = __uint_as_float(static_cast<uint32_t>(static_cast<uint16_t>(s)) << 16);
  return s;
}

// x = x0 + x1 + x2 with bf16 parts (exact up to ~2^-24 |x|)
__device__ __forceinline__ void split3(float x, short &s0, short &s1, short &s2) {
  asm("" : "+v"(x));   // rounded to FP32 first: converted straight from FP64, x0 differs now and then
  float v0, v1, v2;
  s0 = bf16_rne(x, v0);
  const float r1 = x - v0;
  s1 = bf16_rne(r1, v1);
  const float r2 = r1 - v1;
  s2 = bf16_rne(r2, v2);
}

// One DPP lane move of an FP64 value (both halves); lanes of rows outside row_mask get 0.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_f64(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, ROW_MASK, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, ROW_MASK, 0xf, false);
  return __hiloint2double(hi, lo);
}

// Fixed-order sum over groups of GW (8 or 32) consecutive lanes, on the VALU (DPP):
// quad swaps (lanes ^1, ^2), the half-row mirror (8 lanes) and the row mirror (16
// lanes); for 32 lanes the first row's total is then broadcast into the second row.
// The group sum ends in every lane of the group (GW = 8) or in its second row (GW = 32).
template <int GW>
__device__ __forceinline__ double group_sum(double x) {
  x += dpp_f64<0xB1, 0xf>(x);    // quad_perm [1,0,3,2]
  x += dpp_f64<0x4E, 0xf>(x);    // quad_perm [2,3,0,1]
  x += dpp_f64<0x141, 0xf>(x);   // row_half_mirror
  if constexpr (GW == 32) {
    x += dpp_f64<0x140, 0xf>(x);   // row_mirror
    x += dpp_f64<0x142, 0xa>(x);   // row_bcast15 into rows 1 and 3
  }
  return x;
}

template <int NB>
struct Dims {
  static constexpr int ND = 3 * NB;                    // element DOFs
  static constexpr int R = NB == 8 ? 1 : 2;            // lattice reach of a node's neighbours
  static constexpr int S = 2 * R + 1;
  static constexpr int MP = (ND + 15) / 16 * 16;       // padded operand rows (MFMA)
  static constexpr int KP = 32;                        // padded quadrature dimension (MFMA)
  // LDS row stride of the operand parts, in bf16: 40 (80 B) puts the 16 rows of an
  // MFMA tile on distinct bank pairs (a 64 B stride put them on two banks: 8-way
  // conflicts on every operand read) and keeps rows 16-byte aligned
  static constexpr int KS = 40;
  // FP64 form: quadrature dimension padded to the 4 of v_mfma_f64_16x16x4f64, and an odd
  // LDS row stride in doubles (the 16 rows of an operand read fall on distinct bank pairs)
  static constexpr int KP64 = NB == 8 ? 8 : 28;
  static constexpr int KS64 = KP64 + 1;
  // FP32 form: the same padding for v_mfma_f32_16x16x4f32; a row stride in floats whose 16
  // multiples are distinct multiples of 4 modulo the 64 banks, so the 16 rows x 4 points of an
  // operand read fall on 64 distinct banks
  static constexpr int KS32 = NB == 8 ? 12 : 36;
};

template <int NB, int NQ, int MODE>
struct Smem {
  using D = Dims<NB>;
  using TReal = typename std::conditional<MODE == MODE_F64, double, float>::type;
  // 1D tables on [-1, 1]: Gauss rule, field basis (2 or 3 nodes) and the linear
  // geometry basis, values and derivatives at each Gauss point
  double bL[3][3], bdL[3][3], gL[2][3], gdL[2][3], w1[3];
  int8_t off[NB][3];         // lattice offset of each element node
  double X[8][3];
  double Ji[NQ][9];
  double det[NQ];
  double wm[NQ];             // w det J (the sign of the first point is applied where used)
  double sw[NQ];             // sqrt(w |det J|)
  double u[D::ND], v[D::ND], a[D::ND], r[D::ND];
  TReal M[NB][NB];
  double fa[3][NB];          // integral of each basis function, by plane of points
  // VALU modes: gradients G and the Gram matrix T.  MFMA mode: the bf16 operand
  // parts, then T over the same bytes once the products are in registers.  The
  // operand rows are read as 8-byte vectors: the union is 16-byte aligned whatever
  // the fields before it add up to.
  // FP64 rows are not padded (81 doubles is already an odd bank stride), which keeps
  // the FP64 form under half of a CU's LDS: two workgroups per CU.
  static constexpr int TP = MODE == MODE_F64 ? D::ND : D::ND + 1;
  // (the bf16 MFMA form uses neither T nor G of `v`, the FP64 form no G: they shrink to one entry)
  static constexpr int VR = MODE == MODE_SPLIT ? 1 : D::ND;
  union alignas(16) {
    struct {
      TReal T[VR][TP];
      TReal G[1];
    } v;
    short ops[3 * D::MP * D::KS];
    float T32[D::ND][D::ND + 1];
    // FP64 form: the operands of T = A^T B, A = (w det sgn) G and B = G, rows (k, a) padded
    // to MP, points padded to KP64 (zero); T goes over them once the products are in registers
    double opd[MODE == MODE_F64 ? 2 * D::MP * D::KS64 : 1];
    // FP32 form: the same operands in FP32 for v_mfma_f32_16x16x4f32
    float opf[MODE == MODE_F32 ? 2 * D::MP * D::KS32 : 1];
  } w;
};

// Bound by VALU issue and, beside the gather, by the block stores.  The FP32 and split hex27 forms are held
// to three waves per SIMD (162 VGPRs; at four, 128 and 29 spilled, the split form takes 7.93 ms).  64^3
// with the gather, against blocks staged in LDS and copied out after the pair phase, five-step sums of
// every residual value, the source load per DOF by one thread and the bf16 parts by integer rounding:
// split 7.86 -> 7.18 ms, FP32 8.34 -> 7.66 ms (its own stores cached: 8.33 ms).
template <int NB, int NQ, int BS, int MODE>
__global__ __launch_bounds__(BS, MODE == MODE_F64 || NB == 8 ? 1 : 3) void k_elastic(ElasticParams p) {
  using D = Dims<NB>;
  using TReal = typename Smem<NB, NQ, MODE>::TReal;
  constexpr int ND = D::ND;
  constexpr int Q1 = NQ == 27 ? 3 : 2;        // Gauss points per axis
  // final phase: lane (a, b) forms the 3x3 block of node pair (a, b); a group of GW
  // lanes shares a and runs over b
  constexpr int GW = NB == 27 ? 32 : 8;
  constexpr int GPW = 64 / GW;
  constexpr int AP = (BS / 64) * GPW;          // nodes a per pass
  constexpr int NPASS = (NB + AP - 1) / AP;
  __shared__ Smem<NB, NQ, MODE> sm;
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  const int gb = lane % GW, ga = wave * GPW + lane / GW;
  const bool tr = p.transient && p.xdot;
  const bool tra = tr && p.xddot;
  const bool has_src = p.src[0] != 0.0 || p.src[1] != 0.0 || p.src[2] != 0.0;

  if (t == 0) {
    // Gauss-Legendre on [-1, 1]; Lagrange bases on the nodes {-1, 1} or {-1, 0, 1}
    const double g3 = 0.77459666924148337704;   // sqrt(3/5)
    const double g2 = 0.57735026918962576451;   // 1/sqrt(3)
    for (int q = 0; q < Q1; ++q) {
      const double xi = Q1 == 3 ? (q - 1) * g3 : (2 * q - 1) * g2;
      sm.w1[q] = Q1 == 3 ? (q == 1 ? 8.0 / 9.0 : 5.0 / 9.0) : 1.0;
      sm.gL[0][q] = 0.5 * (1.0 - xi);
      sm.gL[1][q] = 0.5 * (1.0 + xi);
      sm.gdL[0][q] = -0.5;
      sm.gdL[1][q] = 0.5;
      if (NB == 27) {
        sm.bL[0][q] = 0.5 * xi * (xi - 1.0);
        sm.bL[1][q] = 1.0 - xi * xi;
        sm.bL[2][q] = 0.5 * xi * (xi + 1.0);
        sm.bdL[0][q] = xi - 0.5;
        sm.bdL[1][q] = -2.0 * xi;
        sm.bdL[2][q] = xi + 0.5;
      } else {
        sm.bL[0][q] = sm.gL[0][q];
        sm.bL[1][q] = sm.gL[1][q];
        sm.bdL[0][q] = -0.5;
        sm.bdL[1][q] = 0.5;
      }
    }
  }
  for (int i = t; i < NB * 3; i += BS) sm.off[i / 3][i % 3] = NB == 8 ? kHexV[i / 3][i % 3] : kQ2[i / 3][i % 3];
  __syncthreads();

  // Gather data of the element after this one, fetched while this one is computed: the
  // coordinates, state and coefficient (thread t < 24: one vertex coordinate; t < ND:
  // one DOF) beside the Gram matrix, from the connectivity and LIDs fetched one element
  // earlier; they are waited for before the pair phase and put in LDS after it.
  // No global load is then pending when the block stores go out, so the next element
  // starts without waiting for those stores (one counter tracks both).  The loads have
  // no branch (indices clamped to a valid element and lane; the extra values are not
  // used): a conditional load would be copied, and so waited for, where the branch joins.
  static_assert(BS >= ND && BS >= 24, "one gather entry per thread");
  int64_t gn = 0;
  int32_t gL = 0;
  double gX = 0.0, gu = 0.0, gv = 0.0, gac = 0.0, gE = 0.0;
  auto fetch_index = [&](int64_t e) {
    const int64_t ec = e < p.e1 ? e : p.e1 - 1;
    gn = p.conn[ec * p.nconn + min(t, 23) / 3];
    gL = p.elem_lid[ec * ND + min(t, ND - 1)];
  };
  auto fetch_data = [&](int64_t e) {
    const int64_t ec = e < p.e1 ? e : p.e1 - 1;
    const int d = t % 3;
    const double *P = d == 0 ? p.X : (d == 1 ? p.Y : p.Z);
    gX = P[gn];
    gu = p.x[gL];
    gv = tr ? p.xdot[gL] : 0.0;
    gac = tra ? p.xddot[gL] : 0.0;
    gE = p.coef[ec];
  };
  auto put_data = [&]() {
    if (t < 24) sm.X[t / 3][t % 3] = gX;
    if (t < ND) {
      sm.u[t] = gu;
      sm.v[t] = gv;
      sm.a[t] = gac;
    }
    asm volatile("" : "+v"(gE));   // the coefficient is taken here too, not after the block store
  };
  fetch_index(p.e0 + blockIdx.x);
  fetch_data(p.e0 + blockIdx.x);
  put_data();
  double E = gE;
  fetch_index(p.e0 + blockIdx.x + gridDim.x);

  for (int64_t e = p.e0 + blockIdx.x; e < p.e1; e += gridDim.x) {
    __syncthreads();   // this element's vertices and state are in LDS
    // ---- geometry (FP64)
    if (t < NQ) {
      const int qx = t % Q1, qy = (t / Q1) % Q1, qz = t / (Q1 * Q1);
      double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll
      for (int vtx = 0; vtx < 8; ++vtx) {
        const int ox = kHexV[vtx][0], oy = kHexV[vtx][1], oz = kHexV[vtx][2];
        const double gx = sm.gL[ox][qx], gy = sm.gL[oy][qy], gz = sm.gL[oz][qz];
        const double d[3] = {sm.gdL[ox][qx] * gy * gz, gx * sm.gdL[oy][qy] * gz, gx * gy * sm.gdL[oz][qz]};
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int j = 0; j < 3; ++j) J[i][j] += sm.X[vtx][i] * d[j];
      }
      const double c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
      const double c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2];
      const double c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
      const double det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
      const double id = 1.0 / det;
      double *Ji = sm.Ji[t];
      Ji[0] = c00 * id;
      Ji[1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * id;
      Ji[2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * id;
      Ji[3] = c01 * id;
      Ji[4] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * id;
      Ji[5] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * id;
      Ji[6] = c02 * id;
      Ji[7] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * id;
      Ji[8] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * id;
      sm.det[t] = det;
      sm.wm[t] = sm.w1[qx] * sm.w1[qy] * sm.w1[qz] * det;
    }
    if constexpr (MODE == MODE_SPLIT) {
      // operand rows >= ND are zero (T covered them in the previous element)
      constexpr int PADV = (D::MP - ND) * D::KS / 8;   // 16-byte vectors per part
      for (int i = t; i < 3 * PADV; i += BS) {
        const int s = i / PADV, o = i % PADV;
        reinterpret_cast<uint4 *>(sm.w.ops + (s * D::MP + ND) * D::KS)[o] = make_uint4(0, 0, 0, 0);
      }
    }
    if constexpr (MODE == MODE_F64) {
      constexpr int PADD = (D::MP - ND) * D::KS64;   // doubles per operand
      for (int i = t; i < 2 * PADD; i += BS) sm.w.opd[((i / PADD) * D::MP + ND) * D::KS64 + i % PADD] = 0.0;
    }
    if constexpr (MODE == MODE_F32) {
      constexpr int PADF = (D::MP - ND) * D::KS32;   // floats per operand
      for (int i = t; i < 2 * PADF; i += BS) sm.w.opf[((i / PADF) * D::MP + ND) * D::KS32 + i % PADF] = 0.0f;
    }
    __syncthreads();
    // measure w |det J| with the sign of the first point (Intrepid2 computeCellMeasure)
    const double sg = sm.det[0] < 0.0 ? -1.0 : 1.0;
    if (t < NQ) sm.sw[t] = sqrt(sg * sm.wm[t]);
    if (has_src)
      for (int i = t; i < Q1 * NB; i += BS) {
        const int a = i % NB, qz = i / NB;
        const double *bx = sm.bL[sm.off[a][0]], *by = sm.bL[sm.off[a][1]];
        double F = 0.0;
#pragma unroll
        for (int qy = 0; qy < Q1; ++qy) {
          double l = 0.0;
#pragma unroll
          for (int qx = 0; qx < Q1; ++qx) l += sm.wm[(qz * Q1 + qy) * Q1 + qx] * bx[qx];
          F += l * by[qy];
        }
        sm.fa[qz][a] = F * sm.bL[sm.off[a][2]][qz];
      }
    // mass matrix (inertia and Rayleigh terms only)
    if (tr)
      for (int i = t; i < NB * NB; i += BS) {
        const int a = i / NB, b = i % NB;
        double s = 0.0;
        for (int q = 0; q < NQ; ++q) {
          const int qx = q % Q1, qy = (q / Q1) % Q1, qz = q / (Q1 * Q1);
          s += sm.wm[q] * (sm.bL[sm.off[a][0]][qx] * sm.bL[sm.off[a][1]][qy] * sm.bL[sm.off[a][2]][qz]) *
               (sm.bL[sm.off[b][0]][qx] * sm.bL[sm.off[b][1]][qy] * sm.bL[sm.off[b][2]][qz]);
        }
        sm.M[a][b] = static_cast<TReal>(sg * s);
      }
    __syncthreads();
    // ---- physical gradients at the quadrature points (MFMA mode: also the zero columns q >= NQ);
    // q runs fastest over the threads, so the operand writes of a wave are consecutive in LDS
    constexpr int QG = MODE == MODE_SPLIT ? D::KP : D::KP64;
    // when BS is a multiple of QG every thread keeps one q: its J^-1 and sqrt(w |det J|)
    // are read from LDS once
    constexpr bool QFIX = BS % QG == 0;
    double Jq[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, sqq = 1.0;
    if constexpr (QFIX) {
      const int q = t % QG;
      if (q < NQ) {
#pragma unroll
        for (int r = 0; r < 9; ++r) Jq[r] = sm.Ji[q][r];
        if constexpr (MODE == MODE_SPLIT) sqq = sm.sw[q];
      }
    }
    for (int i = t; i < QG * NB; i += BS) {
      const int q = i % QG, a = i / QG;
      if (MODE == MODE_SPLIT && q >= NQ) {
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
          for (int s = 0; s < 3; ++s) sm.w.ops[(s * D::MP + k * NB + a) * D::KS + q] = 0;
        continue;
      }
      if (MODE == MODE_F64 && q >= NQ) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          sm.w.opd[(0 * D::MP + k * NB + a) * D::KS64 + q] = 0.0;
          sm.w.opd[(1 * D::MP + k * NB + a) * D::KS64 + q] = 0.0;
        }
        continue;
      }
      if (MODE == MODE_F32 && q >= NQ) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          sm.w.opf[(0 * D::MP + k * NB + a) * D::KS32 + q] = 0.0f;
          sm.w.opf[(1 * D::MP + k * NB + a) * D::KS32 + q] = 0.0f;
        }
        continue;
      }
      const int qx = q % Q1, qy = (q / Q1) % Q1, qz = q / (Q1 * Q1);
      const int ax = sm.off[a][0], ay = sm.off[a][1], az = sm.off[a][2];
      const double lx = sm.bL[ax][qx], ly = sm.bL[ay][qy], lz = sm.bL[az][qz];
      const double dn[3] = {sm.bdL[ax][qx] * ly * lz, lx * sm.bdL[ay][qy] * lz, lx * ly * sm.bdL[az][qz]};
      const double *Ji = sm.Ji[q];
      auto ji = [&](int r) { return QFIX ? Jq[r] : Ji[r]; };
      const double sq = QFIX ? sqq : (MODE == MODE_SPLIT ? sm.sw[q] : 1.0);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const double g = ji(0 * 3 + k) * dn[0] + ji(1 * 3 + k) * dn[1] + ji(2 * 3 + k) * dn[2];
        if constexpr (MODE == MODE_SPLIT) {
          // operand [m = (k,a)][q] = sqrt(w |det J|) g in three bf16 parts: T = O^T O
          short s0, s1, s2;
          split3(static_cast<float>(sq * g), s0, s1, s2);
          const int m = k * NB + a;
          sm.w.ops[(0 * D::MP + m) * D::KS + q] = s0;
          sm.w.ops[(1 * D::MP + m) * D::KS + q] = s1;
          sm.w.ops[(2 * D::MP + m) * D::KS + q] = s2;
        } else if constexpr (MODE == MODE_F64) {
          // T[(k,a),(l,b)] = sum_q (sgn w det g_ka) g_lb
          const int m = k * NB + a;
          sm.w.opd[(0 * D::MP + m) * D::KS64 + q] = sg * sm.wm[q] * g;
          sm.w.opd[(1 * D::MP + m) * D::KS64 + q] = g;
        } else {
          // T[(k,a),(l,b)] = sum_q (sgn w det g_ka) g_lb, operands rounded to FP32 once
          const int m = k * NB + a;
          sm.w.opf[(0 * D::MP + m) * D::KS32 + q] = static_cast<float>(sg * sm.wm[q] * g);
          sm.w.opf[(1 * D::MP + m) * D::KS32 + q] = static_cast<float>(g);
        }
      }
    }
    __syncthreads();
    fetch_data(e + gridDim.x);
    fetch_index(e + 2 * static_cast<int64_t>(gridDim.x));
    // ---- gradient Gram matrix T
    if constexpr (MODE == MODE_SPLIT) {
      constexpr int NT = D::MP / 16;                 // 16x16 tiles per side
      constexpr int NTILE = NT * (NT + 1) / 2;       // upper triangle
      constexpr int TPW = (NTILE + BS / 64 - 1) / (BS / 64);
      const short *O = sm.w.ops;
      v4f acc[TPW];
#pragma unroll
      for (int k = 0; k < TPW; ++k) {
        acc[k] = v4f{0.f, 0.f, 0.f, 0.f};
        const int ti = wave + k * (BS / 64);
        if (ti >= NTILE) continue;
        int tm = 0, rem = ti;
        while (rem >= NT - tm) { rem -= NT - tm; ++tm; }
        const int tn = tm + rem;
        // gfx950's K = 32 bf16 product: lane l brings eight points of row l % 16, the eighth
        // 8 (l / 16) .. 8 (l / 16) + 7, of A and of B alike (whatever order the instruction gives
        // the eight, the sum over all 32 points is the same)
#pragma unroll
        for (int ks = 0; ks < D::KP / 32; ++ks) {
          const int k0 = ks * 32 + 8 * (lane >> 4);
          const int ma = tm * 16 + (lane & 15), nb = tn * 16 + (lane & 15);
          v8bf a_[3], b_[3];
#pragma unroll
          for (int s = 0; s < 3; ++s) {
            a_[s] = __builtin_bit_cast(v8bf, *reinterpret_cast<const v8s *>(O + (s * D::MP + ma) * D::KS + k0));
            b_[s] = __builtin_bit_cast(v8bf, *reinterpret_cast<const v8s *>(O + (s * D::MP + nb) * D::KS + k0));
          }
          // products of order 2^-16, 2^-8 and 1 (smallest first)
          acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_[2], b_[0], acc[k], 0, 0, 0);
          acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_[1], b_[1], acc[k], 0, 0, 0);
          acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_[0], b_[2], acc[k], 0, 0, 0);
          acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_[1], b_[0], acc[k], 0, 0, 0);
          acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_[0], b_[1], acc[k], 0, 0, 0);
          acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_[0], b_[0], acc[k], 0, 0, 0);
        }
      }
      __syncthreads();   // every wave has read the operands: T goes over them
#pragma unroll
      for (int k = 0; k < TPW; ++k) {
        const int ti = wave + k * (BS / 64);
        if (ti >= NTILE) continue;
        int tm = 0, rem = ti;
        while (rem >= NT - tm) { rem -= NT - tm; ++tm; }
        const int tn = tm + rem;
        // D[4 (lane/16) + i][lane % 16] of the tile; off-diagonal tiles also fill the
        // mirrored tile (the summation order of the split products differs between
        // (m, n) and (n, m), so a diagonal tile keeps its own entries on both sides)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int rr = tm * 16 + 4 * (lane >> 4) + i, cc = tn * 16 + (lane & 15);
          if (rr < ND && cc < ND) {
            sm.w.T32[rr][cc] = acc[k][i];
            if (tm != tn) sm.w.T32[cc][rr] = acc[k][i];
          }
        }
      }
    } else if constexpr (MODE == MODE_F64) {
      // T = A^T B on v_mfma_f64_16x16x4f64 over the upper-triangle 16x16 tiles: lane l holds
      // A and B element [row l % 16][point 4 ks + l / 16]; the tile's D[l/16 + 4 i][l % 16]
      // lands in component i (rows interleaved, unlike the FP32-accumulating 16x16 forms)
      constexpr int NT = D::MP / 16;
      constexpr int NTILE = NT * (NT + 1) / 2;
      constexpr int TPW = (NTILE + BS / 64 - 1) / (BS / 64);
      const double *A = sm.w.opd, *B = sm.w.opd + D::MP * D::KS64;
      v4d acc[TPW];
#pragma unroll
      for (int k = 0; k < TPW; ++k) {
        acc[k] = v4d{0.0, 0.0, 0.0, 0.0};
        const int ti = wave + k * (BS / 64);
        if (ti >= NTILE) continue;
        int tm = 0, rem = ti;
        while (rem >= NT - tm) { rem -= NT - tm; ++tm; }
        const int tn = tm + rem;
        const double *ar = A + (tm * 16 + (lane & 15)) * D::KS64 + (lane >> 4);
        const double *br = B + (tn * 16 + (lane & 15)) * D::KS64 + (lane >> 4);
#pragma unroll
        for (int ks = 0; ks < D::KP64 / 4; ++ks)
          acc[k] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[4 * ks], br[4 * ks], acc[k], 0, 0, 0);
      }
      __syncthreads();   // every wave has read the operands: T goes over them
#pragma unroll
      for (int k = 0; k < TPW; ++k) {
        const int ti = wave + k * (BS / 64);
        if (ti >= NTILE) continue;
        int tm = 0, rem = ti;
        while (rem >= NT - tm) { rem -= NT - tm; ++tm; }
        const int tn = tm + rem;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int rr = tm * 16 + (lane >> 4) + 4 * i, cc = tn * 16 + (lane & 15);
          if (rr < ND && cc < ND) {
            sm.w.v.T[rr][cc] = acc[k][i];
            if (tm != tn) sm.w.v.T[cc][rr] = acc[k][i];
          }
        }
      }
    } else {
      // T = A^T B on v_mfma_f32_16x16x4f32 over the upper-triangle 16x16 tiles: lane l holds A
      // and B element [row l % 16][point 4 ks + l / 16]; D[4 (l / 16) + i][l % 16] in component i
      constexpr int NT = D::MP / 16;
      constexpr int NTILE = NT * (NT + 1) / 2;
      constexpr int TPW = (NTILE + BS / 64 - 1) / (BS / 64);
      const float *A = sm.w.opf, *B = sm.w.opf + D::MP * D::KS32;
      v4f acc[TPW];
#pragma unroll
      for (int k = 0; k < TPW; ++k) {
        acc[k] = v4f{0.f, 0.f, 0.f, 0.f};
        const int ti = wave + k * (BS / 64);
        if (ti >= NTILE) continue;
        int tm = 0, rem = ti;
        while (rem >= NT - tm) { rem -= NT - tm; ++tm; }
        const int tn = tm + rem;
        const float *ar = A + (tm * 16 + (lane & 15)) * D::KS32 + (lane >> 4);
        const float *br = B + (tn * 16 + (lane & 15)) * D::KS32 + (lane >> 4);
#pragma unroll
        for (int ks = 0; ks < D::KP64 / 4; ++ks)
          acc[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(ar[4 * ks], br[4 * ks], acc[k], 0, 0, 0);
      }
      __syncthreads();   // every wave has read the operands: T goes over them
#pragma unroll
      for (int k = 0; k < TPW; ++k) {
        const int ti = wave + k * (BS / 64);
        if (ti >= NTILE) continue;
        int tm = 0, rem = ti;
        while (rem >= NT - tm) { rem -= NT - tm; ++tm; }
        const int tn = tm + rem;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int rr = tm * 16 + 4 * (lane >> 4) + i, cc = tn * 16 + (lane & 15);
          if (rr < ND && cc < ND) {
            sm.w.v.T[rr][cc] = acc[k][i];
            if (tm != tn) sm.w.v.T[cc][rr] = acc[k][i];
          }
        }
      }
    }
    __syncthreads();
    // ---- 3x3 blocks of node pairs: residual rows, Jacobian values to the workspace, node-major (node
    // a: rows i NB + a, i = 0..2, of the Gram layout; the padding is not written): the lanes of a node
    // on consecutive entries
    //   K_ij = lambda T[(i,a),(j,b)] + mu T[(j,a),(i,b)] + delta_ij mu sum_k T[(k,a),(k,b)]
    const double lam = E * p.nu / ((1.0 + p.nu) * (1.0 - 2.0 * p.nu));
    const double mu = E / (2.0 * (1.0 + p.nu));
    // the next element's data is here before the block stores go out (one counter tracks both)
    asm volatile("" : "+v"(gX), "+v"(gu), "+v"(gv), "+v"(gac), "+v"(gE), "+v"(gn), "+v"(gL));
    constexpr int NP = block_stride(NB);
    double rp[NPASS][3];
    auto Tref = [&](int r, int c) -> TReal {
      if constexpr (MODE == MODE_SPLIT) return sm.w.T32[r][c];
      else return sm.w.v.T[r][c];
    };
    const double cK = tr ? p.beta + p.alpha * p.rb : p.beta;
    const double cM = tr ? p.alpha * p.ra + (tra ? p.gamma2 : 0.0) : 0.0;
#pragma unroll
    for (int k = 0; k < NPASS; ++k) {
      const int a = ga + k * AP, b = gb;
      double rr[3] = {0.0, 0.0, 0.0};
      if (a < NB && b < NB) {
        double t9[3][3];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int j = 0; j < 3; ++j) t9[i][j] = static_cast<double>(Tref(i * NB + a, j * NB + b));
        const double trs = t9[0][0] + t9[1][1] + t9[2][2];
        const double Mab = tr ? p.rho * static_cast<double>(sm.M[a][b]) : 0.0;
        // with C = a_R M + b_R K:  J = (beta + alpha b_R) K + (alpha a_R + gamma2) M  and
        // R = K (u + b_R v) + M (a_R v + a), node b's state combined once for its nine entries
        double ut[3], mt[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          ut[j] = tr ? sm.u[3 * b + j] + p.rb * sm.v[3 * b + j] : sm.u[3 * b + j];
          mt[j] = tr ? p.ra * sm.v[3 * b + j] + (tra ? sm.a[3 * b + j] : 0.0) : 0.0;
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            const double Kv = lam * t9[i][j] + mu * t9[j][i] + (i == j ? mu * trs : 0.0);
            rr[i] += Kv * ut[j];
            double jv = cK * Kv;
            if (i == j) {
              jv += cM * Mab;
              rr[i] += Mab * mt[j];
            }
            if (p.jbuf) {
              TReal *o = &static_cast<TReal *>(p.jbuf)[(e * NB + a) * NP + i * ND + j * NB + b];
              // hex27 blocks stream past the caches (measured faster); hex8 blocks as plain stores
              if (NB == 27) __builtin_nontemporal_store(static_cast<TReal>(jv), o);
              else *o = static_cast<TReal>(jv);
            }
          }
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) rp[k][i] = rr[i];
    }
    // row residuals: fixed-order reduction over each group's b (lanes b >= NB add 0)
    static_assert(GW == 8 || GW == 32, "group width");
    if constexpr (GW == 32) {
      // the lanes' twelve values (pass, i) together, halved as the lanes they are summed over are: value
      // 4 m + 2 h + r ends in the lanes of row parity r, half row h
      static_assert(NPASS == 4, "twelve values");
      const double *v = &rp[0][0];
      double u6[6], u3[3];
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(v[2 * j]), __double2loint(v[2 * j + 1]), false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(v[2 * j]), __double2hiint(v[2 * j + 1]), false, false);
        u6[j] = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
      }
      const bool h8 = lane & 8;
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        const double keep = h8 ? u6[2 * m + 1] : u6[2 * m], send = h8 ? u6[2 * m] : u6[2 * m + 1];
        u3[m] = group_sum<8>(keep + dpp_f64<0x128, 0xf>(send));   // row_ror:8
        const int val = 4 * m + 2 * (h8 ? 1 : 0) + ((lane >> 4) & 1), a = ga + val / 3 * AP;
        if ((lane & 7) == 0 && a < NB) sm.r[3 * a + val % 3] = u3[m];
      }
    } else {
#pragma unroll
      for (int k = 0; k < NPASS; ++k)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const double r = group_sum<GW>(rp[k][i]);
          if (ga + k * AP < NB && gb == 0) sm.r[3 * (ga + k * AP) + i] = r;
        }
    }
    __syncthreads();
    put_data();   // the next element's vertices and state (LDS X, u, v, a are free now)
    if (p.rbuf)
      for (int i = t; i < ND; i += BS) {
        double F = 0.0;
        if (has_src) {
          const int a = i / 3;
#pragma unroll
          for (int k = 0; k < Q1; ++k) F += sm.fa[k][a];
          // a select, not an indexed read: src[i % 3] would be a vector load from the
          // parameters, and waiting for it would wait for the block stores
          const int c = i % 3;
          F *= sg * (c == 0 ? p.src[0] : (c == 1 ? p.src[1] : p.src[2]));
        }
        p.rbuf[e * ND + i] = sm.r[i] - F;
      }
    E = gE;
  }
}

// Second phase: node-centric gather.  One wave per lattice node assembles the
// node's three CRS rows (consecutive LIDs with one column structure) in LDS in
// FP64 from the blocks of the elements around it, in a fixed element order, then
// writes them once, coalesced, with the residual.
struct GatherParams {
  int nx, ny, nz;
  int64_t px, py, pz, npoints;
  int64_t p0, p1;             // lattice points [p0, p1) of this launch
  const int32_t *point_lid;   // [points][3]
  const int64_t *rowptr;
  const uint16_t *nperm;
  int nperm_w;
  const void *jbuf;
  const double *rbuf;
  double *f, *vals;
};

// One wave stores n consecutive FP64 values from LDS to dst, non-temporally (written once,
// not re-read here), in chunks aligned to 128-byte lines: only the first and the last line
// of the range are partial.
__device__ __forceinline__ void row_store(const double *src, double *dst, int n, int lane) {
  const int lead = static_cast<int>((reinterpret_cast<uintptr_t>(dst) >> 3) & 15);
  for (int k = lane - lead; k < n; k += 64)
    if (k >= 0) __builtin_nontemporal_store(src[k], dst + k);
}

__device__ __forceinline__ void gather_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int NB, typename JT>
__global__ __launch_bounds__(256) void k_elastic_gather(GatherParams g) {
  constexpr int ND = 3 * NB;
  constexpr int R = NB == 8 ? 1 : 2, S = 2 * R + 1;
  constexpr int STEP = NB == 8 ? 1 : 2;        // lattice points per cell edge
  constexpr int MAXLEN = 3 * S * S * S;        // entries per row
  __shared__ double buf[4][3 * MAXLEN];
  __shared__ int8_t inv[3][3][3];
  // the wave index is uniform: everything derived from the node stays in scalar registers
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int NR = (3 * ND + 63) / 64;   // block entries per lane and element
  constexpr int NP = block_stride(NB);
  // per lane and r: entry idx = lane + 64 r of the node's three block rows (row field
  // idx / ND, Gram column idx % ND = field j, node bn), and the lattice offset index of
  // its column node plus R in each axis; the entry sits at idx in the node's part of the block
  int lterm[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int idx = lane + 64 * r, c = idx % ND;
    const int bn = c % NB;
    const int8_t *o = NB == 8 ? kHexV[bn] : kQ2[bn];
    lterm[r] = (o[0] + R) + S * (o[1] + R) + S * S * (o[2] + R);
  }
  for (int i = threadIdx.x; i < NB; i += 256) {
    const int8_t *o = NB == 8 ? kHexV[i] : kQ2[i];
    inv[o[0]][o[1]][o[2]] = static_cast<int8_t>(i);
  }
  __syncthreads();
  double *b = buf[w];
  const JT *J = static_cast<const JT *>(g.jbuf);
  // The node's LID and row pointers are wave-uniform: they are read through the scalar
  // cache (constant address space; neither array changes during the kernel), whose
  // counter is not the one the row stores use, and one node ahead.  Read as vector loads,
  // each node began by waiting for them and with them for every store of the node before.
  using cint = const __attribute__((address_space(4))) int32_t;
  using clong = const __attribute__((address_space(4))) int64_t;
  const cint *plid = (const cint *)g.point_lid;
  const clong *prow = (const clong *)g.rowptr;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 4;
  int64_t pt = g.p0 + static_cast<int64_t>(blockIdx.x) * 4 + w;
  int32_t Lc = plid[min(pt, g.p1 - 1) * 3];
  int64_t bc = prow[Lc], ec = prow[Lc + 1];
  // lattice coordinates of the node, advanced by the stride's own coordinates with
  // carries: the divisions happen once, not per node
  const int64_t pxy = g.px * g.py;
  int64_t I = pt % g.px, Jy = (pt / g.px) % g.py, K = pt / pxy;
  const int64_t sI = stride % g.px, sJ = (stride / g.px) % g.py, sK = stride / pxy;
  for (; pt < g.p1; pt += stride) {
    const int32_t L0 = Lc;
    const int64_t base = bc;
    // row length (at most S^3 neighbours x 3 fields; clamped so the LDS rows never overflow)
    const int len = min(static_cast<int>(ec - bc), MAXLEN);
    const int32_t Ln = plid[min(pt + stride, g.p1 - 1) * 3];   // the next node's LID
    const int64_t node = L0 / 3;
    const uint16_t *np = g.nperm + node * g.nperm_w;
    for (int k = lane; k < 3 * len; k += 64) b[k] = 0.0;
    gather_lds_sync();
    // cells containing the node (at most 8), per axis [c_lo, c_hi]
    const int64_t cx_lo = I % STEP == 0 ? I / STEP - 1 : I / STEP, cx_hi = I / STEP;
    const int64_t cy_lo = Jy % STEP == 0 ? Jy / STEP - 1 : Jy / STEP, cy_hi = Jy / STEP;
    const int64_t cz_lo = K % STEP == 0 ? K / STEP - 1 : K / STEP, cz_hi = K / STEP;
    int64_t ce[8];
    int ca[8], cs[8];
    int ne = 0;
    for (int64_t cz = cz_lo; cz <= cz_hi; ++cz)
      for (int64_t cy = cy_lo; cy <= cy_hi; ++cy)
        for (int64_t cx = cx_lo; cx <= cx_hi; ++cx)
          if (cx >= 0 && cx < g.nx && cy >= 0 && cy < g.ny && cz >= 0 && cz < g.nz) {
            const int ox = static_cast<int>(I - STEP * cx), oy = static_cast<int>(Jy - STEP * cy),
                      oz = static_cast<int>(K - STEP * cz);   // lattice offset of the node in the cell
            ce[ne] = cx + g.nx * (cy + g.ny * cz);
            ca[ne] = inv[ox][oy][oz];
            cs[ne] = ox + S * oy + S * S * oz;
            ++ne;
          }
    // every load first (one round trip per node), then the additions in element order
    JT val[8][NR];
    uint16_t pos[8][NR];
    double rr[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      rr[c] = 0.0;
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        val[c][r] = JT(0);
        pos[c][r] = 0xffffu;
        const int idx = lane + 64 * r;
        if (c < ne && idx < 3 * ND && J) {
          val[c][r] = J[(ce[c] * NB + ca[c]) * NP + idx];   // node ca's rows: one contiguous run
          pos[c][r] = np[lterm[r] - cs[c]];
        }
      }
      if (c < ne && lane < 3 && g.rbuf) rr[c] = g.rbuf[ce[c] * ND + 3 * ca[c] + lane];
    }
    const int64_t bn = prow[Ln], en = prow[Ln + 1];   // the next node's row pointers
    // the values stay opaque until here, so no conversion pulls a wait in among the loads
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int r = 0; r < NR; ++r) asm volatile("" : "+v"(val[c][r]));
    // LDS atomic adds, issued back to back: the LDS executes one wave's operations in
    // order and no two lanes of one instruction share an entry, so every entry is summed
    // in cell order, as one read-add-write round per cell did, without a round trip per cell
    double racc = 0.0;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      if (c < ne) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          const int idx = lane + 64 * r;
          const int i = idx / ND, j = (idx % ND) / NB;
          const uint16_t ps = pos[c][r];
          if (idx < 3 * ND && ps != 0xffffu && ps + j < len) atomicAdd(&b[i * len + ps + j], static_cast<double>(val[c][r]));
        }
        racc += rr[c];
      }
    }
    gather_lds_sync();   // all additions done before the rows are read
    if (g.vals)
      row_store(b, g.vals + base, 3 * len, lane);
    if (g.f && lane < 3) g.f[L0 + lane] = racc;
    gather_lds_sync();   // the buffer is reused by the next node
    Lc = Ln;
    bc = bn;
    ec = en;
    I += sI;
    Jy += sJ;
    K += sK;
    if (I >= g.px) { I -= g.px; ++Jy; }
    if (Jy >= g.py) { Jy -= g.py; ++K; }
  }
}

// The same gather on an uploaded hex8 / hex27 mesh of one block: node n (rows 3n, 3n + 1, 3n + 2:
// the first-touch numbering gives a node's three fields consecutive LIDs) takes its element
// instances (e, a) from the node's list, ascending, eight at a time, and the row position of
// each element node's field 0 from the instance's slot map.
struct GatherUParams {
  int64_t nnodes;
  const int64_t *occ_ptr;   // [nnodes + 1]
  const int32_t *occ;       // e * NB + a per instance
  const uint16_t *slot;     // [instances][NB] position of (element node b, field 0) in row 3n
  const int64_t *rowptr;
  const void *jbuf;
  const double *rbuf;
  double *f, *vals;
};

template <int NB, typename JT>
__global__ __launch_bounds__(256) void k_elastic_gather_u(GatherUParams g) {
  constexpr int ND = 3 * NB;
  constexpr int R = NB == 8 ? 1 : 2, S = 2 * R + 1;
  constexpr int MAXLEN = 3 * S * S * S;        // entries per row (checked when the lists are built)
  __shared__ double buf[4][3 * MAXLEN];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int NR = (3 * ND + 63) / 64;
  constexpr int NP = block_stride(NB);
  double *b = buf[w];
  const JT *J = static_cast<const JT *>(g.jbuf);
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 4;
  for (int64_t n = static_cast<int64_t>(blockIdx.x) * 4 + w; n < g.nnodes; n += stride) {
    const int32_t L0 = static_cast<int32_t>(3 * n);
    const int64_t base = g.rowptr[L0];
    const int len = min(static_cast<int>(g.rowptr[L0 + 1] - base), MAXLEN);
    for (int k = lane; k < 3 * len; k += 64) b[k] = 0.0;
    gather_lds_sync();
    const int64_t o0 = g.occ_ptr[n], o1 = g.occ_ptr[n + 1];
    double racc = 0.0;
    for (int64_t k0 = o0; k0 < o1; k0 += 8) {
      const int ne = static_cast<int>(o1 - k0 < 8 ? o1 - k0 : 8);
      JT val[8][NR];
      uint16_t pos[8][NR];
      double rr[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        rr[c] = 0.0;
        const int32_t v = c < ne ? g.occ[k0 + c] : 0;
        const int64_t e = v / NB;
        const int a = v - static_cast<int>(e) * NB;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          val[c][r] = JT(0);
          pos[c][r] = 0xffffu;
          const int idx = lane + 64 * r;
          if (c < ne && idx < 3 * ND && J) {
            val[c][r] = J[(e * NB + a) * NP + idx];
            pos[c][r] = g.slot[(k0 + c) * NB + (idx % ND) % NB];
          }
        }
        if (c < ne && lane < 3 && g.rbuf) rr[c] = g.rbuf[e * ND + 3 * a + lane];
      }
#pragma unroll
      for (int c = 0; c < 8; ++c)
#pragma unroll
        for (int r = 0; r < NR; ++r) asm volatile("" : "+v"(val[c][r]));
      // one wave's LDS operations execute in order and no two lanes of one instruction share
      // an entry: every entry is summed in instance order
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        if (c < ne) {
#pragma unroll
          for (int r = 0; r < NR; ++r) {
            const int idx = lane + 64 * r;
            const int i = idx / ND, j = (idx % ND) / NB;
            const uint16_t ps = pos[c][r];
            if (idx < 3 * ND && ps != 0xffffu && ps + j < len)
              atomicAdd(&b[i * len + ps + j], static_cast<double>(val[c][r]));
          }
          racc += rr[c];
        }
      }
    }
    gather_lds_sync();
    if (g.vals)
      row_store(b, g.vals + base, 3 * len, lane);
    if (g.f && lane < 3) g.f[L0 + lane] = racc;
    gather_lds_sync();
  }
}

// Element instances of each node of an uploaded 3-field mesh (field-0 positions of elem_lid)
__global__ void k_uocc_count(int64_t npos0, int nb, const int32_t *__restrict__ elem_lid,
                             unsigned long long *__restrict__ cnt) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= npos0) return;   // t = e * nb + a
  atomicAdd(cnt + elem_lid[3 * t] / 3, 1ull);
}

__global__ void k_uocc_fill(int64_t npos0, int nb, const int32_t *__restrict__ elem_lid,
                            unsigned long long *__restrict__ cursor, int32_t *__restrict__ occ) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= npos0) return;
  occ[atomicAdd(cursor + elem_lid[3 * t] / 3, 1ull)] = static_cast<int32_t>(t);
}

// Sorts each node's list (ascending e * nb + a: a fixed summation order), the slot map of each
// instance, and the longest row and list (out[0], out[1]).
__global__ void k_uocc_finish(int64_t nnodes, int nb, const int64_t *__restrict__ optr, int32_t *__restrict__ occ,
                              const int32_t *__restrict__ elem_lid, const int64_t *__restrict__ rowptr,
                              const int32_t *__restrict__ col, uint16_t *__restrict__ slot, int *__restrict__ out) {
  const int64_t n = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (n >= nnodes) return;
  const int64_t lo = optr[n], hi = optr[n + 1];
  for (int64_t i = lo + 1; i < hi; ++i) {
    const int32_t v = occ[i];
    int64_t j = i;
    for (; j > lo && occ[j - 1] > v; --j) occ[j] = occ[j - 1];
    occ[j] = v;
  }
  const int64_t r0 = rowptr[3 * n], len = rowptr[3 * n + 1] - r0;
  atomicMax(out, static_cast<int>(len));
  atomicMax(out + 1, static_cast<int>(hi - lo));
  for (int64_t i = lo; i < hi; ++i) {
    const int64_t e = occ[i] / nb;
    for (int b = 0; b < nb; ++b) {
      const int32_t key = elem_lid[(e * nb + b) * 3];
      int64_t l = 0, h = len;
      while (l < h) {
        const int64_t m = (l + h) >> 1;
        if (col[r0 + m] < key) l = m + 1; else h = m;
      }
      slot[i * nb + b] = l < len && col[r0 + l] == key && l < 0xffff ? static_cast<uint16_t>(l) : uint16_t(0xffff);
    }
  }
}

// Row position of (neighbour, field 0) for every node and lattice offset in
// [-R, R]^3 (0xffff: not a neighbour), by binary search in the node's first row.
__global__ void k_node_perm(int64_t px, int64_t py, int64_t pz, int R, int nf, int W,
                            const int32_t *__restrict__ point_lid, const int64_t *__restrict__ rowptr,
                            const int32_t *__restrict__ col, uint16_t *__restrict__ nperm) {
  const int64_t pt = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (pt >= px * py * pz) return;
  const int64_t i = pt % px, j = (pt / px) % py, k = pt / (px * py);
  const int32_t row = point_lid[pt * nf];
  const int64_t lo0 = rowptr[row], hi0 = rowptr[row + 1];
  uint16_t *out = nperm + static_cast<int64_t>(row / nf) * W;
  const int S = 2 * R + 1;
  for (int s = 0; s < W; ++s) {
    uint16_t v = 0xffffu;
    if (s < S * S * S) {
      const int64_t ii = i + s % S - R, jj = j + (s / S) % S - R, kk = k + s / (S * S) - R;
      if (ii >= 0 && ii < px && jj >= 0 && jj < py && kk >= 0 && kk < pz) {
        const int32_t key = point_lid[(ii + px * (jj + py * kk)) * nf];
        int64_t lo = lo0, hi = hi0;
        while (lo < hi) {
          const int64_t m = (lo + hi) >> 1;
          if (col[m] < key) lo = m + 1; else hi = m;
        }
        if (lo < hi0 && col[lo] == key) v = static_cast<uint16_t>(lo - lo0);
      }
    }
    out[s] = v;
  }
}

// Affine HEX8 bricks (every cell a parallelepiped), three fields: node-centric assembly with
// no workspace.  The 3x3 block of a node's vertex a and another vertex b of a cell has a closed
// form: with J = dx/dxi constant over the cell and C its cofactor matrix,
//   T_ab = |det J| J^-T S_ab J^-1 = C S_ab C^T / |det J|,
//   S_ab[m][n] = sum_q dN_a/dxi_m dN_b/dxi_n   (2x2x2 Gauss)
//              = s_a^m s_b^n f_d / 4 (m != n, d the third axis),  s_a^m s_b^m f_d1 f_d2 / 2 (m = n),
// with s the vertex's sign along an axis and f = 2/3 where a and b share it, 1/3 otherwise;
// the mass entry rho |det J| f_x f_y f_z, the source load src |det J| per vertex.  Blocks of
// cells that share a vertex are summed in a fixed order (bitwise reproducible), each node's three
// rows written once (k_elastic8_affine).
struct Elastic8Params {
  int nx, ny, nz;
  int64_t npoints;
  const int32_t *point_lid;   // [points][3]
  const int64_t *rowptr;
  const uint16_t *nperm;
  int nperm_w;
  const double *geom;         // [cells][10]: cofactors of J scaled by |det J|^-1/2, then |det J|
  const double *coef;         // Young's modulus per cell
  double nu, rho, src[3], ra, rb;
  const double *x, *xdot, *xddot;
  double alpha, beta, gamma2;
  int transient;
  double *f, *vals;
};

// Geometry of each parallelepiped cell, once per mesh: its constant Jacobian
// J[d][j] = (1/8) sum_b s_b^j X_b^d (s_b^j = -1 / +1 for vertex b's j-th bit 0 / 1), the
// cofactor matrix C (adj J = C^T) and |det J|, stored as C |det J|^-1/2 and |det J|, so that
// C S C^T / |det J| = Chat S Chat^T in the node kernel.  One thread per cell.
__global__ void k_cell_geom(int nx, int ny, int nz, int64_t nv, const double *__restrict__ xyz,
                            double *__restrict__ geom) {
  const int64_t c = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (c >= static_cast<int64_t>(nx) * ny * nz) return;
  const int64_t i = c % nx, j = (c / nx) % ny, k = c / (static_cast<int64_t>(nx) * ny);
  double Jm[3][3] = {};
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const int bx = b & 1, by = (b >> 1) & 1, bz = b >> 2;
    const int64_t v = (i + bx) + (nx + 1) * ((j + by) + static_cast<int64_t>(ny + 1) * (k + bz));
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double X = xyz[d * nv + v];
      Jm[d][0] += bx ? X : -X;
      Jm[d][1] += by ? X : -X;
      Jm[d][2] += bz ? X : -X;
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int jj = 0; jj < 3; ++jj) Jm[d][jj] *= 0.125;
  double C[9];
  C[0] = Jm[1][1] * Jm[2][2] - Jm[1][2] * Jm[2][1];
  C[1] = Jm[1][2] * Jm[2][0] - Jm[1][0] * Jm[2][2];
  C[2] = Jm[1][0] * Jm[2][1] - Jm[1][1] * Jm[2][0];
  C[3] = Jm[0][2] * Jm[2][1] - Jm[0][1] * Jm[2][2];
  C[4] = Jm[0][0] * Jm[2][2] - Jm[0][2] * Jm[2][0];
  C[5] = Jm[0][1] * Jm[2][0] - Jm[0][0] * Jm[2][1];
  C[6] = Jm[0][1] * Jm[1][2] - Jm[0][2] * Jm[1][1];
  C[7] = Jm[0][2] * Jm[1][0] - Jm[0][0] * Jm[1][2];
  C[8] = Jm[0][0] * Jm[1][1] - Jm[0][1] * Jm[1][0];
  const double adet = fabs(Jm[0][0] * C[0] + Jm[0][1] * C[1] + Jm[0][2] * C[2]);
  const double sc = 1.0 / sqrt(adet);
  double *g = geom + 10 * c;
#pragma unroll
  for (int t = 0; t < 9; ++t) g[t] = C[t] * sc;
  g[9] = adet;
}

constexpr int kN8 = 4;                                      // nodes along x and y per workgroup
constexpr int kV8 = (kN8 + 2) * (kN8 + 2) * 3;              // vertices around them
constexpr int kC8 = (kN8 + 1) * (kN8 + 1) * 2;              // cells around them
constexpr int kRow8 = 3 * 81;                               // entries of a node's rows at most

// Lane of a node in the tile kernels: cell (ox, oy, oz) of the eight around it (I - 1 + ox, ...) and
// half h (the vertices on the cell's low / high z side), as lane ^ = ox ^ 2 oy ^ 8 oz ^ 15 h, so that
// the partner cell along x is lane ^ 1, along y lane ^ 2, and the (upper cell, low half) of lanes
// 8-11 meets the (lower cell, high half) of lanes 12-15 at lane ^ 7: one DPP move each.
struct NodeLane {
  int ox, oy, oz, h;
  __device__ __forceinline__ explicit NodeLane(int l16) {
    h = (l16 >> 2) & 1;
    const int lu = h ? l16 ^ 15 : l16;
    ox = lu & 1;
    oy = (lu >> 1) & 1;
    oz = lu >> 3;
  }
};

// Entry of block k (vertex on the cell's outer side along x / y, or with bit 0 / 1 of k the node's own
// side) summed over the cells that share its vertex: along x, then y, then z.
template <int K>
__device__ __forceinline__ double meet(double v, bool upper) {   // upper: lanes 8-15 of the node
  if (K & 1) v += dpp_f64<0xB1, 0xf>(v);
  if (K & 2) v += dpp_f64<0x4E, 0xf>(v);
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x141, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x141, 0xf, 0xf, true);
  return v + __hiloint2double(upper ? hi : 0, upper ? lo : 0);
}
// whether this lane writes block k's sum
__device__ __forceinline__ bool owns_block(const NodeLane &q, int k) {
  return (q.oz == q.h || q.h) && !((k & 1) && q.ox) && !((k & 2) && q.oy);
}

// One wave stores the rows of its line of four nodes (rows + n kRow8 in LDS, or one range where the
// nodes' LIDs follow each other: run).
__device__ __forceinline__ void store_line(const double *rows, double *vals, int64_t base, int len, bool run, int nok,
                                           int lane) {
  if (run) {
    const int64_t base0 = __shfl(base, 0);
    const int last = 16 * (nok - 1);
    row_store(rows, vals + base0, static_cast<int>(__shfl(base, last) - base0) + 3 * __shfl(len, last), lane);
  } else {
    for (int m = 0; m < nok; ++m)
      row_store(rows + m * kRow8, vals + __shfl(base, 16 * m), 3 * __shfl(len, 16 * m), lane);
  }
}

// One wave per line of four nodes along x, 16 lanes per node; each lane forms the blocks of its cell's
// four vertices on one z side one after another.  With the cell's cofactor columns signed by the node's
// corner (c_m s_a^m), T_ab = sum_mn c_m F_mn sigma_n c_n^T where sigma_n = +1 / -1 and f_n = 2/3 / 1/3 as a
// and b agree or not along n, F_mm = f_d1 f_d2 / 2, F_mn = f_d / 4 (d the third axis): x and y known per
// block, z per lane.  The state of the 6 x 3 x 3 vertices is staged in LDS, the next line's loaded before
// this line's row stores (one counter tracks a wave's loads and stores); the waves of a workgroup share
// nothing.
//
// Bound by VALU issue (296 instructions per node, 67% busy at three waves per SIMD) and the row
// stores.  Transient FP64, against one wave per node with 64 lanes of one block each, eight ordered
// LDS adds per entry and the state loaded once per lane (390 instructions per node): 128^3 2.56 ->
// 1.71 ms, 115^3 1.82 -> 1.22 ms, 64^3 319 -> 229 us; the same tiles staged per workgroup behind two
// barriers at two waves per SIMD 2.15 ms at 128^3.
template <bool TR>
__global__ __launch_bounds__(256, 3) void k_elastic8_affine(Elastic8Params p) {
  constexpr int NV = (kN8 + 2) * 9;
  __shared__ double state[4][TR ? 6 : 3][NV];           // u + b_R v, a_R v + a
  __shared__ double row[4][kN8 * kRow8];
  int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  auto &vtx = state[w];
  const int l16 = lane & 15, n = lane >> 4;
  NodeLane q(l16);
  const int sx = p.nx + 1, sxy = sx * (p.ny + 1);
  const int gx = (sx + kN8 - 1) / kN8, gy = p.ny + 1;
  const int ntile = gx * gy * (p.nz + 1);
  const bool tra = TR && p.xddot;
  const double ratio = 2.0 * p.nu / (1.0 - 2.0 * p.nu), muf = 0.5 / (1.0 + p.nu);
  const double cK = TR ? p.beta + p.alpha * p.rb : p.beta;
  const double cM = TR ? p.alpha * p.ra + (tra ? p.gamma2 : 0.0) : 0.0;
  double vu[3], vm[3], En;
  // LID of this lane's node; its cell (one outside the mesh: the nearest, which has this node and every
  // vertex that the two share, so a degenerate cell reaches the rows of its own vertices only)
  int32_t Ln, Cn;
  auto load_tile = [&](int tile) {
    const int I0 = tile % gx * kN8, J0 = tile / gx % gy, K = tile / (gx * gy);
    const int t = min(lane, NV - 1);
    const int ix = min(max(I0 - 1 + t % (kN8 + 2), 0), p.nx);
    const int iy = min(max(J0 - 1 + t / (kN8 + 2) % 3, 0), p.ny);
    const int iz = min(max(K - 1 + t / (3 * (kN8 + 2)), 0), p.nz);
    const int32_t L = p.point_lid[3 * (ix + sx * iy + sxy * iz)];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      vu[j] = p.x[L + j];
      if constexpr (TR) {
        const double v = p.xdot[L + j], a = tra ? p.xddot[L + j] : 0.0;
        vu[j] += p.rb * v;
        vm[j] = p.ra * v + a;
      }
    }
    Ln = p.point_lid[3 * (min(I0 + n, p.nx) + sx * J0 + sxy * K)];
    const int cx = min(max(I0 + n - 1 + q.ox, 0), p.nx - 1), cy = min(max(J0 - 1 + q.oy, 0), p.ny - 1),
              cz = min(max(K - 1 + q.oz, 0), p.nz - 1);
    Cn = cx + p.nx * (cy + p.ny * cz);
    En = p.coef[Cn];
  };
  const int stride = static_cast<int>(gridDim.x) * 4;
  int tile = static_cast<int>(blockIdx.x) * 4 + w;
  load_tile(min(tile, ntile - 1));
  for (; tile < ntile; tile += stride) {
    // indices and lane factors are formed per tile, not kept in registers
    asm volatile("" : "+v"(lane), "+v"(q.ox), "+v"(q.oy), "+v"(q.oz), "+v"(q.h));
    const bool zsame = q.h != q.oz;                       // b on the node's side along z
    const double fz = zsame ? 2.0 / 3.0 : 1.0 / 3.0;
    const int I0 = tile % gx * kN8, J0 = tile / gx % gy, K = tile / (gx * gy);
    if (lane < NV)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        vtx[j][lane] = vu[j];
        if constexpr (TR) vtx[3 + j][lane] = vm[j];
      }
    const int I = I0 + n, Jy = J0;
    const bool node_ok = I <= p.nx;
    const int32_t L0 = Ln;
    const int cx = I - 1 + q.ox, cy = Jy - 1 + q.oy, cz = K - 1 + q.oz;
    const bool cell_ok = node_ok && cx >= 0 && cx < p.nx && cy >= 0 && cy < p.ny && cz >= 0 && cz < p.nz;
    const double E = cell_ok ? En : 0.0;
    double2 G[5];
    const double2 *gp = reinterpret_cast<const double2 *>(p.geom + 10 * static_cast<int64_t>(Cn));
#pragma unroll
    for (int t = 0; t < 5; ++t) G[t] = gp[t];
    const int64_t base = p.rowptr[L0];
    const int len = min(static_cast<int>(p.rowptr[L0 + 1] - base), 81);
    const uint16_t *np = p.nperm + static_cast<int64_t>(L0 / 3) * p.nperm_w;
    int pos[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) pos[k] = np[((k & 1) ? 1 : 2 * q.ox) + 3 * ((k & 2) ? 1 : 2 * q.oy) + 9 * (q.oz + q.h)];
    gather_lds_sync();
    // cofactor columns (scaled by |det J|^-1/2), signed by the node's corner of the cell
    const double ax = q.ox ? -1.0 : 1.0, ay = q.oy ? -1.0 : 1.0, az = q.oz ? -1.0 : 1.0;
    const double c[3][3] = {{ax * G[0].x, ax * G[1].y, ax * G[3].x}, {ay * G[0].y, ay * G[2].x, ay * G[3].y},
                            {az * G[1].x, az * G[2].y, az * G[4].x}};   // c[m]: column m
    const double adet = cell_ok ? G[4].y : 0.0;
    // the second factor carries mu: T below is mu T_ab, and lambda = mu * 2 nu / (1 - 2 nu)
    const double mu = E * muf;
    double cm[3][3];
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
      for (int l = 0; l < 3; ++l) cm[m][l] = mu * (m == 2 && !zsame ? -c[m][l] : c[m][l]);
    const int64_t base0 = __shfl(base, 0);
    const bool run = __all(!node_ok || L0 == __shfl(L0, 0) + 3 * n);
    double *mine = row[w] + (run ? static_cast<int>(base - base0) : n * kRow8);
    double rr[3] = {0.0, 0.0, 0.0};
    auto block = [&](auto kc) {
      constexpr int k = decltype(kc)::value;
      constexpr double fx = (k & 1) ? 2.0 / 3.0 : 1.0 / 3.0, fy = (k & 2) ? 2.0 / 3.0 : 1.0 / 3.0;
      constexpr double gx_ = (k & 1) ? 1.0 : -1.0, gy_ = (k & 2) ? 1.0 : -1.0;   // sigma
      double P[3][3], T[3][3];
#pragma unroll
      for (int l = 0; l < 3; ++l) {
        P[0][l] = (0.5 * fy * gx_ * fz) * cm[0][l] + (0.25 * gy_ * fz) * cm[1][l] + (0.25 * fy) * cm[2][l];
        P[1][l] = (0.25 * gx_ * fz) * cm[0][l] + (0.5 * fx * gy_ * fz) * cm[1][l] + (0.25 * fx) * cm[2][l];
        P[2][l] = (0.25 * fy * gx_) * cm[0][l] + (0.25 * fx * gy_) * cm[1][l] + (0.5 * fx * fy) * cm[2][l];
      }
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int l = 0; l < 3; ++l) T[i][l] = c[0][i] * P[0][l] + c[1][i] * P[1][l] + c[2][i] * P[2][l];
      const int bx = q.ox ^ (k & 1), by = q.oy ^ (k >> 1);
      const int vi = (n + q.ox + bx) + (kN8 + 2) * ((q.oy + by) + 3 * (q.oz + q.h));
      const double trs = T[0][0] + T[1][1] + T[2][2];
      const double Mab = TR ? p.rho * adet * (fx * fy * fz) : 0.0;
      double ut[3], mt[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) { ut[j] = vtx[j][vi]; mt[j] = TR ? vtx[TR ? 3 + j : 0][vi] : 0.0; }
      const bool put = p.vals && node_ok && owns_block(q, k) && pos[k] + 2 < len;
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const double Kv = ratio * T[i][j] + T[j][i] + (i == j ? trs : 0.0);
          rr[i] += Kv * ut[j];
          double jv = cK * Kv;
          if (TR && i == j) {
            jv += cM * Mab;
            rr[i] += Mab * mt[j];
          }
          P[i][j] = meet<k>(jv, l16 > 7);
        }
      if (put)
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int j = 0; j < 3; ++j) mine[i * len + pos[k] + j] = P[i][j];
      // one block's values in registers at a time: the next one's inputs wait for these sums
      asm volatile("" : "+v"(rr[0]), "+v"(rr[1]), "+v"(rr[2]), "+v"(cm[0][0]), "+v"(cm[0][1]), "+v"(cm[0][2]),
                   "+v"(cm[1][0]), "+v"(cm[1][1]), "+v"(cm[1][2]), "+v"(cm[2][0]), "+v"(cm[2][1]), "+v"(cm[2][2])
                   : : "memory");
    };
    block(std::integral_constant<int, 0>());
    block(std::integral_constant<int, 1>());
    block(std::integral_constant<int, 2>());
    block(std::integral_constant<int, 3>());
    load_tile(min(tile + stride, ntile - 1));
    // residual: the cell's source load enters once, then the sum over the node's 16 lanes
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      double r = cell_ok ? rr[i] - (q.h == 0 ? p.src[i] * adet : 0.0) : 0.0;   // selected: 0 times an Inf state is NaN
      r += dpp_f64<0xB1, 0xf>(r);
      r += dpp_f64<0x4E, 0xf>(r);
      r += dpp_f64<0x141, 0xf>(r);
      r += dpp_f64<0x140, 0xf>(r);
      rr[i] = r;
    }
    if (p.f && node_ok && l16 < 3) p.f[L0 + l16] = l16 == 0 ? rr[0] : (l16 == 1 ? rr[1] : rr[2]);
    gather_lds_sync();   // a wave writes and reads its own line's rows
    if (p.vals) store_line(row[w], p.vals, base, len, run, min(kN8, sx - I0), lane);
    gather_lds_sync();   // the staged state and the rows are read
  }
}

// General (trilinear) hex8 cells, three fields, FP64: node-centric assembly with no workspace.
//
// The element stiffness block of vertices a and b is T_ab = sum_q s_q g_a(q) g_b(q)^T over the
// 2x2x2 Gauss points, with g_b(q) = C_q d_b(q) (C_q the cofactors of the point's Jacobian, d_b the
// reference gradient) and s_q its weight over det^2.  Everything about a point's Jacobian is formed
// once per (cell, point) and put in LDS; each lane then forms blocks of one row of the matrix.
//
// Signs and scales.  With J' the Jacobian from edge differences (hi - lo without their signs and
// halves: dN_b/dxi_m = s_bm L L / 2, L = (1 +- 1/sqrt3)/2), a lane at point q sees
// J = J' S_q / 2, S_q = diag of the point's signs, so J^-T dN_b = C' d(q ^ b) / det J' with
// d(r)_x = sigma(r_x) L(r_y) L(r_z), sigma = +1 where point and vertex agree on the axis, -1 where
// not, L the larger weight where they agree: the reference gradients depend on r = q ^ b only.
constexpr double kLp = 0.78867513459481288225, kLm = 0.21132486540518711775;   // (1 +- 1/sqrt3) / 2
constexpr int kPtStride = 12;   // doubles per (cell, point): C' (9), s, w |det J|, padding

__device__ __forceinline__ constexpr double gL(int r) { return r ? kLm : kLp; }
__device__ __forceinline__ constexpr double gS(int r) { return r ? -1.0 : 1.0; }

// Lane t of a group of eight <-> corner bits: z = t >> 2, (x, y) = (t & 3), complemented where z = 1,
// so that the neighbour along x, y, z is lane t ^ 1, t ^ 2, t ^ 7: one DPP move each.
__device__ __forceinline__ int corner_of_lane(int t) { return (t & 4) ? (t ^ 3) : t; }

template <int AXIS>
__device__ __forceinline__ double corner_swap(double x) {
  return dpp_f64<AXIS == 0 ? 0xB1 : (AXIS == 1 ? 0x4E : 0x141), 0xf>(x);
}

// J' at this lane's point from this lane's corner value of one coordinate (eight lanes per cell).
__device__ __forceinline__ void corner_grad(double X, double &gx, double &gy, double &gz) {
  const double px = corner_swap<0>(X);
  const double ex = X - px, ix = kLp * X + kLm * px;
  const double py = corner_swap<1>(ix), pe = corner_swap<1>(ex);
  const double ey = ix - py, iy = kLp * ix + kLm * py, exy = kLp * ex + kLm * pe;
  const double pz = corner_swap<2>(iy), p0 = corner_swap<2>(exy), p1 = corner_swap<2>(ey);
  gz = iy - pz;
  gx = kLp * exy + kLm * p0;
  gy = kLp * ey + kLm * p1;
}

// The point table entry of this lane: corner coordinates in, C', s and w |det J| out.
// (ok false: a cell outside the mesh, whose point weights are zero.)
__device__ __forceinline__ void point_entry(double X, double Y, double Z, int t, bool ok, double *tab) {
  double J[3][3];
  corner_grad(X, J[0][0], J[0][1], J[0][2]);
  corner_grad(Y, J[1][0], J[1][1], J[1][2]);
  corner_grad(Z, J[2][0], J[2][1], J[2][2]);
  double C[9];
  C[0] = J[1][1] * J[2][2] - J[1][2] * J[2][1];
  C[1] = J[1][2] * J[2][0] - J[1][0] * J[2][2];
  C[2] = J[1][0] * J[2][1] - J[1][1] * J[2][0];
  C[3] = J[0][2] * J[2][1] - J[0][1] * J[2][2];
  C[4] = J[0][0] * J[2][2] - J[0][2] * J[2][0];
  C[5] = J[0][1] * J[2][0] - J[0][0] * J[2][1];
  C[6] = J[0][1] * J[1][2] - J[0][2] * J[1][1];
  C[7] = J[0][2] * J[1][0] - J[0][0] * J[1][2];
  C[8] = J[0][0] * J[1][1] - J[0][1] * J[1][0];
  const double det = J[0][0] * C[0] + J[0][1] * C[1] + J[0][2] * C[2];
  const int q = corner_of_lane(t);
  // sign of S_q: an odd number of low sides is negative; the true determinant is det * S_q / 8, and
  // the measure takes the sign of the first point's (Intrepid2 computeCellMeasure)
  const double s8 = (__popc(q) & 1) ? 0.125 : -0.125;
  const int hi = __double2hiint(det * s8);
  int h0 = __builtin_amdgcn_update_dpp(0, hi, 0x00, 0xf, 0xf, false);    // lanes 0-3: lane 0's
  const int h1 = __builtin_amdgcn_update_dpp(0, h0, 0x141, 0xf, 0xf, false);   // lanes 4-7: lane 3's copy
  h0 = (t & 4) ? h1 : h0;
  const double w = ok ? (h0 < 0 ? -s8 : s8) : 0.0;
  double id = __builtin_amdgcn_rcp(det);   // 1 / det to within an ulp: two Newton steps
  id = __builtin_fma(__builtin_fma(-det, id, 1.0), id, id);
  id = __builtin_fma(__builtin_fma(-det, id, 1.0), id, id);
  double2 *o = reinterpret_cast<double2 *>(tab + q * kPtStride);
  o[0] = make_double2(C[0], C[1]);
  o[1] = make_double2(C[2], C[3]);
  o[2] = make_double2(C[4], C[5]);
  o[3] = make_double2(C[6], C[7]);
  o[4] = make_double2(C[8], ok ? w * id : 0.0);
  o[5] = make_double2(w * det, 0.0);
}

// Blocks T_ab (and mass sums) of one row vertex a and NBL = 2^NX vertices b that differ in their
// first NX axes (index k of block: corner bits bb ^ k on those axes, bb the lane's base corner), over
// the eight points of the lane's cell.  fa = a ^ bb.  m0 = sum_q w |det| N_a.
template <int NX, bool TR>
__device__ __forceinline__ void row_blocks(const double *tab, int bb, int fa, double (&T)[1 << NX][3][3],
                                           double (&M)[1 << NX], double &m0) {
  constexpr int NBL = 1 << NX;
  // of vertex a along each axis at the point on base corner bb's side (0) and the other (1)
  const bool ax = fa & 1, ay = fa & 2, az = fa & 4;
  const double Lx[2] = {ax ? kLm : kLp, ax ? kLp : kLm}, Ly[2] = {ay ? kLm : kLp, ay ? kLp : kLm},
               Lz[2] = {az ? kLm : kLp, az ? kLp : kLm};
  const double sx = ax ? -1.0 : 1.0, sy = ay ? -1.0 : 1.0, sz = az ? -1.0 : 1.0;
  double YZ[2][2], XZ[2][2], XY[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      YZ[i][j] = sx * Ly[i] * Lz[j];
      XZ[i][j] = sy * Lx[i] * Lz[j];
      XY[i][j] = sz * Lx[i] * Ly[j];
    }
  const double Lzs[2] = {sz * Lz[0], sz * Lz[1]};
#pragma unroll
  for (int k = 0; k < NBL; ++k) {
    M[k] = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) T[k][i][j] = 0.0;
  }
  m0 = 0.0;
#pragma unroll
  for (int kq = 0; kq < 8; ++kq) {
    const int qx = kq & 1, qy = (kq >> 1) & 1, qz = kq >> 2;   // the point relative to corner bb
    const double2 *o = reinterpret_cast<const double2 *>(tab + (bb ^ kq) * kPtStride);
    const double2 c0 = o[0], c1 = o[1], c2 = o[2], c3 = o[3], c4 = o[4];
    const double C[3][3] = {{c0.x, c0.y, c1.x}, {c1.y, c2.x, c2.y}, {c3.x, c3.y, c4.x}};
    const double mu = o[5].x * XY[qx][qy] * Lzs[qz];   // w |det| N_a
    const double dx = gS(qx) * c4.y * YZ[qy][qz], dy = gS(qy) * c4.y * XZ[qx][qz], dz = gS(qz) * c4.y * XY[qx][qy];
    double v[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) v[i] = C[i][0] * dx + C[i][1] * dy + C[i][2] * dz;
    m0 += mu;
    // the gradients of two vertices along x differ in the sign of P and the weight of Q
    double P[NX][3], Q[NX][3];
#pragma unroll
    for (int y = 0; y < NX; ++y)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        P[y][j] = C[j][0] * (gL(qy ^ y) * gL(qz));
        Q[y][j] = __builtin_fma(C[j][2], gL(qy ^ y) * gS(qz), (y ? -1.0 : 1.0) * (C[j][1] * (gS(qy) * gL(qz))));
      }
#pragma unroll
    for (int k = 0; k < NBL; ++k) {
      const int rx = qx ^ (k & 1), ry = NX > 1 ? qy ^ ((k >> 1) & 1) : qy, rz = qz;
      double g[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) g[j] = __builtin_fma(Q[k >> 1][j], gL(rx), gS(rx) * P[k >> 1][j]);
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) T[k][i][j] += v[i] * g[j];
      if (TR) M[k] += mu * (gL(rx) * gL(ry) * gL(rz));
    }
    // one point's data in registers at a time: the next point's address waits for these sums (left
    // to itself the compiler loads all eight points first and spills)
#pragma unroll
    for (int k = 0; k < NBL; ++k)
      asm volatile("" : "+v"(bb), "+v"(T[k][0][0]), "+v"(T[k][0][1]), "+v"(T[k][0][2]), "+v"(T[k][1][0]), "+v"(T[k][1][1]),
                   "+v"(T[k][1][2]), "+v"(T[k][2][0]), "+v"(T[k][2][1]), "+v"(T[k][2][2]), "+v"(M[k]));
  }
}

// One workgroup: 4 x 4 nodes of one lattice plane, a wave per line of four nodes along x, 16 lanes
// per node: lane (cell c around the node, half h) forms the blocks of the four vertices of c on its
// low / high z side.  The 5 x 5 x 2 cells' points are formed once for the 16 nodes (50 cells instead
// of 128).  Blocks of different cells that meet in one neighbour are summed by DPP moves along x, y,
// z in that order, one lane then writes each neighbour's block into the row buffer (which lies over
// the point table) and the wave stores the rows, its four nodes as one range where their LIDs follow
// each other.  Every sum has a fixed order: results are bitwise reproducible.
// Bound by VALU issue (about 515 instructions per node, 63% busy at two workgroups per CU, 208
// VGPRs; held to 168 for three it spills and takes 18% longer) and waits (32% of wave time).  Transient FP64, against the element
// kernel with its 4.6 KB of blocks per element and the gather: 128^3 8.23 -> 2.84 ms, 96^3 3.61 ->
// 1.21 ms, 18^3 238 -> 28 us.
struct Elastic8GParams {
  Elastic8Params p;
  const double *X, *Y, *Z;
};

template <bool TR>
__global__ __launch_bounds__(256, 2) void k_elastic8_general(Elastic8GParams gp) {
  const Elastic8Params &p = gp.p;
  __shared__ __align__(16) double tab[kC8 * 8 * kPtStride];   // points; then the rows of the 16 nodes
  __shared__ double vtx[TR ? 9 : 6][kV8];                            // x, y, z, u + b_R v, a_R v + a
  static_assert(kN8 * kN8 * kRow8 <= kC8 * 8 * kPtStride, "rows fit over the point table");
  int tid = threadIdx.x;
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, n = lane >> 4;
  const NodeLane q(l16);
  const int ox = q.ox, oy = q.oy, oz = q.oz, h = q.h;
  const int sx = p.nx + 1, sxy = sx * (p.ny + 1);
  const int gx = (sx + kN8 - 1) / kN8, gy = (p.ny + 1 + kN8 - 1) / kN8;
  const int ntile = gx * gy * (p.nz + 1);
  const bool tra = TR && p.xddot;
  const double lamf = p.nu / ((1.0 + p.nu) * (1.0 - 2.0 * p.nu)), muf = 0.5 / (1.0 + p.nu);
  const double cK = TR ? p.beta + p.alpha * p.rb : p.beta;
  const double cM = TR ? p.alpha * p.ra + (tra ? p.gamma2 : 0.0) : 0.0;
  // A tile's vertices (clamped into the mesh: what lies outside belongs to no cell of the mesh) are
  // loaded while the tile before is computed, ahead of its row stores: one counter tracks a wave's
  // loads and stores, so loads issued after the stores would wait for them.
  double vx[3], vu[3], vm[3];
  auto load_vertex = [&](int tile) {
    const int t = min(tid, kV8 - 1);
    const int I0 = tile % gx * kN8, J0 = tile / gx % gy * kN8, K = tile / (gx * gy);
    const int ix = min(max(I0 - 1 + t % (kN8 + 2), 0), p.nx);
    const int iy = min(max(J0 - 1 + t / (kN8 + 2) % (kN8 + 2), 0), p.ny);
    const int iz = min(max(K - 1 + t / ((kN8 + 2) * (kN8 + 2)), 0), p.nz);
    const int vi = ix + sx * iy + sxy * iz;
    const int32_t L = p.point_lid[3 * vi];
    vx[0] = gp.X[vi];
    vx[1] = gp.Y[vi];
    vx[2] = gp.Z[vi];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      vu[j] = p.x[L + j];
      if constexpr (TR) {
        const double v = p.xdot[L + j], a = tra ? p.xddot[L + j] : 0.0;
        vu[j] += p.rb * v;
        vm[j] = p.ra * v + a;
      }
    }
  };
  // LID of this lane's node and modulus of its cell, with the tile's vertices
  int32_t Ln;
  double En;
  auto load_node = [&](int tile) {
    const int I = tile % gx * kN8 + n, J = tile / gx % gy * kN8 + w, K = tile / (gx * gy);
    Ln = p.point_lid[3 * (min(I, p.nx) + sx * min(J, p.ny) + sxy * K)];
    const int cx = min(max(I - 1 + ox, 0), p.nx - 1), cy = min(max(J - 1 + oy, 0), p.ny - 1),
              cz = min(max(K - 1 + oz, 0), p.nz - 1);
    En = p.coef[cx + p.nx * (cy + p.ny * cz)];
  };
  load_vertex(min(static_cast<int>(blockIdx.x), ntile - 1));
  load_node(min(static_cast<int>(blockIdx.x), ntile - 1));
  for (int tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
    asm volatile("" : "+v"(tid));   // the staging indices are formed per tile, not kept in registers
    const int I0 = tile % gx * kN8, J0 = tile / gx % gy * kN8, K = tile / (gx * gy);
    if (tid < kV8)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        vtx[j][tid] = vx[j];
        vtx[3 + j][tid] = vu[j];
        if constexpr (TR) vtx[6 + j][tid] = vm[j];
      }
    // this lane's node and cell
    const int I = I0 + n, Jy = J0 + w;
    const bool node_ok = I <= p.nx && Jy <= p.ny;
    const int32_t L0 = Ln;
    const int cx = I - 1 + ox, cy = Jy - 1 + oy, cz = K - 1 + oz;
    const bool cell_ok = node_ok && cx >= 0 && cx < p.nx && cy >= 0 && cy < p.ny && cz >= 0 && cz < p.nz;
    const double E = En;
    __syncthreads();
    // points of the cells
#pragma unroll 1
    for (int task = tid; task < kC8 * 8; task += 256) {
      const int c = task >> 3, t = task & 7, b = corner_of_lane(t);
      const int lx = c % (kN8 + 1), ly = c / (kN8 + 1) % (kN8 + 1), lz = c / ((kN8 + 1) * (kN8 + 1));
      const int vi = lx + (b & 1) + (kN8 + 2) * (ly + ((b >> 1) & 1) + (kN8 + 2) * (lz + (b >> 2)));
      const bool ok = static_cast<unsigned>(I0 - 1 + lx) < static_cast<unsigned>(p.nx) &&
                      static_cast<unsigned>(J0 - 1 + ly) < static_cast<unsigned>(p.ny) &&
                      static_cast<unsigned>(K - 1 + lz) < static_cast<unsigned>(p.nz);
      point_entry(vtx[0][vi], vtx[1][vi], vtx[2][vi], t, ok, tab + c * 8 * kPtStride);
    }
    const int64_t base = p.rowptr[L0];
    const int len = min(static_cast<int>(p.rowptr[L0 + 1] - base), 81);
    const uint16_t *np = p.nperm + static_cast<int64_t>(L0 / 3) * p.nperm_w;
    // neighbour slot of block k: dx = 0 where k complements the cell's side, -1 / +1 otherwise
    int pos[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int dx = (k & 1) ? 1 : 2 * ox, dy = (k & 2) ? 1 : 2 * oy, dz = oz + h;
      pos[k] = np[dx + 3 * dy + 9 * dz];
    }
    __syncthreads();
    double T[4][3][3], M[4], m0;
    const int bb = ox + 2 * oy + 4 * h;           // base corner: the cell's far side, half h
    const int av = (1 - ox) + 2 * (1 - oy) + 4 * (1 - oz);
    const int cl = (n + ox) + (kN8 + 1) * (w + oy + (kN8 + 1) * oz);
    row_blocks<2, TR>(tab + cl * 8 * kPtStride, bb, av ^ bb, T, M, m0);
    const double lam = cell_ok ? E * lamf : 0.0, mu = cell_ok ? E * muf : 0.0;
    double rr[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int bx = ox ^ (k & 1), by = oy ^ (k >> 1);
      const int vi = (n + ox + bx) + (kN8 + 2) * ((w + oy + by) + (kN8 + 2) * (oz + h));
      const double trs = T[k][0][0] + T[k][1][1] + T[k][2][2];
      const double Mab = TR ? p.rho * M[k] : 0.0;
      double ut[3], mt[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) { ut[j] = vtx[3 + j][vi]; mt[j] = TR ? vtx[TR ? 6 + j : 0][vi] : 0.0; }
      double t9[3][3];
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) t9[i][j] = T[k][i][j];
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const double Kv = lam * t9[i][j] + mu * t9[j][i] + (i == j ? mu * trs : 0.0);
          rr[i] += Kv * ut[j];
          double jv = cK * Kv;
          if (TR && i == j) {
            jv += cM * Mab;
            rr[i] += Mab * mt[j];
          }
          T[k][i][j] = jv;
        }
    }
    // residual: the cell's source load enters once, then the sum over the node's 16 lanes
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      double r = cell_ok ? rr[i] - (h == 0 ? p.src[i] * m0 : 0.0) : 0.0;   // selected: 0 times an Inf state is NaN
      r += dpp_f64<0xB1, 0xf>(r);
      r += dpp_f64<0x4E, 0xf>(r);
      r += dpp_f64<0x141, 0xf>(r);
      r += dpp_f64<0x140, 0xf>(r);
      rr[i] = r;
    }
    if (p.f && node_ok && l16 < 3) p.f[L0 + l16] = l16 == 0 ? rr[0] : (l16 == 1 ? rr[1] : rr[2]);
    load_vertex(min(tile + static_cast<int>(gridDim.x), ntile - 1));
    load_node(min(tile + static_cast<int>(gridDim.x), ntile - 1));
    if (p.vals) {
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          T[0][i][j] = meet<0>(T[0][i][j], l16 > 7);
          T[1][i][j] = meet<1>(T[1][i][j], l16 > 7);
          T[2][i][j] = meet<2>(T[2][i][j], l16 > 7);
          T[3][i][j] = meet<3>(T[3][i][j], l16 > 7);
        }
    }
    __syncthreads();   // every wave is done with the points and the vertices: the rows go over the points
    if (p.vals) {
      // the rows of the wave's nodes, one after another as in the matrix where their LIDs are
      const int64_t base0 = __shfl(base, 0);
      const int32_t L00 = __shfl(L0, 0);
      const bool run = __all(!node_ok || L0 == L00 + 3 * n);
      double *rows = tab + w * kN8 * kRow8;
      double *mine = rows + (run ? static_cast<int>(base - base0) : n * kRow8);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (node_ok && pos[k] + 2 < len && owns_block(q, k)) {
#pragma unroll
          for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) mine[i * len + pos[k] + j] = T[k][i][j];
        }
      }
      gather_lds_sync();
      if (Jy <= p.ny) store_line(rows, p.vals, base, len, run, min(kN8, sx - I0), lane);
    }
    __syncthreads();
  }
}

// The same row blocks on an uploaded hex8 mesh (one block): one wave per two nodes (LIDs 3 n, 3 n + 1,
// 3 n + 2), 32 lanes per node: lane (element instance c of eight at a time, corner y and z) forms the
// blocks of the two vertices along x.  Bound by LDS (70% busy: points and row adds) and VALU issue (about
// 657 instructions per node, 47% busy: no two nodes share a point table) at two waves per SIMD (245 VGPRs,
// 16 KB of LDS per wave).  Transient FP64, shuffled 64x61x67: 1.19 -> 0.64 ms (element kernel and gather
// before).  Instances come from the node's list (ascending), the row positions from their slot maps; the
// blocks are added into the node's rows in LDS instance by instance, so the sums have a fixed order, and
// the rows are stored once.
struct Elastic8UParams {
  Elastic8Params p;
  const double *X, *Y, *Z;
  int64_t nnodes;
  const int64_t *conn;      // [E][8] vertex ids
  const int32_t *elem_lid;  // [E][24]
  const int64_t *occ_ptr;   // [nnodes + 1]
  const int32_t *occ;       // e * 8 + a per instance
  const uint16_t *slot;     // [instances][8]
};

template <bool TR>
__global__ __launch_bounds__(64, 2) void k_elastic8_upload(Elastic8UParams gp) {
  const Elastic8Params &p = gp.p;
  __shared__ __align__(16) double tab[2 * 8 * 8 * kPtStride];
  __shared__ double rows[2][kRow8];
  const int lane = threadIdx.x;
  const int n = lane >> 5, c = (lane >> 2) & 7, bb = (lane & 3) << 1;   // base corner (0, y, z)
  const int t = lane & 7, tb = corner_of_lane(t);
  const int ts = tb ^ ((tb >> 1) & 1);   // binary corner -> element vertex order (its own inverse)
  const bool tra = TR && p.xddot;
  const double lamf = p.nu / ((1.0 + p.nu) * (1.0 - 2.0 * p.nu)), muf = 0.5 / (1.0 + p.nu);
  const double cK = TR ? p.beta + p.alpha * p.rb : p.beta;
  const double cM = TR ? p.alpha * p.ra + (tra ? p.gamma2 : 0.0) : 0.0;
  const int64_t npair = (gp.nnodes + 1) / 2;
  // The first eight instances of a pair are found and their coordinates loaded while the pair before
  // is computed, a step of the chain (list ends, instance, vertices, coordinates) at a time, the
  // coordinates ahead of that pair's row stores.
  int64_t rn[3];            // list ends of both nodes
  int32_t on[3];            // instance of this lane's points for either node, and of its blocks
  int64_t vn[2];
  int32_t Ln[2];
  double Xn[2][3];
  auto load_ends = [&](int64_t pair) {
    const int64_t q = min(pair, npair - 1);
    rn[0] = gp.occ_ptr[2 * q];
    rn[1] = gp.occ_ptr[2 * q + 1];
    rn[2] = gp.occ_ptr[min(2 * q + 2, gp.nnodes)];
  };
  // (past a list's end: its first instance, never used)
  auto load_occ = [&]() {
    const int64_t k = lane >> 3;
    on[0] = gp.occ[rn[0] + k < rn[1] ? rn[0] + k : rn[0]];
    on[1] = gp.occ[rn[1] + k < rn[2] ? rn[1] + k : rn[0]];
    const int64_t lo = n ? rn[1] : rn[0], hi = n ? rn[2] : rn[1];
    on[2] = gp.occ[lo + c < hi ? lo + c : rn[0]];
  };
  auto load_vertices = [&]() {
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      vn[m] = gp.conn[(static_cast<int64_t>(on[m]) & ~int64_t(7)) + ts];
      Ln[m] = gp.elem_lid[((static_cast<int64_t>(on[2]) & ~int64_t(7)) + ((bb | m) ^ ((bb >> 1) & 1))) * 3];
    }
  };
  auto load_coords = [&]() {
#pragma unroll
    for (int m = 0; m < 2; ++m) { Xn[m][0] = gp.X[vn[m]]; Xn[m][1] = gp.Y[vn[m]]; Xn[m][2] = gp.Z[vn[m]]; }
  };
  load_ends(blockIdx.x);
  load_occ();
  load_vertices();
  load_coords();
  for (int64_t pair = blockIdx.x; pair < npair; pair += gridDim.x) {
    const int64_t node0 = 2 * pair, node = min(node0 + n, gp.nnodes - 1);
    const bool node_ok = node0 + n < gp.nnodes;
    // instance ranges of both nodes (wave-uniform) and of this lane's
    const int64_t r0 = rn[0], r1 = rn[1], r2 = rn[2];
    load_ends(pair + gridDim.x);
    const int64_t first = n ? r1 : r0;
    const int cnt = node_ok ? static_cast<int>((n ? r2 : r1) - first) : 0;
    const int most = max(static_cast<int>(r1 - r0), static_cast<int>(r2 - r1));
    const int32_t L0 = static_cast<int32_t>(3 * node);
    const int64_t base = p.rowptr[L0];
    const int len = min(static_cast<int>(p.rowptr[L0 + 1] - base), 81);
    if (p.vals)
      for (int k = lane; k < 2 * kRow8; k += 64) (&rows[0][0])[k] = 0.0;
    double racc[3] = {0.0, 0.0, 0.0};
    const int32_t on2 = on[2], L2[2] = {Ln[0], Ln[1]};
    for (int g = 0; g < most; g += 8) {
      // points: eight lanes per instance, node 0's instances, then node 1's
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int64_t lo = m ? r1 : r0, hi = m ? r2 : r1;
        const int64_t k = lo + g + (lane >> 3);
        const bool ok = k < hi;
        double X = Xn[m][0], Y = Xn[m][1], Z = Xn[m][2];
        if (g > 0) {   // a node of more than eight instances (uniform over the wave)
          const int64_t v = gp.conn[(ok ? static_cast<int64_t>(gp.occ[k]) & ~int64_t(7) : 0) + ts];
          X = gp.X[v];
          Y = gp.Y[v];
          Z = gp.Z[v];
        }
        point_entry(X, Y, Z, t, ok, tab + (m * 8 + (lane >> 3)) * 8 * kPtStride);
      }
      // this lane's instance, its modulus, vertices' state and row positions
      const bool ok = g + c < cnt;
      const int64_t k = ok ? first + g + c : r0;
      const int32_t occ = g == 0 ? on2 : gp.occ[k];
      const int64_t e = occ >> 3;
      const int as = occ & 7, av = as ^ ((as >> 1) & 1);
      const double E = p.coef[e];
      double ut[2][3], mt[2][3];
      int pos[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int bs = (bb | b) ^ ((bb >> 1) & 1);
        const int32_t L = g == 0 ? L2[b] : gp.elem_lid[(8 * e + bs) * 3];
        pos[b] = gp.slot[8 * k + bs];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          ut[b][j] = p.x[L + j];
          mt[b][j] = 0.0;
          if constexpr (TR) {
            const double v = p.xdot[L + j], a = tra ? p.xddot[L + j] : 0.0;
            ut[b][j] += p.rb * v;
            mt[b][j] = p.ra * v + a;
          }
        }
      }
      if (g == 0) load_occ();
      gather_lds_sync();
      double T[2][3][3], M[2], m0;
      row_blocks<1, TR>(tab + (n * 8 + c) * 8 * kPtStride, bb, av ^ bb, T, M, m0);
      if (g == 0) load_vertices();
      const double lam = ok ? E * lamf : 0.0, mu = ok ? E * muf : 0.0;
      if (!ok) m0 = 0.0;
      double rr[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const double trs = T[b][0][0] + T[b][1][1] + T[b][2][2];
        const double Mab = TR ? p.rho * M[b] : 0.0;
        double t9[3][3];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int j = 0; j < 3; ++j) t9[i][j] = T[b][i][j];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            const double Kv = lam * t9[i][j] + mu * t9[j][i] + (i == j ? mu * trs : 0.0);
            rr[i] += Kv * ut[b][j];
            double jv = cK * Kv;
            if (TR && i == j) {
              jv += cM * Mab;
              rr[i] += Mab * mt[b][j];
            }
            T[b][i][j] = jv;
          }
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) racc[i] += ok ? rr[i] - (bb == 0 ? p.src[i] * m0 : 0.0) : 0.0;
      if (p.vals) {
        // one wave's LDS operations execute in order and the lanes of one step hit distinct entries:
        // every entry is summed in instance order
#pragma unroll
        for (int cc = 0; cc < 8; ++cc)
          if (c == cc && ok)
#pragma unroll
            for (int b = 0; b < 2; ++b)
              if (pos[b] + 2 < len)
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                  for (int j = 0; j < 3; ++j) atomicAdd(&rows[n][i * len + pos[b] + j], T[b][i][j]);
      }
      gather_lds_sync();   // the points are read; the next eight instances go over them
    }
    load_coords();
    // residual over the node's 32 lanes (the total ends in the second row of 16), rows
#pragma unroll
    for (int i = 0; i < 3; ++i) racc[i] = group_sum<32>(racc[i]);
    const int l32 = lane & 31;
    if (p.f && node_ok && l32 >= 16 && l32 < 19) p.f[L0 + l32 - 16] = l32 == 16 ? racc[0] : (l32 == 17 ? racc[1] : racc[2]);
    if (p.vals) {
      for (int m = 0; m < 2 && node0 + m < gp.nnodes; ++m)
        row_store(rows[m], p.vals + __shfl(base, 32 * m), 3 * __shfl(len, 32 * m), lane);
      gather_lds_sync();
    }
  }
}

// hex27 bricks, FP64 calls that want the matrix: node rows without element blocks.  k_points27 writes the
// points of each cell (27 x 128 bytes); one wave then owns the nodes of a line along x of one class, the
// parity (py, pz) of their y and z lattice coordinates, and marches over the line's cells.  The cells
// around such a line are 4, 2, 2 or 1 per x position for (py, pz) = (0,0), (1,0), (0,1), (1,1).  Per cell
// the wave forms the 3 x 3 blocks of its three nodes (x lattice 0, 1, 2 of the cell) with the cell's 27
// nodes on v_mfma_f64_16x16x4f64:
//   T[(a,k),(b,l)] = sum_q s_q (C dN_a)_k (C dN_b)_l,   C the cofactors of J, s = w / det.
// Operand row l % 16 = a + 4 k, columns b in two tiles per l: as lane l of the product holds D rows
// l / 16 + 4 i, it ends up with all nine entries of the pair (a = l / 16, b = l % 16), so no Gram matrix
// goes through LDS.  Row group 3 is w det N_a: its sum over the points is the source load.  A lane
// holds one of the 16 values of each of its row's points (one coalesced load per cell) and the operands are
// formed from DPP broadcasts of them: read from LDS instead (16 lanes the same 16 bytes), they took 61% of
// its cycles (1.84 ms against 1.53 at 33^3).  Blocks are added in lattice order into the rows in LDS (one
// wave's LDS operations execute in order and the lanes of one add hit distinct entries: a fixed order of
// sums, the same for every split of a
// line), and rows are stored once in CRS order when their last cell is done.
//
// Bound by issue: an FP64 product takes its SIMD's 64 cycles whole (a wave's VALU work, and the other
// waves', wait for it: measured), 0.90 M of 2.71 M cycles per SIMD at 33^3 (46% of its rows and columns are
// used), and 238 k VALU instructions 0.95 M more, at seven waves per CU (23 KB of LDS each).  FP64 33^3,
// against the element kernel with its 55 KB of blocks per element and the gather: steady 1.79 -> 1.17 ms,
// transient 2.16 -> 1.72 ms (with the mass matrix on the products too, 2.29 ms: it spilled); 12^3 steady
// 225 -> 125 us, transient 263 -> 150 us, 4^3 steady 124 -> 48 us.
// The FP32 and split-BF16 forms keep those: their results are rounded there.
struct Node27Params {
  Elastic8Params p;
  const double *pts;        // [cells][27][4][4]: rows k of C with s; w det, 0, 0, 1
  int chunk, nchunk;        // x positions per workgroup, workgroups per line
};

__global__ __launch_bounds__(256) void k_points27(int nx, int ny, int64_t ncell, const double *__restrict__ X,
                                                  const double *__restrict__ Y, const double *__restrict__ Z,
                                                  double *__restrict__ pts) {
  // entries staged in LDS and stored by consecutive lanes: 47 -> 27 us at 33^3 (124 MB)
  __shared__ double out[256][17];
  const int64_t id0 = static_cast<int64_t>(blockIdx.x) * 256, n = ncell * 27;
  const int64_t id = min(id0 + threadIdx.x, n - 1);   // past the last point: that point again, not stored
  const int64_t c = id / 27;
  const int q = static_cast<int>(id - 27 * c), qd[3] = {q % 3, q / 3 % 3, q / 9};
  const int64_t i = c % nx, j = c / nx % ny, k = c / (static_cast<int64_t>(nx) * ny);
  const int64_t v0 = i + (nx + 1) * (j + static_cast<int64_t>(ny + 1) * k), sy = nx + 1,
                sz = static_cast<int64_t>(nx + 1) * (ny + 1);
  double L[2][3], w = 1.0;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double xi = (qd[d] - 1) * 0.77459666924148337704;
    L[0][d] = 0.5 * (1.0 - xi);
    L[1][d] = 0.5 * (1.0 + xi);
    w *= qd[d] == 1 ? 8.0 / 9.0 : 5.0 / 9.0;
  }
  double J[3][3] = {};
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const int ox = kHexV[b][0], oy = kHexV[b][1], oz = kHexV[b][2];
    const int64_t v = v0 + ox + oy * sy + oz * sz;
    const double gx = L[ox][0], gy = L[oy][1], gz = L[oz][2], P[3] = {X[v], Y[v], Z[v]};
    const double d[3] = {(ox ? 0.5 : -0.5) * gy * gz, gx * (oy ? 0.5 : -0.5) * gz, gx * gy * (oz ? 0.5 : -0.5)};
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) J[i][j] += P[i] * d[j];
  }
  double C[9];
  C[0] = J[1][1] * J[2][2] - J[1][2] * J[2][1];
  C[1] = J[1][2] * J[2][0] - J[1][0] * J[2][2];
  C[2] = J[1][0] * J[2][1] - J[1][1] * J[2][0];
  C[3] = J[0][2] * J[2][1] - J[0][1] * J[2][2];
  C[4] = J[0][0] * J[2][2] - J[0][2] * J[2][0];
  C[5] = J[0][1] * J[2][0] - J[0][0] * J[2][1];
  C[6] = J[0][1] * J[1][2] - J[0][2] * J[1][1];
  C[7] = J[0][2] * J[1][0] - J[0][0] * J[1][2];
  C[8] = J[0][0] * J[1][1] - J[0][1] * J[1][0];
  const double det = J[0][0] * C[0] + J[0][1] * C[1] + J[0][2] * C[2];
  const double s = w / det;
  double *o = out[threadIdx.x];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
#pragma unroll
    for (int m = 0; m < 3; ++m) o[4 * k + m] = C[3 * k + m];
    o[4 * k + 3] = s;
  }
  o[12] = w * det;
  o[13] = o[14] = 0.0;
  o[15] = 1.0;
  __syncthreads();
  const int left = static_cast<int>(min(n - id0, int64_t(256))) * 16;
#pragma unroll
  for (int k = threadIdx.x; k < 4096; k += 256)
    if (k < left) pts[16 * id0 + k] = out[k >> 4][k & 15];
}

constexpr int rows27(int n9) { return 5 * n9 + 2 * 3 * n9; }   // current, middle and next nodes of a line
constexpr int kRows27 = rows27(25 * 9);

// entry N of the row of 16 lanes' values, in all its lanes; entry N of each quad's
template <int N>
__device__ __forceinline__ double row_entry(double v) { return __builtin_amdgcn_update_dpp(v, v, 0x150 + N, 0xf, 0xf, true); }
template <int N>
__device__ __forceinline__ double quad_entry(double v) {
  return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), N * 0x55, 0xf, 0xf, true),
                          __builtin_amdgcn_mov_dpp(__double2loint(v), N * 0x55, 0xf, 0xf, true));
}

// Stores a node's three rows from lattice order (slot (dx Dy + dy) Dz + dz, nine entries each) in CRS
// order.  np0, np1: the node's nperm entries lane, lane + 64; inv: of each neighbour, its slot's entries.
__device__ __forceinline__ void store_node27(const double *buf, uint16_t *inv, int rx, int ry, int rz, int np0, int np1,
                                             double *vals, int64_t base, int len, int lane) {
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int s = lane + 64 * r, ps = r ? np1 : np0;
    const int dx = s % 5 - 2 + rx, dy = s / 5 % 5 - 2 + ry, dz = s / 25 - 2 + rz;
    if (s < 125 && ps < 375) inv[ps / 3] = static_cast<uint16_t>(9 * ((dx * (2 * ry + 1) + dy) * (2 * rz + 1) + dz));
  }
  gather_lds_sync();
  double *dst = vals + base;
#pragma unroll 1
  for (int k = lane; k < len; k += 64) {
    const int nb = (k * 21846) >> 16;   // k / 3
    const double *b = buf + inv[nb] + (k - 3 * nb);
    __builtin_nontemporal_store(b[0], dst + k);
    __builtin_nontemporal_store(b[3], dst + len + k);
    __builtin_nontemporal_store(b[6], dst + 2 * len + k);
  }
}

template <bool TR>
__global__ __launch_bounds__(64, 2) void k_elastic27_nodes(Node27Params gp) {
  const Elastic8Params &p = gp.p;
  __shared__ double mem[kRows27];
  __shared__ double2 T1[9];          // 1D basis: value and derivative of node d at Gauss point q, [3 d + q]
  __shared__ double TA[9][3][9];     // [node y + 3 z][N N', N' N, N N of y, z][point y + 3 z]: of the row operand
  __shared__ double PP[3][3][3];     // N_a N_b of two 1D nodes at the points
  __shared__ double wdl[TR ? 28 : 1];   // the cell's w det
  __shared__ double st[27][TR ? 6 : 3];   // the cell's nodes: u + b_R v, a_R v + a
  uint16_t *inv = reinterpret_cast<uint16_t *>(&st[0][0]);   // of store_node27, between two cells
  const int lane = threadIdx.x;
  if (threadIdx.x < 9) {
    const int d = threadIdx.x / 3;
    const double xi = (static_cast<int>(threadIdx.x) % 3 - 1) * 0.77459666924148337704;
    T1[threadIdx.x] = d == 0 ? make_double2(0.5 * xi * (xi - 1.0), xi - 0.5)
                             : (d == 1 ? make_double2(1.0 - xi * xi, -2.0 * xi) : make_double2(0.5 * xi * (xi + 1.0), xi + 0.5));
  }
  __syncthreads();
  if (TR && lane < 27) PP[lane / 9][lane / 3 % 3][lane % 3] = T1[3 * (lane / 9) + lane % 3].x * T1[3 * (lane / 3 % 3) + lane % 3].x;
  for (int i = lane; i < 81; i += 64) {
    const int n = i / 9, q = i % 9;
    const double2 y = T1[3 * (n % 3) + q % 3], z = T1[3 * (n / 3) + q / 3];
    TA[n][0][q] = y.x * z.x;
    TA[n][1][q] = y.y * z.x;
    TA[n][2][q] = y.x * z.y;
  }
  __syncthreads();
  const int px = 2 * p.nx + 1, py = 2 * p.ny + 1;
  const int l16 = lane & 15, g = lane >> 4;
  const int ka = l16 >> 2, ax = min(l16 & 3, 2);   // operand row: node ax, component ka (3: the mass row)
  // nodes of this lane's columns: lattice offsets, and x basis and derivative at point 4 ks + g, of index
  // (ks + g) % 3 along x: entry ks % 3 (the y and z factors come from TA)
  int bo[2][3];
  double xb[2][3], xbd[2][3];
#pragma unroll
  for (int cb = 0; cb < 2; ++cb) {
    const int b = min(16 * cb + l16, 26);   // x fastest
    bo[cb][0] = b % 3;
    bo[cb][1] = b / 3 % 3;
    bo[cb][2] = b / 9;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const double2 x = T1[3 * bo[cb][0] + (r + g) % 3];
      xb[cb][r] = x.x;
      xbd[cb][r] = x.y;
      asm volatile("" : "+v"(xb[cb][r]), "+v"(xbd[cb][r]));
    }
  }
  // node min(lane, 26)'s LID entry from the cell's first
  const int bl = min(lane, 26);
  const unsigned lo = 3 * (bl % 3 + px * (bl / 3 % 3 + py * (bl / 9)));
  // the row node's
  double xa[3], xd[3];
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const double2 t = T1[3 * ax + (r + g) % 3];
    xa[r] = t.x;
    xd[r] = t.y;
    if (ka == 3) xd[r] = t.x;   // the mass row takes N_a alone
    asm volatile("" : "+v"(xa[r]), "+v"(xd[r]));
  }
  const bool tra = TR && p.xddot;
  const double lamf = p.nu / ((1.0 + p.nu) * (1.0 - 2.0 * p.nu)), muf = 0.5 / (1.0 + p.nu);
  const double cK = TR ? p.beta + p.alpha * p.rb : p.beta;
  const double cM = TR ? p.alpha * p.ra + (tra ? p.gamma2 : 0.0) : 0.0;
  using cint = const __attribute__((address_space(4))) int32_t;
  using clong = const __attribute__((address_space(4))) int64_t;
  const cint *plid = (const cint *)p.point_lid;
  const clong *prow = (const clong *)p.rowptr;
  // part 0: class (0,0); 1: (1,0) and (1,1); 2: (0,1).  The longest part's workgroups start first.
  const int nw = static_cast<int>(gridDim.x) / 3, part = static_cast<int>(blockIdx.x) / nw, wi = static_cast<int>(blockIdx.x) % nw;
  const int line = wi / gp.nchunk, ck = wi % gp.nchunk;
  const int LY = line % (p.ny + 1), LZ = line / (p.ny + 1);
  const int x0 = ck * gp.chunk, x1 = min(x0 + gp.chunk, p.nx);
  if (x0 >= x1) return;
  for (int cls = part; cls < 4; cls += part == 1 ? 2 : 4) {   // bit 0: py, bit 1: pz
    const int qy = cls & 1, qz = cls >> 1;
    if ((qy && LY == p.ny) || (qz && LZ == p.nz)) continue;
    const int ry = qy ? 1 : 2, rz = qz ? 1 : 2;            // reach of the nodes' neighbours
    const int Dy = 2 * ry + 1, Dz = 2 * rz + 1, n9 = Dy * Dz * 9;
    double *cur = mem, *mid = cur + 5 * n9, *nxt = mid + 3 * n9;
    for (int k = lane; k < 11 * n9; k += 64) cur[k] = 0.0;
    // cells around the line: y in [cy0, cy1], z in [cz0, cz1]
    const int cy0 = qy ? LY : max(LY - 1, 0), cy1 = min(LY, p.ny - 1);
    const int cz0 = qz ? LZ : max(LZ - 1, 0), cz1 = min(LZ, p.nz - 1);
    const int my = cy1 - cy0 + 1, nc = my * (cz1 - cz0 + 1);
    const int xs = x0 > 0 ? x0 - 1 : 0;                    // the cell before the chunk: its upper nodes
    const int nunit = (x1 - xs) * nc;
    // a cell's points and state are loaded while the cell before is computed, its nodes' LIDs one cell
    // earlier; a point's register takes the next cell's once its operands are formed
    int32_t Ln;
    double tn[7], un[3], vn[3], an[3], En;
    auto cell_of = [&](int u, int &x, int &y, int &z) {
      const int uc = min(u, nunit - 1), c = uc % nc;
      x = xs + uc / nc;
      y = cy0 + c % my;
      z = cz0 + c / my;
    };
    auto load_lid = [&](int u) {
      int x, y, z;
      cell_of(u, x, y, z);
      const int32_t *l = p.point_lid + 6 * (x + px * (y + py * z));
      Ln = l[lo];
    };
    auto points_of = [&](int u) {
      int x, y, z;
      cell_of(u, x, y, z);
      return gp.pts + (x + static_cast<int64_t>(p.nx) * (y + static_cast<int64_t>(p.ny) * z)) * (27 * 16);
    };
    auto load_state = [&](int u) {
      int x, y, z;
      cell_of(u, x, y, z);
      En = p.coef[x + static_cast<int64_t>(p.nx) * (y + static_cast<int64_t>(p.ny) * z)];
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        un[j] = p.x[Ln + j];
        vn[j] = TR ? p.xdot[Ln + j] : 0.0;
        an[j] = tra ? p.xddot[Ln + j] : 0.0;
      }
    };
    const double *pn = points_of(0);
#pragma unroll
    for (int ks = 0; ks < 7; ++ks) tn[ks] = pn[lane + 64 * ks];   // lane 16 g + e: entry e of point 4 ks + g (27: past the cell)
    load_lid(0);
    load_state(0);
    load_lid(1);
    double rr[3] = {0.0, 0.0, 0.0}, carry[3] = {0.0, 0.0, 0.0}, msum = 0.0;
    int u = 0;
    for (int x = xs; x < x1; ++x) {
      // where the step's finished nodes go
      const int P0 = 2 * x + px * (2 * LY + qy + py * (2 * LZ + qz));
      const int32_t Lc = plid[3 * P0], Lm = plid[3 * P0 + 3];
      const int64_t basec = prow[Lc], basem = prow[Lm];
      const int lenc = static_cast<int>(prow[Lc + 1] - basec), lenm = static_cast<int>(prow[Lm + 1] - basem);
      const uint16_t *npc = p.nperm + static_cast<int64_t>(Lc / 3) * p.nperm_w, *npm = p.nperm + static_cast<int64_t>(Lm / 3) * p.nperm_w;
      int nc0 = npc[lane], nc1 = npc[lane + 64], nm0 = npm[lane], nm1 = npm[lane + 64];   // nperm_w = 128
      for (int c = 0; c < nc; ++c, ++u) {
        const int ay = qy ? 1 : 2 * (LY - cy0 - c % my), az = qz ? 1 : 2 * (LZ - cz0 - c / my);
        if (g == 3) tn[6] = 0.0;   // 27 points: no 28th
        if (lane < 27)
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            st[lane][j] = TR ? un[j] + p.rb * vn[j] : un[j];
            if constexpr (TR) st[lane][3 + j] = p.ra * vn[j] + an[j];
          }
        if (TR && l16 == 12)
#pragma unroll
          for (int ks = 0; ks < 7; ++ks) wdl[4 * ks + g] = tn[ks];
        const double E = En;
        gather_lds_sync();
        load_state(u + 1);
        load_lid(u + 2);
        pn = points_of(u + 1);
        // the measure takes the sign of the first point's determinant (Intrepid2 computeCellMeasure)
        const double sg = __builtin_amdgcn_readlane(__double2hiint(tn[0]), 12) < 0 ? -1.0 : 1.0;
        double Mb[2] = {0.0, 0.0};
        if constexpr (TR) {   // sum_q w det N_a N_b, an axis at a time
#pragma unroll
          for (int cb = 0; cb < 2; ++cb) {
            const double *x = PP[min(g, 2)][bo[cb][0]], *y = PP[ay][bo[cb][1]], *z = PP[az][bo[cb][2]];
            const double x0 = x[0], x1 = x[1], x2 = x[2], y0 = y[0], y1 = y[1], y2 = y[2];
#pragma unroll
            for (int qz = 0; qz < 3; ++qz) {
              asm volatile("" : "+v"(Mb[cb]) : : "memory");   // nine weights in registers at a time
              const double *w = wdl + 9 * qz;
              Mb[cb] += z[qz] * (y0 * (x0 * w[0] + x1 * w[1] + x2 * w[2]) + y1 * (x0 * w[3] + x1 * w[4] + x2 * w[5]) +
                                 y2 * (x0 * w[6] + x1 * w[7] + x2 * w[8]));
            }
          }
        }
        v4d acc[2][3];
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
#pragma unroll
          for (int j = 0; j < 3; ++j) acc[cb][j] = v4d{0.0, 0.0, 0.0, 0.0};
        }
        double ml = 0.0;
        int gq = g;
        const double *ta = &TA[ay + 3 * az][0][0];
#pragma unroll
        for (int ks = 0; ks < 7; ++ks) {
          asm volatile("" : "+v"(gq), "+v"(ml));   // a k-step's operands in registers at a time
          const int qyz = ks < 6 ? (4 * ks + gq) * 11 >> 5 : 8;   // the point's index over y and z
          const double yz = ta[qyz], dz_ = ta[9 + qyz], zd = ta[18 + qyz];
          const double t = tn[ks];
          tn[ks] = pn[lane + 64 * ks];
          // rows 0-2: s C dN_a; row 3: w det, 0, 0, 1 with N_a first
          const double A = quad_entry<3>(t) * (quad_entry<0>(t) * (xd[ks % 3] * yz) + quad_entry<1>(t) * (xa[ks % 3] * dz_) +
                                               quad_entry<2>(t) * (xa[ks % 3] * zd));
          ml += A;
          const double C[9] = {row_entry<0>(t), row_entry<1>(t), row_entry<2>(t), row_entry<4>(t), row_entry<5>(t),
                               row_entry<6>(t), row_entry<8>(t), row_entry<9>(t), row_entry<10>(t)};
#pragma unroll
          for (int cb = 0; cb < 2; ++cb) {
            const double *tb = &TA[bo[cb][1] + 3 * bo[cb][2]][0][0];
            const double d[3] = {xbd[cb][ks % 3] * tb[qyz], xb[cb][ks % 3] * tb[9 + qyz], xb[cb][ks % 3] * tb[18 + qyz]};
            acc[cb][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(A, C[0] * d[0] + C[1] * d[1] + C[2] * d[2], acc[cb][0], 0, 0, 0);
            acc[cb][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(A, C[3] * d[0] + C[4] * d[1] + C[5] * d[2], acc[cb][1], 0, 0, 0);
            acc[cb][2] = __builtin_amdgcn_mfma_f64_16x16x4f64(A, C[6] * d[0] + C[7] * d[1] + C[8] * d[2], acc[cb][2], 0, 0, 0);
          }
        }
        msum += sg * ml;
        const double lam = sg * E * lamf, mu = sg * E * muf, rho = TR ? sg * p.rho : 0.0;
        // node a = g: 0 the current node, 1 the middle one, 2 the next; slots in dx, dy, dz
        double *dst = g == 0 ? cur + 2 * n9 : (g == 1 ? mid : nxt);
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
          const double trs = acc[cb][0][0] + acc[cb][1][1] + acc[cb][2][2];
          const double Mab = TR ? rho * Mb[cb] : 0.0;
          double jv[3][3];
          const bool in = 16 * cb + l16 < 27;
          const int bn = min(16 * cb + l16, 26);
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            double r = 0.0;
#pragma unroll
            for (int j = 0; j < 3; ++j) {
              const double Kv = lam * acc[cb][j][i] + mu * acc[cb][i][j] + (i == j ? mu * trs : 0.0);
              r += Kv * st[bn][j];
              jv[i][j] = cK * Kv;
              if (TR && i == j) {
                jv[i][j] += cM * Mab;
                r += Mab * st[bn][TR ? 3 + j : 0];
              }
            }
            rr[i] += in ? r : 0.0;
          }
          if (in && g < 3) {
            double *o = dst + bo[cb][0] * n9 + ((bo[cb][1] - ay + ry) * Dz + bo[cb][2] - az + rz) * 9;
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
              for (int j = 0; j < 3; ++j) atomicAdd(&o[3 * i + j], jv[i][j]);
          }
        }
      }
      // residuals: over the row of 16 lanes, less the source load (its sums are in lanes 12 + a, + 16 ...)
      double ms4 = msum;
      ms4 += __shfl_xor(ms4, 16);
      ms4 += __shfl_xor(ms4, 32);
      const double ma = __shfl(ms4, 12 + min(g, 2));
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        double r = rr[i];
        r += dpp_f64<0xB1, 0xf>(r);
        r += dpp_f64<0x4E, 0xf>(r);
        r += dpp_f64<0x141, 0xf>(r);
        r += dpp_f64<0x140, 0xf>(r);
        r = (carry[i] + r) - p.src[i] * ma;
        rr[i] = r;
        carry[i] = __shfl(r, (lane & 15) + 32);   // the next node's, for lanes of row 0
        if (g != 0) carry[i] = 0.0;
      }
      msum = 0.0;
      // everything loaded is here before the stores go out: one counter tracks loads and stores
#pragma unroll
      for (int ks = 0; ks < 7; ++ks) asm volatile("" : "+v"(tn[ks]));
#pragma unroll
      for (int j = 0; j < 3; ++j) asm volatile("" : "+v"(un[j]), "+v"(vn[j]), "+v"(an[j]));
      asm volatile("" : "+v"(Ln), "+v"(En), "+v"(nc0), "+v"(nc1), "+v"(nm0), "+v"(nm1));
      gather_lds_sync();
      if (x >= x0) {
        if (p.f && l16 < 3 && g < 2) p.f[(g ? Lm : Lc) + l16] = l16 == 0 ? rr[0] : (l16 == 1 ? rr[1] : rr[2]);
        store_node27(cur, inv, 2, ry, rz, nc0, nc1, p.vals, basec, lenc, lane);
        store_node27(mid, inv, 1, ry, rz, nm0, nm1, p.vals, basem, lenm, lane);
        gather_lds_sync();
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) rr[i] = 0.0;
      for (int k = lane; k < 3 * n9; k += 64) {
        cur[k] = nxt[k];
        nxt[k] = 0.0;
        mid[k] = 0.0;
      }
      for (int k = 3 * n9 + lane; k < 5 * n9; k += 64) cur[k] = 0.0;
      gather_lds_sync();
    }
    if (x1 == p.nx) {   // the line's last node has no cell above
      const int P0 = 2 * p.nx + px * (2 * LY + qy + py * (2 * LZ + qz));
      const int32_t Lc = plid[3 * P0];
      const int64_t basec = prow[Lc];
      const int lenc = static_cast<int>(prow[Lc + 1] - basec);
      const uint16_t *npc = p.nperm + static_cast<int64_t>(Lc / 3) * p.nperm_w;
      const int n0 = npc[lane], n1 = npc[lane + 64];
      if (p.f && l16 < 3 && g == 0) p.f[Lc + l16] = l16 == 0 ? carry[0] : (l16 == 1 ? carry[1] : carry[2]);
      store_node27(cur, inv, 2, ry, rz, n0, n1, p.vals, basec, lenc, lane);
      gather_lds_sync();
    }
  }
}

template <int NB, int NQ, int BS, int MODE>
void launch(const ElasticParams &p, hipStream_t s) {
  int dev = 0, ncu = 0;
  TXA_HIP(hipGetDevice(&dev));
  TXA_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  // grid-stride over elements with exactly the resident workgroups: a workgroup that
  // only starts when another ends would stretch the tail by its whole share
  int per_cu = 0;
  TXA_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_elastic<NB, NQ, BS, MODE>, BS, 0));
  const int64_t want = static_cast<int64_t>(ncu) * std::max(per_cu, 1);
  const unsigned grid = static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>(p.e1 - p.e0, want)));
  hipLaunchKernelGGL((k_elastic<NB, NQ, BS, MODE>), dim3(grid), dim3(BS), 0, s, p);
  TXA_HIP(hipGetLastError());
}

constexpr size_t kWsAlign = 256;

size_t ws_round(size_t b) { return (b + kWsAlign - 1) / kWsAlign * kWsAlign; }

// workspace bytes: residuals [E][ND] FP64 when f is wanted, blocks [E][ND][ND] when vals are
// affine HEX8 bricks take the node-centric kernel (no workspace) in every precision
bool affine_hex8(const Mesh &m) {
  return m.topo == TXA_HEX8 && m.affine && m.structured && m.nfields == 3;
}

// hex8 elasticity on general cells in FP64: the node kernels on bricks and on uploads whose
// rows fit them
bool general_hex8(const Mesh &m, int precision) {
  if (m.topo != TXA_HEX8 || m.nfields != 3 || precision != TXA_FP64) return false;
  return m.structured ? !m.affine : m.uocc.p != nullptr;   // three int32 LIDs per point: under 2^31 points
}

// hex27 bricks in FP64 take the line kernel where the matrix is wanted.  f alone keeps the element kernel
// and gather: its workspace (648 bytes per element, against the line kernel's 3456 of points) bounds the
// sizes that calls without allocation accept, and small calls are faster (6^3 35 us against 50, 33^3 1.20
// ms against 1.16 of the full call).  The two sum in different orders: f agrees to rounding, not bit for bit.
bool line_hex27(const Mesh &m, int precision, bool want_vals) {
  return m.topo == TXA_HEX27 && m.structured && m.nfields == 3 && precision == TXA_FP64 && want_vals;
}

// Streams and events of the element / gather slab pipeline, one set per host thread and device
// (a context is driven by one thread at a time; the events are recorded and waited on within
// one call, so calls in sequence may reuse them).  Created on first use; kept until the
// process ends.
constexpr int kSlabs = 8;
struct SlabPipe {
  hipStream_t e = nullptr, g = nullptr;
  hipEvent_t ev[kSlabs] = {}, ev0 = nullptr, evg = nullptr;
};

SlabPipe &slab_pipe(int dev) {
  thread_local std::map<int, SlabPipe> pipes;
  SlabPipe &sp = pipes[dev];
  if (!sp.e) {
    TXA_HIP(hipStreamCreateWithFlags(&sp.g, hipStreamNonBlocking));
    for (int k = 0; k < kSlabs; ++k) TXA_HIP(hipEventCreateWithFlags(&sp.ev[k], hipEventDisableTiming));
    TXA_HIP(hipEventCreateWithFlags(&sp.ev0, hipEventDisableTiming));
    TXA_HIP(hipEventCreateWithFlags(&sp.evg, hipEventDisableTiming));
    TXA_HIP(hipStreamCreateWithFlags(&sp.e, hipStreamNonBlocking));   // last: marks the set complete
  }
  return sp;
}

void ws_parts(const Mesh &m, int precision, bool want_f, bool want_vals, size_t *rbytes, size_t *jbytes) {
  const size_t nd = static_cast<size_t>(m.ndof_elem), ne = static_cast<size_t>(m.nelem);
  *rbytes = want_f ? ws_round(ne * nd * sizeof(double)) : 0;
  const size_t nb = nd / 3;
  *jbytes = want_vals ? ws_round(ne * nb * static_cast<size_t>(block_stride(static_cast<int>(nb))) *
                                 (precision == TXA_FP64 ? sizeof(double) : sizeof(float)))
                      : 0;
}

}  // namespace

bool elastic_supported(const Mesh &m, const txa_assembly_args &a) {
  if (a.physics != TXA_ELASTICITY || m.nfields != 3 || !(m.nperm.p || m.uocc.p)) return false;
  if (m.topo == TXA_HEX8) return a.precision == TXA_FP64 || a.precision == TXA_FP32;
  return m.topo == TXA_HEX27;
}

size_t elastic_workspace_bytes(const Mesh &m, int precision, bool want_f, bool want_vals, bool footprint) {
  size_t r = 0, j = 0;
  if (affine_hex8(m) || (!footprint && general_hex8(m, precision))) return 0;
  if (!footprint && line_hex27(m, precision, want_vals)) return ws_round(static_cast<size_t>(m.nelem) * 27 * 16 * sizeof(double) + 16 * sizeof(double));
  ws_parts(m, precision, want_f, want_vals, &r, &j);
  return r + j;
}

void node_perm_build(Mesh &m, hipStream_t s) {
  m.cell_geom.release();
  m.uocc_ptr.release();
  m.uocc.release();
  m.uslot.release();
  if (!m.structured && m.nfields == 3 && m.blocks.size() == 1 && (m.topo == TXA_HEX8 || m.topo == TXA_HEX27)) {
    // uploaded mesh: element instances of each node and their slot maps, for the general gather
    const int nb = m.nconn;
    const int64_t nnodes = m.ndofs / 3, npos0 = m.nelem * nb;
    if (npos0 >= (int64_t(1) << 31)) return;
    DevBuf<unsigned long long> cnt;
    cnt.alloc(nnodes + 1);
    TXA_HIP(hipMemsetAsync(cnt.p, 0, cnt.bytes(), s));
    const unsigned gp = static_cast<unsigned>((npos0 + 255) / 256), gn = static_cast<unsigned>((nnodes + 255) / 256);
    hipLaunchKernelGGL(k_uocc_count, dim3(gp), dim3(256), 0, s, npos0, nb, m.elem_lid.p, cnt.p);
    TXA_HIP(hipGetLastError());
    m.uocc_ptr.alloc(nnodes + 1);
    exclusive_scan_i64(reinterpret_cast<const int64_t *>(cnt.p), m.uocc_ptr.p, nnodes + 1, s);
    TXA_HIP(hipMemcpyAsync(cnt.p, m.uocc_ptr.p, sizeof(int64_t) * (nnodes + 1), hipMemcpyDeviceToDevice, s));
    m.uocc.alloc(npos0);
    hipLaunchKernelGGL(k_uocc_fill, dim3(gp), dim3(256), 0, s, npos0, nb, m.elem_lid.p, cnt.p, m.uocc.p);
    TXA_HIP(hipGetLastError());
    m.uslot.alloc(npos0 * nb);
    DevBuf<int> mx;
    mx.alloc(2);
    TXA_HIP(hipMemsetAsync(mx.p, 0, 2 * sizeof(int), s));
    hipLaunchKernelGGL(k_uocc_finish, dim3(gn), dim3(256), 0, s, nnodes, nb, m.uocc_ptr.p, m.uocc.p, m.elem_lid.p,
                       m.rowptr.p, m.col.p, m.uslot.p, mx.p);
    TXA_HIP(hipGetLastError());
    int h[2];
    TXA_HIP(hipMemcpyAsync(h, mx.p, sizeof(h), hipMemcpyDeviceToHost, s));
    TXA_HIP(hipStreamSynchronize(s));
    const int S = nb == 8 ? 3 : 5;
    if (h[0] > 3 * S * S * S) {   // a row longer than the gather's LDS rows: the generic kernel
      m.uocc_ptr.release();
      m.uocc.release();
      m.uslot.release();
    }
    return;
  }
  if (!m.structured || m.nfields != 3 || (m.topo != TXA_HEX8 && m.topo != TXA_HEX27)) return;
  const int R = m.topo == TXA_HEX8 ? 1 : 2;
  const int64_t px = m.topo == TXA_HEX8 ? m.nx + 1 : 2 * static_cast<int64_t>(m.nx) + 1;
  const int64_t py = m.topo == TXA_HEX8 ? m.ny + 1 : 2 * static_cast<int64_t>(m.ny) + 1;
  const int64_t pz = m.topo == TXA_HEX8 ? m.nz + 1 : 2 * static_cast<int64_t>(m.nz) + 1;
  TXA_REQUIRE(px * py * pz == m.npoints, TXA_ERR_LOGIC, "lattice size mismatch");
  m.nperm_w = R == 1 ? 32 : 128;
  m.nperm.alloc(static_cast<size_t>(m.npoints) * m.nperm_w);
  const int64_t nt = m.npoints;
  hipLaunchKernelGGL(k_node_perm, dim3(static_cast<unsigned>((nt + 255) / 256)), dim3(256), 0, s, px, py, pz, R,
                     m.nfields, m.nperm_w, m.point_lid.p, m.rowptr.p, m.col.p, m.nperm.p);
  TXA_HIP(hipGetLastError());
  if (affine_hex8(m)) {
    const int64_t nc = static_cast<int64_t>(m.nx) * m.ny * m.nz;
    m.cell_geom.alloc(static_cast<size_t>(nc) * 10);
    hipLaunchKernelGGL(k_cell_geom, dim3(static_cast<unsigned>((nc + 255) / 256)), dim3(256), 0, s, m.nx, m.ny, m.nz,
                       m.nverts, m.xyz.p, m.cell_geom.p);
    TXA_HIP(hipGetLastError());
  }
}

namespace {

Elastic8Params elastic8_params(const Mesh &m, const txa_assembly_args &a) {
  Elastic8Params q;
  q.nx = m.nx; q.ny = m.ny; q.nz = m.nz;
  q.npoints = m.npoints;
  q.point_lid = m.point_lid.p;
  q.rowptr = m.rowptr.p;
  q.nperm = m.nperm.p;
  q.nperm_w = m.nperm_w;
  q.geom = m.cell_geom.p;
  q.coef = a.coef;
  q.nu = a.nu; q.rho = a.rho;
  q.src[0] = a.src[0]; q.src[1] = a.src[1]; q.src[2] = a.src[2];
  q.ra = a.rayleigh_a; q.rb = a.rayleigh_b;
  q.x = a.x; q.xdot = a.xdot; q.xddot = a.xddot;
  q.alpha = a.alpha; q.beta = a.beta; q.gamma2 = a.gamma2;
  q.transient = a.transient;
  q.f = a.f; q.vals = a.vals;
  return q;
}

// tiles of the hex8 node kernels on a brick
int64_t tiles8(const Mesh &m) {
  return static_cast<int64_t>((m.nx + kN8) / kN8) * ((m.ny + kN8) / kN8) * (m.nz + 1);
}

// workgroups for a grid-stride kernel: the resident ones, or as many as there are items
template <class Kernel>
unsigned resident_grid(Kernel k, int64_t items, int threads = 256) {
  int dev = 0, ncu = 0, per_cu = 0;
  TXA_HIP(hipGetDevice(&dev));
  TXA_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  TXA_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, threads, 0));
  const int64_t want = static_cast<int64_t>(ncu) * std::max(per_cu, 1);
  return static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>(items, want)));
}

}  // namespace

void launch_elastic(Mesh &m, const txa_assembly_args &a, hipStream_t s, void *ws) {
  if (!a.f && !a.vals) return;
  if (affine_hex8(m)) {
    TXA_REQUIRE(m.cell_geom.p != nullptr, TXA_ERR_LOGIC, "cell geometry missing (graph_build)");
    const Elastic8Params q = elastic8_params(m, a);
    const int64_t groups = (static_cast<int64_t>((m.nx + kN8) / kN8) * (m.ny + 1) * (m.nz + 1) + 3) / 4;   // four lines each
    if (a.transient && a.xdot)
      hipLaunchKernelGGL(k_elastic8_affine<true>, dim3(resident_grid(k_elastic8_affine<true>, groups)), dim3(256), 0, s, q);
    else
      hipLaunchKernelGGL(k_elastic8_affine<false>, dim3(resident_grid(k_elastic8_affine<false>, groups)), dim3(256), 0, s, q);
    TXA_HIP(hipGetLastError());
    return;
  }
  if (general_hex8(m, a.precision) && m.structured) {
    Elastic8GParams q;
    q.p = elastic8_params(m, a);
    q.X = m.xyz.p; q.Y = m.xyz.p + m.nverts; q.Z = m.xyz.p + 2 * m.nverts;
    const int64_t tiles = tiles8(m);
    if (a.transient && a.xdot)
      hipLaunchKernelGGL(k_elastic8_general<true>, dim3(resident_grid(k_elastic8_general<true>, tiles)), dim3(256), 0, s, q);
    else
      hipLaunchKernelGGL(k_elastic8_general<false>, dim3(resident_grid(k_elastic8_general<false>, tiles)), dim3(256), 0, s, q);
    TXA_HIP(hipGetLastError());
    return;
  }
  if (general_hex8(m, a.precision)) {
    Elastic8UParams q;
    q.p = elastic8_params(m, a);
    q.X = m.xyz.p; q.Y = m.xyz.p + m.nverts; q.Z = m.xyz.p + 2 * m.nverts;
    q.nnodes = m.ndofs / 3;
    q.conn = m.conn.p; q.elem_lid = m.elem_lid.p;
    q.occ_ptr = m.uocc_ptr.p; q.occ = m.uocc.p; q.slot = m.uslot.p;
    const int64_t pairs = (q.nnodes + 1) / 2;
    if (a.transient && a.xdot)
      hipLaunchKernelGGL(k_elastic8_upload<true>, dim3(resident_grid(k_elastic8_upload<true>, pairs, 64)), dim3(64), 0, s, q);
    else
      hipLaunchKernelGGL(k_elastic8_upload<false>, dim3(resident_grid(k_elastic8_upload<false>, pairs, 64)), dim3(64), 0, s, q);
    TXA_HIP(hipGetLastError());
    return;
  }
  if (line_hex27(m, a.precision, a.vals != nullptr)) {
    TXA_REQUIRE(ws != nullptr, TXA_ERR_LOGIC, "elasticity assembly needs its workspace");
    Node27Params q;
    q.p = elastic8_params(m, a);
    q.pts = static_cast<const double *>(ws);
    const int64_t lines = static_cast<int64_t>(m.ny + 1) * (m.nz + 1);
    const bool tr = a.transient && a.xdot;
    // x positions per workgroup: the mean load of a wave (nine units per position and line, one more
    // position per part of a split line) and half of the longest workgroup, which may start last.
    // Measured with 1, 2, 3, 4, 6 parts: 6^3 109, 80, 66, 66, 52 us (six chosen), 10^3 173, 115, 103, 93, 93
    // (ten: 102), 24^3 571, 515, 508, 522, 548 (four), 33^3 1215, 1159, 1165, 1299, 1285 us (three).
    const double slots = tr ? resident_grid(k_elastic27_nodes<true>, INT32_MAX, 64) : resident_grid(k_elastic27_nodes<false>, INT32_MAX, 64);
    double best = 1e300;
    q.chunk = m.nx;
    for (int k = 1; k <= m.nx && k <= 32; ++k) {
      const int len = (m.nx + k - 1) / k, n = (m.nx + len - 1) / len, extra = n > 1;
      const double t = std::max(1.0, 9.0 * lines * n / (4.0 * slots)) * 4.0 * (static_cast<double>(m.nx) / n + extra) + 2.0 * (len + extra);
      if (t < best) { best = t; q.chunk = len; }
    }
    q.nchunk = (m.nx + q.chunk - 1) / q.chunk;
    const int64_t np = m.nelem * 27;
    hipLaunchKernelGGL(k_points27, dim3(static_cast<unsigned>((np + 255) / 256)), dim3(256), 0, s, m.nx, m.ny, m.nelem, m.xyz.p,
                       m.xyz.p + m.nverts, m.xyz.p + 2 * m.nverts, static_cast<double *>(ws));
    TXA_HIP(hipGetLastError());
    const dim3 grid(static_cast<unsigned>(3 * lines * q.nchunk));
    if (tr) hipLaunchKernelGGL(k_elastic27_nodes<true>, grid, dim3(64), 0, s, q);
    else hipLaunchKernelGGL(k_elastic27_nodes<false>, grid, dim3(64), 0, s, q);
    TXA_HIP(hipGetLastError());
    return;
  }
  size_t rbytes = 0, jbytes = 0;
  ws_parts(m, a.precision, a.f != nullptr, a.vals != nullptr, &rbytes, &jbytes);
  char *w = static_cast<char *>(ws);
  TXA_REQUIRE(w != nullptr, TXA_ERR_LOGIC, "elasticity assembly needs its workspace");
  ElasticParams p;
  p.nq = m.topo == TXA_HEX8 ? 8 : 27;
  p.nelem = m.nelem;
  p.e0 = 0;
  p.e1 = m.nelem;
  p.nconn = m.nconn;
  p.conn = m.conn.p;
  p.X = m.xyz.p; p.Y = m.xyz.p + m.nverts; p.Z = m.xyz.p + 2 * m.nverts;
  p.elem_lid = m.elem_lid.p;
  p.coef = a.coef;
  p.nu = a.nu; p.rho = a.rho;
  p.src[0] = a.src[0]; p.src[1] = a.src[1]; p.src[2] = a.src[2];
  p.ra = a.rayleigh_a; p.rb = a.rayleigh_b;
  p.x = a.x; p.xdot = a.xdot; p.xddot = a.xddot;
  p.alpha = a.alpha; p.beta = a.beta; p.gamma2 = a.gamma2;
  p.transient = a.transient;
  p.rbuf = rbytes ? reinterpret_cast<double *>(w) : nullptr;
  p.jbuf = jbytes ? static_cast<void *>(w + rbytes) : nullptr;
  auto elem_launch = [&](const ElasticParams &pp, hipStream_t st) {
    if (m.topo == TXA_HEX8) {
      launch<8, 8, 64, MODE_F32>(pp, st);   // FP64: the node kernels
    } else {
      if (a.precision == TXA_SPLIT_BF16) launch<27, 27, 256, MODE_SPLIT>(pp, st);
      else if (a.precision == TXA_FP32) launch<27, 27, 256, MODE_F32>(pp, st);
      else launch<27, 27, 256, MODE_F64>(pp, st);
    }
  };
  if (!m.structured) elem_launch(p, s);   // bricks: element slabs interleaved with the gather below
  int dev = 0, ncu = 0;
  TXA_HIP(hipGetDevice(&dev));
  TXA_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  const bool wide = a.precision == TXA_FP64;
  if (!m.structured) {
    GatherUParams u;
    u.nnodes = m.ndofs / 3;
    u.occ_ptr = m.uocc_ptr.p;
    u.occ = m.uocc.p;
    u.slot = m.uslot.p;
    u.rowptr = m.rowptr.p;
    u.jbuf = p.jbuf;
    u.rbuf = p.rbuf;
    u.f = a.f;
    u.vals = a.vals;
    const unsigned ug = static_cast<unsigned>(std::min<int64_t>((u.nnodes + 3) / 4, static_cast<int64_t>(ncu) * 16));
    if (m.topo == TXA_HEX8) {
      hipLaunchKernelGGL((k_elastic_gather_u<8, float>), dim3(ug), dim3(256), 0, s, u);
    } else {
      if (wide) hipLaunchKernelGGL((k_elastic_gather_u<27, double>), dim3(ug), dim3(256), 0, s, u);
      else hipLaunchKernelGGL((k_elastic_gather_u<27, float>), dim3(ug), dim3(256), 0, s, u);
    }
    TXA_HIP(hipGetLastError());
    return;
  }
  GatherParams g;
  g.nx = m.nx; g.ny = m.ny; g.nz = m.nz;
  const int64_t st = m.topo == TXA_HEX8 ? 1 : 2;
  g.px = st * m.nx + 1; g.py = st * m.ny + 1; g.pz = st * m.nz + 1;
  g.npoints = m.npoints;
  g.p0 = 0;
  g.p1 = m.npoints;
  g.point_lid = m.point_lid.p;
  g.rowptr = m.rowptr.p;
  g.nperm = m.nperm.p;
  g.nperm_w = m.nperm_w;
  g.jbuf = p.jbuf;
  g.rbuf = p.rbuf;
  g.f = a.f;
  g.vals = a.vals;
  auto gather_launch = [&](const GatherParams &gg, hipStream_t st) {
    const unsigned grid = static_cast<unsigned>(std::min<int64_t>((gg.p1 - gg.p0 + 3) / 4, static_cast<int64_t>(ncu) * 16));
    if (m.topo == TXA_HEX8) {
      hipLaunchKernelGGL((k_elastic_gather<8, float>), dim3(grid), dim3(256), 0, st, gg);
    } else {
      if (wide) hipLaunchKernelGGL((k_elastic_gather<27, double>), dim3(grid), dim3(256), 0, st, gg);
      else hipLaunchKernelGGL((k_elastic_gather<27, float>), dim3(grid), dim3(256), 0, st, gg);
    }
    TXA_HIP(hipGetLastError());
  };
  // Slab pipeline: the elements in z slabs on one stream, the gather of each slab's node planes
  // on another once that slab (and the one below) is done, so the element kernel (bound by
  // its per-element latency and VALU) of slab k+1 runs beside the gather (bound by HBM) of
  // slab k.  Node plane st*z1 at a slab's top needs the next slab: the next gather takes it.
  // A stream under graph capture (or a brick of one slab) takes the two kernels in order
  // on that stream: no streams or events are created inside a capture.
  // A slab below some 24,000 elements costs more in launches, events and emptied CUs than the overlap
  // gives (hex27 split, one slab against eight: 8^3 48 and 174 us, 20^3 273 and 366, 36^3 1374 and 1459;
  // four against one and eight: 46^3 2801, 2848 and 2865 us; eight against four: 64^3 7.40 and 7.48 ms;
  // hex8 FP32 on general cells, against eight: 32^3 in one 121 and 250 us, 48^3 in four 397 and 443).
  const int nslab = std::min({kSlabs, m.nz, static_cast<int>(std::min<int64_t>(m.nelem / 24000, kSlabs))});
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  TXA_HIP(hipStreamIsCapturing(s, &cs));
  if (cs != hipStreamCaptureStatusNone || nslab < 2) {
    elem_launch(p, s);
    gather_launch(g, s);
    return;
  }
  SlabPipe &sp = slab_pipe(dev);
  const int64_t layer = static_cast<int64_t>(m.nx) * m.ny, pxy = g.px * g.py;
  TXA_HIP(hipEventRecord(sp.ev0, s));
  TXA_HIP(hipStreamWaitEvent(sp.e, sp.ev0, 0));
  TXA_HIP(hipStreamWaitEvent(sp.g, sp.ev0, 0));
  for (int k = 0; k < nslab; ++k) {
    const int64_t z0 = static_cast<int64_t>(m.nz) * k / nslab, z1 = static_cast<int64_t>(m.nz) * (k + 1) / nslab;
    ElasticParams pk = p;
    pk.e0 = z0 * layer;
    pk.e1 = z1 * layer;
    elem_launch(pk, sp.e);
    TXA_HIP(hipEventRecord(sp.ev[k], sp.e));
    TXA_HIP(hipStreamWaitEvent(sp.g, sp.ev[k], 0));
    GatherParams gk = g;
    gk.p0 = st * z0 * pxy;
    gk.p1 = k == nslab - 1 ? m.npoints : st * z1 * pxy;
    gather_launch(gk, sp.g);
  }
  TXA_HIP(hipEventRecord(sp.evg, sp.g));
  TXA_HIP(hipStreamWaitEvent(s, sp.evg, 0));
}

}  // namespace txa
