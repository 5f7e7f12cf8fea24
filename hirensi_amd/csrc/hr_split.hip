// Split stage path: the RK4 stages of the elastic system with the hybrid
// displacement-stress PML (Solver_PETSc_Explicit.F90:1001-1046 forward,
// :1319-1364 adjoint), the PML nodes by nodal kernels and the regular domain by
// an element kernel.
//
// The operator is linear and fixed, so the four stages are taken as successive
// time derivatives: with L(v1, v2, v3) = -M^-1 (G v1 + K v2 + C v3) (adjoint:
// the transposes with the signs of the adjoint system),
//   a1 = L(x1, x2, x3) + s1,  a2 = L(x2, x3, a1) + s2,
//   a3 = L(x3, a1, a2),       a4 = L(a1, a2, a3) + s4,
//   x1 += h x2 + h^2/2 x3 + h^3/6 a1 + h^4/24 a2        (x2, x3 likewise, from one
//   component later), s1 = f0, s2 = 2 (fm - f0) / h, s4 = 4 (f0 - 2 fm + f1) / h^3
// for the source at the start, middle and end of the step (s4 goes into x3 alone, as
// h times (f0 - 2 fm + f1) / 6: neither 1 / h^3 nor h^4 is formed for it).  Expanding the
// classical k1..k4 in powers of the operator gives the same polynomial in h, source
// terms included, so the step is the reference's RK4 up to rounding; but a stage
// reads three vectors instead of 3, 4, 5 and 6, and the last one the state
// besides.  K acts on v2 alone, and at regular-domain nodes nothing else does:
// their a1 and a2 need x2 and x3 only and one pass forms both, a second one a3, a4
// and the update, which leaves two element passes a step instead of four.
// Against the stages on k1..k4 with four element passes (forward and adjoint, one
// MI355X): 64x64x32 elements, PML 6: 0.68 -> 0.56 ms per step; 37x29x19: 0.31 -> 0.16;
// 16x16x8: 0.23 -> 0.09; with the passes as below 0.49, 0.118 and 0.061.

#include <hip/hip_runtime.h>
#include "hr_gradient.h"
#include "hr_lattice.h"
#include "hr_split.h"

// Fused multiply-add is allowed here, as in the fused stage kernel.
#pragma clang fp contract(fast)

namespace hr {
namespace {

// Blocks of consecutive PML nodes in lattice order (sp_pml_node), one node per thread:
// SPLIT_OWN nodes and two on each side.  XCD x = blockIdx % 8 takes the logical
// blocks [x C, (x + 1) C) of the launch, so that each XCD's L2 holds a contiguous run of
// the list (the neighbouring rows and planes of its nodes); a launch has 8 C blocks.
__device__ __forceinline__ int split_block(int blk, int nblk) {
  const int C = (nblk + 7) / 8;
  return (blk & 7) * C + (blk >> 3);
}
// Flux records D of the split path, per shot 12 NN doubles: two arrays (ax =
// y, z) of six doubles per lattice node, (G_{x,ax}, G_{y,ax}, G_{z,ax},
// w_{ax,x}, w_{ax,y}, w_{ax,z}) with G_{i,ax} the nodal PML flux and w_{ax,i}
// the F-weighted inputs: a line along ax reads three 16-byte pairs per node.
// The x-lines are summed by the nodal pass itself, from LDS.
__device__ __forceinline__ unsigned d_rec(int ax, unsigned NN, unsigned n) {
  return 48u * ((unsigned)(ax - 1) * NN + n);
}

// Operator inputs of one component: as stored, with the adjoint's signs on v1, v3
template <bool TR>
__device__ __forceinline__ void operator_inputs(const double* X, double& v1, double& v2, double& v3) {
  v1 = TR ? -X[0] : X[0];
  v2 = X[1];
  v3 = TR ? -X[2] : X[2];
}

// A thread's list entry.  Block lb owns [lb SPLIT_OWN, (lb + 1) SPLIT_OWN) and computes
// two entries more on each side, for their x records; a thread without an
// entry runs node 0 (in bounds) and stores nothing.
struct Entry {
  int i, j, k;
  bool valid, own;
  unsigned n;
};
__device__ __forceinline__ Entry list_entry(const Geo3& g, int lb) {
  Entry E;
  const int tid = threadIdx.x;
  const long long t = (long long)lb * SPLIT_OWN - 2 + tid;
  E.i = E.j = E.k = 0;
  E.valid = t >= 0 && sp_pml_node((unsigned)t, g.NX, g.NY, g.NZ, g.rlo, g.rhi, E.i, E.j, E.k);
  if (!E.valid) E.i = E.j = E.k = 0;
  E.own = E.valid && tid >= 2 && tid < SPLIT_NT - 2;
  E.n = (unsigned)E.i + (unsigned)g.NX * ((unsigned)E.j + (unsigned)g.NY * (unsigned)E.k);
  return E;
}

// place of a column's interface nodes in the regular-domain sums, and the step per plane
__device__ __forceinline__ unsigned iface_column(const Geo3& g, int i, int j) {
  return sp_iface_column(i - 2 * g.rlo[0], j - 2 * g.rlo[1], 2 * (g.rhi[0] - g.rlo[0]) + 1, 2 * (g.rhi[1] - g.rlo[1]) + 1,
                         g.NZ - 2 * g.rlo[2]);
}
__device__ __forceinline__ unsigned iface_rim(const Geo3& g) {
  return sp_rim(2 * (g.rhi[0] - g.rlo[0]) + 1, 2 * (g.rhi[1] - g.rlo[1]) + 1);
}

struct NodalLds {
  double xr[6][SPLIT_NT];         // x flux records of the block's entries
  unsigned xn[SPLIT_NT];          // their lattice nodes (~0: no entry)
};

// one vector's components at a node
__device__ __forceinline__ void ld_node(const double* ip, unsigned offu, unsigned offs, double* v) {
  ld3(ip, offu, v[0], v[1], v[2]);
  ld2(ip, offs, v[3], v[4]);
  ld2(ip, offs + 16u, v[5], v[6]);
  ld2(ip, offs + 32u, v[7], v[8]);
}
// and its active components back
__device__ __forceinline__ void st_node(double* dst, unsigned offu, unsigned offs, bool ua, int sm, const double* v) {
  if (ua) st3(dst, offu, v[0], v[1], v[2]);
  if (sm == 0x3f) st6(dst, offs, &v[3]);
  else {
    if (sm & 7) st3m(dst, offs, sm & 7, v[3], v[4], v[5]);
    if (sm & 56) st3m(dst, offs + 24u, (sm >> 3) & 7, v[6], v[7], v[8]);
  }
}

// Node-local part of an RK4 stage at one PML node: the flux records of its y-
// and z-lines, and into the stage output the node-local terms -M^-1 (diagonal
// terms + x-line sums).  LAST: the output is the new x3 (scaled by h^4/24, on the
// part of the update that does not need a4), and the new x1, x2 are written here.
// The x-line sums read the x records of the block's entries from LDS:
// consecutive list entries are x-neighbours.  V[q]: the components of v1, v2, v3
// and, LAST, x1, x2, x3.  RAW: an operator product, the plain sums with unit signs.
template <bool LAST, bool TR, bool RAW = false>
__device__ __forceinline__ void nodal_pass(const SplitArgs& A, const Entry& E, int shot,
                                           const double (*V)[9], NodalLds& sh) {
  constexpr int NIN = LAST ? 6 : 3;
  double(&sXr)[6][SPLIT_NT] = sh.xr;
  unsigned(&sXn)[SPLIT_NT] = sh.xn;
  const Geo3& g = A.g;
  const int tid = threadIdx.x;
  const int i = E.i, j = E.j, k = E.k;
  const bool valid = E.valid, own = E.own;
  const unsigned n = E.n;
  const long long so = (long long)shot * A.shot_stride;
  const unsigned NN = (unsigned)g.NN;
  const unsigned SB = 8u * (3u * NN + (NN & 1u));
  const unsigned offu = n * 24u, offs = SB + n * 48u;
  const double* __restrict__ tab = A.tab;
  const double* __restrict__ nodet = A.node;

  double XU[3][NIN], XS6[6][NIN];
#pragma unroll
  for (int q = 0; q < NIN; ++q) {
#pragma unroll
    for (int c = 0; c < 3; ++c) XU[c][q] = V[q][c];
#pragma unroll
    for (int m = 0; m < 6; ++m) XS6[m][q] = V[q][3 + m];
  }
  double lam, mu, ax, bx, ay, by, az, bz;
  ld2(nodet, n * 16u, lam, mu);
  const double minv_u = A.minvu[n], rwp = A.rwp[n];
  ld2(tab, 8u * (unsigned)(TAB_STRETCH + 2 * i), ax, bx);
  ld2(tab, 8u * (unsigned)(TAB_STRETCH + 2 * g.NX + 2 * j), ay, by);
  ld2(tab, 8u * (unsigned)(TAB_STRETCH + 2 * g.NX + 2 * g.NY + 2 * k), az, bz);
  // the node's sides per axis; its PML weight sum and the stress rows' M^-1
  const SpAxis AX = sp_axis(i, g.nex, g.rlo[0], g.rhi[0]), AY = sp_axis(j, g.ney, g.rlo[1], g.rhi[1]),
               AZ = sp_axis(k, g.nez, g.rlo[2], g.nez);
  const double wps = g.detj * sp_pml_weight(AX, AY, AZ);
  const double minv_s = 1.0 / (((ax * ay) * az) * wps);
  const bool ua = u_act3(g, i, j, k);
  const int sm = smask3(g, i, j, k);

  double v1u[3], vu2[3], v3u[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) operator_inputs<TR && !RAW>(XU[c], v1u[c], vu2[c], v3u[c]);
  // F[set][k], set 0 = w (G, v1), 1 = p (K, v2), 2 = e (C, v3)
  double F[3][3];
  F[2][0] = ay * az; F[2][1] = ax * az; F[2][2] = ax * ay;
  F[1][0] = ay * bz + az * by; F[1][1] = ax * bz + az * bx; F[1][2] = ax * by + ay * bx;
  F[0][0] = by * bz; F[0][1] = bx * bz; F[0][2] = bx * by;
  double wv[9];
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int c = 0; c < 3; ++c) wv[3 * d + c] = ((0.0 + F[0][d] * v1u[c]) + F[1][d] * vu2[c]) + F[2][d] * v3u[c];
  // diagonal terms rho W (b v3 + c v2 + d v1) of ELEMENT_EM/EN (PML.F90 items 7..10)
  const double qb = ax * ay * bz + ax * az * by + ay * az * bx;
  const double qc = ax * by * bz + ay * bx * bz + az * bx * by;
  const double qd = bx * by * bz;
  auto diag = [&](double wm, double a1, double a2, double a3) { return wm * (((0.0 + qb * a3) + qc * a2) + qd * a1); };
  double dg[9], c3[9], Gv[9];
#pragma unroll
  for (int m = 0; m < 9; ++m) { c3[m] = 0.0; Gv[m] = 0.0; }
#pragma unroll
  for (int c = 0; c < 3; ++c) dg[c] = diag(rwp, v1u[c], vu2[c], v3u[c]);
  if constexpr (LAST) {
    double xn0[3], xn1[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) rk4_update(XU[c], A.h, A.h2, A.h3, A.h4, xn0[c], xn1[c], c3[c]);
    if (own && ua) {
      st3(A.xn[0] + so, offu, xn0[0], xn0[1], xn0[2]);
      st3(A.xn[1] + so, offu, xn1[0], xn1[1], xn1[2]);
    }
  }
  const double l2m = lam + 2.0 * mu, m2 = 2.0 * mu;
#pragma unroll
  for (int hf = 0; hf < 2; ++hf) {
    const double(*XS)[NIN] = &XS6[3 * hf];
    double s1[3], s2[3], s3[3];
#pragma unroll
    for (int tt = 0; tt < 3; ++tt) operator_inputs<TR && !RAW>(XS[tt], s1[tt], s2[tt], s3[tt]);
#pragma unroll
    for (int X = 0; X < 3; ++X) {
      const double* sv = X == 0 ? s1 : (X == 1 ? s2 : s3);
      if (hf == 0) {
        if constexpr (!TR) {
          // T(s): stress of the auxiliary strain (ELEMENT_EA_3D lower block), normal part
          const double Txx = l2m * sv[0] + lam * sv[1] + lam * sv[2];
          const double Tyy = lam * sv[0] + l2m * sv[1] + lam * sv[2];
          const double Tzz = lam * sv[0] + lam * sv[1] + l2m * sv[2];
          Gv[0] -= F[X][0] * Txx; Gv[4] -= F[X][1] * Tyy; Gv[8] -= F[X][2] * Tzz;
        } else {
          Gv[0] += F[X][0] * sv[0]; Gv[4] += F[X][1] * sv[1]; Gv[8] += F[X][2] * sv[2];
        }
      } else {
        if constexpr (!TR) {
          const double Txy = m2 * sv[0], Txz = m2 * sv[1], Tyz = m2 * sv[2];
          Gv[1] -= F[X][1] * Txy; Gv[2] -= F[X][2] * Txz; Gv[3] -= F[X][0] * Txy;
          Gv[5] -= F[X][2] * Tyz; Gv[6] -= F[X][0] * Txz; Gv[7] -= F[X][1] * Tyz;
        } else {
          Gv[1] += F[X][1] * sv[0]; Gv[2] += F[X][2] * sv[1]; Gv[3] += F[X][0] * sv[0];
          Gv[5] += F[X][2] * sv[2]; Gv[6] += F[X][0] * sv[1]; Gv[7] += F[X][1] * sv[2];
        }
      }
    }
    const double wm = hf == 0 ? wps : 2.0 * wps;
#pragma unroll
    for (int tt = 0; tt < 3; ++tt) dg[3 + 3 * hf + tt] = diag(wm, s1[tt], s2[tt], s3[tt]);
    if constexpr (LAST) {
      double xn0[3], xn1[3];
#pragma unroll
      for (int tt = 0; tt < 3; ++tt) rk4_update(XS[tt], A.h, A.h2, A.h3, A.h4, xn0[tt], xn1[tt], c3[3 + 3 * hf + tt]);
      const int act = own ? (sm >> (3 * hf)) & 7 : 0;
      if (act) {
        st3m(A.xn[0] + so, offs + 24u * hf, act, xn0[0], xn0[1], xn0[2]);
        st3m(A.xn[1] + so, offs + 24u * hf, act, xn1[0], xn1[1], xn1[2]);
      }
    }
  }
  // node-local terms of the stage output, without the x-line sums
  const double sc = LAST ? A.h4 : 1.0;
  double pre[9];
#pragma unroll
  for (int m = 0; m < 9; ++m) {
    const double minv = RAW ? -1.0 : (m < 3 ? minv_u : (m < 6 ? minv_s : 0.5 * minv_s));
    pre[m] = c3[m] - sc * (minv * dg[m]);
  }
  // x records to LDS; y and z records to memory
  sXn[tid] = valid ? n : ~0u;
  sXr[0][tid] = Gv[0]; sXr[1][tid] = Gv[3]; sXr[2][tid] = Gv[6];
  sXr[3][tid] = wv[0]; sXr[4][tid] = wv[1]; sXr[5][tid] = wv[2];
  // flux records: (G_{x,ax}, G_{y,ax}, G_{z,ax}, w_{ax,x}, w_{ax,y}, w_{ax,z}), Gv[3 i + ax], wv[3 ax + i]
  double* const Dp = A.D + (long long)shot * 12 * g.NN;
  if (own) {
#pragma unroll
    for (int a = 1; a < 3; ++a) {
      const unsigned o = d_rec(a, NN, n);
      st2(Dp, o, Gv[a], Gv[3 + a]);
      st2(Dp, o + 16u, Gv[6 + a], wv[3 * a]);
      st2(Dp, o + 32u, wv[3 * a + 1], wv[3 * a + 2]);
    }
  }
  __syncthreads();
  if (!own) return;
  // the x-line of the pull: side-scaled stencil over the x-neighbours' records.
  // The neighbour at lattice offset di (|di| <= 2) is at most |di| entries away
  // in the list (no PML node between, or one); one that is not a PML node (a
  // regular-domain node) has no record; offsets outside the lattice, and of an element that
  // does not hold the node, have zero coefficients and are not read, so that a
  // non-finite value reaches the nodes that share a PML element with it only.
  double cs0, cs1, cu[5];
  sp_side_scales(AX, AY, AZ, cs0, cs1);
  sp_stencil(AX.odd, cs0, cs1, cu);
  double sux[3] = {0.0, 0.0, 0.0}, sdx[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int d = 0; d < 5; ++d) {
    const int di = d - 2;
    int slot = -1;
    if (di == 0) {
      slot = tid;
    } else if (cu[d] != 0.0) {
      const unsigned ne = (unsigned)((int)n + di);
      const int near = tid + (di > 0 ? 1 : -1);
      if (di == 2 || di == -2) slot = sXn[tid + di] == ne ? tid + di : (sXn[near] == ne ? near : -1);
      else slot = sXn[near] == ne ? near : -1;
    }
    // u rows with cu, s rows with every offset but 0 negated
    const double cw = d == 2 ? cu[d] : -cu[d];
    if (slot >= 0) {
      sux[0] += cu[d] * sXr[0][slot]; sux[1] += cu[d] * sXr[1][slot]; sux[2] += cu[d] * sXr[2][slot];
      sdx[0] += cw * sXr[3][slot]; sdx[1] += cw * sXr[4][slot]; sdx[2] += cw * sXr[5][slot];
    }
  }
  // its terms of the sums, taken into the node-local terms
  double rx[9];
#pragma unroll
  for (int c = 0; c < 3; ++c) rx[c] = g.detj * (g.dxi[0] * sux[c]);
  const double cx = g.detj * g.dxi[0];
  const double ddx0 = cx * sdx[0], ddx1 = cx * sdx[1], ddx2 = cx * sdx[2];
  if constexpr (!TR) {
    rx[3] = ddx0; rx[4] = 0.0; rx[5] = 0.0; rx[6] = ddx1; rx[7] = ddx2; rx[8] = 0.0;
  } else {
    rx[3] = -(l2m * ddx0); rx[4] = -(lam * ddx0); rx[5] = -(lam * ddx0);
    rx[6] = -(m2 * ddx1); rx[7] = -(m2 * ddx2); rx[8] = 0.0;
  }
#pragma unroll
  for (int m = 0; m < 9; ++m) {
    const double minv = RAW ? -1.0 : (m < 3 ? minv_u : (m < 6 ? minv_s : 0.5 * minv_s));
    pre[m] = pre[m] - sc * (minv * rx[m]);
  }
  st_node(A.out + so, offu, offs, ua, sm, pre);
}

// block `blk` of the pass over one shot, on vectors in memory
template <bool LAST, bool TR>
__device__ __forceinline__ void nodal_block(const SplitArgs& A, int blk, int shot, NodalLds& sh) {
  const int lb = split_block(blk, A.pnbn);
  if (lb >= A.pnbn) return;
  const Entry E = list_entry(A.g, lb);
  const unsigned NN = (unsigned)A.g.NN;
  const unsigned offu = E.n * 24u, offs = 8u * (3u * NN + (NN & 1u)) + E.n * 48u;
  constexpr int NIN = LAST ? 6 : 3;
  double V[NIN][9];
#pragma unroll
  for (int q = 0; q < NIN; ++q) ld_node((q < 3 ? A.v[q] : A.x[q - 3]) + (long long)shot * A.shot_stride, offu, offs, V[q]);
  nodal_pass<LAST, TR>(A, E, shot, V, sh);
}

// the pass alone
template <bool LAST, bool TR>
__global__ void __launch_bounds__(SPLIT_NT, LAST ? 2 : 3) pml_nodal_kernel(const SplitArgs A) {
  __shared__ NodalLds sh;
  nodal_block<LAST, TR>(A, blockIdx.x, blockIdx.y, sh);
}

// Sources at regular-domain-only nodes, which the element kernel finished: one
// thread per node with entries (the list is in (shot, node) order).
__device__ __forceinline__ void add_domain_sources(const SplitArgs& A, int q) {
  const Src3& sp = A.src;
  if (q >= sp.nrd) return;
  const int shot = sp.rd_shot[q];
  const long long n = sp.node[sp.rd_idx[q]];
  if (q > 0 && sp.rd_shot[q - 1] == shot && sp.node[sp.rd_idx[q - 1]] == n) return;   // not the node's first entry
  const int sdyn = A.step_dev ? *A.step_dev : 0;
  double s[3] = {0.0, 0.0, 0.0};
  for (; q < sp.nrd; ++q) {
    const int jj = sp.rd_idx[q];
    if (sp.rd_shot[q] != shot || sp.node[jj] != n) break;
    const double v = src_value(A, jj, shot, sdyn);
    const int c = sp.comp[jj];
    s[0] += c == 0 ? v : 0.0;
    s[1] += c == 1 ? v : 0.0;
    s[2] += c == 2 ? v : 0.0;
  }
  double* const o = A.a + (long long)shot * A.shot_stride + 3 * n;
#pragma unroll
  for (int c = 0; c < 3; ++c) o[c] += A.ss * s[c];
}

// Pull of an RK4 stage at one PML node: the PML elements' terms from the flux
// records along the y- and z-lines through the node (side-scaled 5-point
// stencils; the x-line terms are in the node-local terms), the regular-domain K
// sums of an interface node from E, the sources, then out = (node-local terms)
// - sc (M^-1 sums) + ss src, sc = ss = 1, in the last stage h^4/24 and h.  The blocks past
// the node blocks add the sources at regular-domain-only nodes.
//
// A block's source entries are evaluated by as many threads at once into LDS and
// each node finds its own through a table over the block's nodes; scanning the
// entries node by node made the adjoint's pull of a 16 x 16 x 8 box, whose blocks
// hold up to 64 receiver entries, 16-19 us long against 6.5 us without sources.
struct PullLds {
  double val[SPLIT_NT];                                // source entries: value,
  int slot[SPLIT_NT], cmp[SPLIT_NT], first[SPLIT_NT];  // node in the block, component; a node's first
};

// the stage's a (or, in the last stage, its part of the new x3) of a node into out; RAW:
// the operator product (E null: no element holds the operator)
template <bool TR, bool RAW = false>
__device__ __forceinline__ void pull_pass(const SplitArgs& A, const Entry& E, int lb, int shot, PullLds& sh,
                                          double* out) {
  double(&sVal)[SPLIT_NT] = sh.val;
  int(&sSlot)[SPLIT_NT] = sh.slot;
  int(&sCmp)[SPLIT_NT] = sh.cmp;
  int(&sFirst)[SPLIT_NT] = sh.first;
  const Geo3& g = A.g;
  const int tid = threadIdx.x;
  int e0 = 0, e1 = 0, jj = -1;          // this block's source entries (a uniform range)
  if (A.src_mode) {
    const int pb = shot * A.src.pnblk + lb;
    e0 = A.src.pblk_ptr[pb];
    e1 = A.src.pblk_ptr[pb + 1];
    if (tid < e1 - e0) jj = A.src.pblk_idx[e0 + tid];
  }
  const int i = E.i, j = E.j, k = E.k;
  const unsigned n = E.n;
  const long long so = (long long)shot * A.shot_stride;
  const unsigned NN = (unsigned)g.NN;
  const unsigned SB = 8u * (3u * NN + (NN & 1u));
  const unsigned offu = n * 24u, offs = SB + n * 48u;

  // node-local terms the nodal pass wrote, and M^-1, issued with the records
  const double minv_u = A.minvu[n];
  const double* __restrict__ tab = A.tab;
  const double sax = tab[TAB_STRETCH + 2 * i], say = tab[TAB_STRETCH + 2 * g.NX + 2 * j],
               saz = tab[TAB_STRETCH + 2 * g.NX + 2 * g.NY + 2 * k];
  double pre[9];
  ld_node(A.out + so, offu, offs, pre);
  double lam = 0.0, mu = 0.0;
  if constexpr (TR) ld2(A.node, n * 16u, lam, mu);
  // interface sums, read with the first batch where a regular-domain element
  // holds the node; other lanes read the shot's first entry (one shared line)
  // and drop it (a list of the interface nodes: as two lattice fields the sums took 6
  // NN doubles a shot, and the pass is as fast)
  const SpAxis ax3[3] = {sp_axis(i, g.nex, g.rlo[0], g.rhi[0]), sp_axis(j, g.ney, g.rlo[1], g.rhi[1]),
                         sp_axis(k, g.nez, g.rlo[2], g.nez)};
  const bool iface = sp_iface(ax3[0], ax3[1], ax3[2]);
  double e3[3] = {0.0, 0.0, 0.0};
  const unsigned eo = (iface ? 24u : 0u) * (iface_column(g, i, j) + iface_rim(g) * (unsigned)(k - 2 * g.rlo[2]));
  if (!RAW || A.E) ld3(A.E + (long long)shot * 3 * A.nif, eo, e3[0], e3[1], e3[2]);
  const int sdyn = (e1 > e0 && A.step_dev) ? *A.step_dev : 0;
  if (e1 > e0) {
    if (jj >= 0) {
      sVal[tid] = src_value(A, jj, shot, sdyn);
      sCmp[tid] = A.src.comp[jj];
      sSlot[tid] = A.src.pblk_slot[e0 + tid];
    }
    sFirst[tid] = -1;
  }
  // M^-1 of the stress rows: 1 / (a W), a the stretch-factor product, W the PML weight sum
  const double minv_s = 1.0 / (((sax * say) * saz) * (g.detj * sp_pml_weight(ax3[0], ax3[1], ax3[2])));
  const double* const Dp = A.D + (long long)shot * 12 * g.NN;
  const int cc[3] = {i, j, k};
  const int nax[3] = {g.NX, g.NY, g.NZ};
  const int str[3] = {1, g.NX, g.NX * g.NY};
  // y- and z-lines (the x-line terms are in the node-local terms): per axis
  // su = sum_d cu[d] G_{.,ax}(n + (d - 2) str), sd the same with the s-row
  // stencil (every offset but 0 negated) on w_{ax,.}
  double su[3][3], sd[3][3];
#pragma unroll
  for (int ax = 1; ax < 3; ++ax) {
    double s0, s1, cu[5];
    sp_side_scales(ax3[ax], ax3[ax == 0 ? 1 : 0], ax3[ax == 2 ? 1 : 2], s0, s1);
    sp_stencil(ax3[ax].odd, s0, s1, cu);
#pragma unroll
    for (int c = 0; c < 3; ++c) { su[ax][c] = 0.0; sd[ax][c] = 0.0; }
#pragma unroll
    for (int d = 0; d < 5; ++d) {
      // odd coordinates have no +-2 terms: skipped (a row of consecutive list
      // entries shares the y and z coordinates)
      if ((d == 0 || d == 4) && ax3[ax].odd) continue;
      // where the coefficient is zero the node itself is read: outside the lattice, and two
      // nodes away across a regular-domain element (one away there is no record).  The
      // product's pull is 2 % faster with addresses that do not wait for the
      // coefficients, the stages' pulls 1 % slower
      const int p = cc[ax] + d - 2;
      const bool use = RAW ? p >= 0 && p < nax[ax] && ((d != 0 && d != 4) || cu[d] != 0.0) : cu[d] != 0.0;
      const unsigned m = use ? (unsigned)((int)n + (d - 2) * str[ax]) : n;
      const unsigned o = d_rec(ax, NN, m);
      double G0, G1, G2, W0, W1, W2;
      ld2(Dp, o, G0, G1);
      ld2(Dp, o + 16u, G2, W0);
      ld2(Dp, o + 32u, W1, W2);
      const double cw = d == 2 ? cu[d] : -cu[d];
      su[ax][0] += cu[d] * G0; su[ax][1] += cu[d] * G1; su[ax][2] += cu[d] * G2;
      sd[ax][0] += cw * W0; sd[ax][1] += cw * W1; sd[ax][2] += cw * W2;
    }
  }
  double raw[9];
#pragma unroll
  for (int c = 0; c < 3; ++c) raw[c] = g.detj * ((0.0 + g.dxi[1] * su[1][c]) + g.dxi[2] * su[2][c]);
#pragma unroll
  for (int c = 0; c < 3; ++c) raw[c] += iface ? e3[c] : 0.0;
  double dd[3][3];
#pragma unroll
  for (int ax = 1; ax < 3; ++ax)
#pragma unroll
    for (int c = 0; c < 3; ++c) dd[ax][c] = (g.detj * g.dxi[ax]) * sd[ax][c];
  const double aE[6] = {0.0, dd[1][1], dd[2][2], dd[1][0], dd[2][0], dd[2][1] + dd[1][2]};
  if constexpr (!TR) {
#pragma unroll
    for (int m = 0; m < 6; ++m) raw[3 + m] = aE[m];
  } else {
    const double l2m = lam + 2.0 * mu, m2 = 2.0 * mu;
    raw[3] = -(l2m * aE[0] + lam * aE[1] + lam * aE[2]);
    raw[4] = -(lam * aE[0] + l2m * aE[1] + lam * aE[2]);
    raw[5] = -(lam * aE[0] + lam * aE[1] + l2m * aE[2]);
    raw[6] = -(m2 * aE[3]);
    raw[7] = -(m2 * aE[4]);
    raw[8] = -(m2 * aE[5]);
  }
  // sources of this node: the block's entries are in node order, so a node's
  // entries follow its first one
  double src[3] = {0.0, 0.0, 0.0};
  for (int c0 = 0; c0 < e1 - e0; c0 += SPLIT_NT) {
    const int ne = min(e1 - e0 - c0, SPLIT_NT);
    if (c0 > 0) {          // more entries than threads (receivers that share DOFs): further batches
      __syncthreads();
      if (tid < ne) {
        const int j2 = A.src.pblk_idx[e0 + c0 + tid];
        sVal[tid] = src_value(A, j2, shot, sdyn);
        sCmp[tid] = A.src.comp[j2];
        sSlot[tid] = A.src.pblk_slot[e0 + c0 + tid];
      }
      sFirst[tid] = -1;
    }
    __syncthreads();
    if (tid < ne && (tid == 0 || sSlot[tid - 1] != sSlot[tid])) sFirst[sSlot[tid]] = tid;
    __syncthreads();
    int e = sFirst[tid];
    if (e >= 0)
      for (; e < ne && sSlot[e] == tid; ++e) {
        const int cpt = sCmp[e];
        src[0] += cpt == 0 ? sVal[e] : 0.0;
        src[1] += cpt == 1 ? sVal[e] : 0.0;
        src[2] += cpt == 2 ? sVal[e] : 0.0;
      }
  }
  // finish on the node-local terms
#pragma unroll
  for (int m = 0; m < 9; ++m) {
    const double minv = RAW ? -1.0 : (m < 3 ? minv_u : (m < 6 ? minv_s : 0.5 * minv_s));
    const double sv = m < 3 ? src[m] : 0.0;
    out[m] = (pre[m] + A.sc * -(minv * raw[m])) + A.ss * sv;
  }
}

// the pull of stages 2 and 4
template <bool TR>
__global__ void __launch_bounds__(SPLIT_NT, 2) pml_pull_kernel(const SplitArgs A) {
  __shared__ PullLds sh;
  const int C8 = 8 * ((A.pnbn + 7) / 8);
  if ((int)blockIdx.x >= C8) {
    if (blockIdx.y == 0) add_domain_sources(A, ((int)blockIdx.x - C8) * SPLIT_NT + threadIdx.x);
    return;
  }
  const int lb = split_block(blockIdx.x, A.pnbn);
  if (lb >= A.pnbn) return;
  const Entry E = list_entry(A.g, lb);
  double out[9];
  pull_pass<TR>(A, E, lb, blockIdx.y, sh, out);
  if (!E.own) return;
  const unsigned NN = (unsigned)A.g.NN;
  st_node(A.a + (long long)blockIdx.y * A.shot_stride, E.n * 24u, 8u * (3u * NN + (NN & 1u)) + E.n * 48u,
          u_act3(A.g, E.i, E.j, E.k), smask3(A.g, E.i, E.j, E.k), out);
}

// The pull of stage 1 or 3 (P) and the nodal pass of the next stage (N) in one pass over
// the PML nodes: the next stage's third input is the a that a node's pull has just
// formed, so it is not read back, and a3, which nothing else reads at PML nodes, is not
// written either (P.a null).  A block forms a for its two entries on each side as
// well, hence a goes to another vector than the node-local terms it starts from, and
// the flux records of odd and even stages alternate.
// Bytes bound the two passes; in one they move 592 a node and stage against 666, and 880
// against 1010 in the last.  64x64x32 elements: stages 1-2 82 us, as before, 3-4 113
// against 126 us (80 and 105 since neighbours of zero coefficient are not read); 96x96x48 per
// step 1.62 -> 1.53 ms; 16x16x8, where launches count, 74 -> 64 us.  Three blocks per CU (six registers spilled) are 1-3 % slower, the next
// stage's other inputs loaded ahead of the pull no faster.
template <bool LAST, bool TR>
__global__ void __launch_bounds__(SPLIT_NT, 2) pull_nodal_kernel(const SplitArgs P, const SplitArgs N) {
  __shared__ union {
    PullLds pull;
    NodalLds nodal;
  } sh;
  constexpr int NIN = LAST ? 6 : 3;
  const int C8 = 8 * ((P.pnbn + 7) / 8);
  if ((int)blockIdx.x >= C8) {
    if (blockIdx.y == 0) add_domain_sources(P, ((int)blockIdx.x - C8) * SPLIT_NT + threadIdx.x);
    return;
  }
  const int lb = split_block(blockIdx.x, P.pnbn);
  if (lb >= P.pnbn) return;
  const int shot = blockIdx.y;
  const Entry E = list_entry(P.g, lb);
  const long long so = (long long)shot * P.shot_stride;
  const unsigned NN = (unsigned)P.g.NN;
  const unsigned offu = E.n * 24u, offs = 8u * (3u * NN + (NN & 1u)) + E.n * 48u;
  double V[NIN][9];
  pull_pass<TR>(P, E, lb, shot, sh.pull, V[2]);
  // inactive components are zero in every vector
  const bool ua = u_act3(P.g, E.i, E.j, E.k);
  const int sm = smask3(P.g, E.i, E.j, E.k);
#pragma unroll
  for (int m = 0; m < 9; ++m)
    if (!(m < 3 ? ua : ((sm >> (m - 3)) & 1) != 0)) V[2][m] = 0.0;
  if (P.a && E.own) st_node(P.a + so, offu, offs, ua, sm, V[2]);
#pragma unroll
  for (int q = 0; q < NIN; ++q)
    if (q != 2) ld_node((q < 2 ? N.v[q] : N.x[q - 3]) + so, offu, offs, V[q]);
  __syncthreads();      // the pull's LDS becomes the nodal pass's
  nodal_pass<LAST, TR>(N, E, shot, V, sh.nodal);
}

// ------------------------------------------------- regular-domain element pass
// Applies K to two displacement fields over the regular-domain elements and
// finishes the regular-domain-only nodes.  UPDATE = false: a1 = -M^-1 K x2 and a2 =
// -M^-1 K x3; UPDATE = true: a3, a4 from a1, a2 and with them the new x2, x3
// (x1 enters PML nodes only, so it is not kept at the others).  The K sums
// of interface nodes (also held by PML elements) go to E for the nodal pull.
//
// A block owns 4 x 4 elements in x-y and a chunk of element layers, and marches up
// the chunk; its window is the owned nodes plus the low-side halo element.  The
// sizes make one thread the unit of every phase: 2 x 121 window positions to load
// per layer, 25 elements x 9 z-lines of GLL points, 3 x 81 owned nodes for the
// sums.  A wavefront holds seven whole elements, so the transposed derivatives
// take the stresses of a line's neighbours by lane shuffles and an element's
// nodal forces leave once, for the owners to sum (at most four a node); summing
// stresses at the owners instead took 27 LDS reads per node and element, in
// branches by the nodes' parities, and 10 us per layer.  A z-line's thread reads its own
// column once for the three points and keeps the column's lambda, mu in registers.
// The loads of the finish and of the next layer are issued when the stresses have
// freed their registers.  Both fields share the window pass and lambda, mu.
// LDS and the latency between its barriers bound it: at 64x64x32 elements 52 of 78 us
// alone are LDS (counters), a quarter of that bank conflicts that no padding of the
// window or the forces removed.  Beside the nodal pass it takes 92 us (first pass) and
// 108 us there; the loads ahead of the stresses 100 us, three blocks per CU (register
// spills) 92-112 us, a form with one lattice column per thread and half the LDS
// traffic 180 us (its widest parity class needs 300 registers), a z-line's own value from
// its register column (45 LDS reads for 63, but 182 registers and so two blocks per
// CU for three) 102 us, 7 x 6 tiles of 512 threads (a quarter less halo work, one
// block per CU) 15 % more at 96x96x48.
constexpr int RT = 4, RW = 2 * RT + 3, RWP = RW * RW, RNE = (RT + 1) * (RT + 1), RO = 2 * RT + 1;
constexpr int REW = 7;                     // elements per wavefront (9 lanes each)
static_assert(4 * REW >= RNE && 2 * RWP <= 256 && 3 * RO * RO <= 256, "one block of four wavefronts");

template <int NF>
struct RdLds {
  double v[NF][3][3][RWP];         // field, plane (k % 3), component, window position
  double r[NF][3][RNE * 27 + 1];   // nodal forces of the elements per field and component, a spare
};

// block `blk` of the pass; NF = 1: K times one field, without the scaling by -M^-1
template <int NF, bool UPDATE>
__device__ __forceinline__ void element_pass(const RdArgs& A, int blk, RdLds<NF>& sh) {
  double(&sV)[NF][3][3][RWP] = sh.v;
  double(&sR)[NF][3][RNE * 27 + 1] = sh.r;
  const Geo3& g = A.g;
  const int tid = threadIdx.x, lane = tid & 63;
  // XCD-aware order: XCD x = blk % 8 takes a contiguous run of the (shot, y, z, x) tiles
  const int ntile = A.ntx * A.nty * A.ntz;
  const int ntot = ntile * A.nshot;
  const int C = (ntot + 7) / 8;
  const int li = (blk & 7) * C + (blk >> 3);
  if (li >= ntot) return;
  const int shot = li / ntile;
  const int t = li - shot * ntile;
  const int tx = t % A.ntx, tz = (t / A.ntx) % A.ntz, ty = t / (A.ntx * A.ntz);
  const int ex0 = g.rlo[0] + RT * tx, ey0 = g.rlo[1] + RT * ty, ez0 = g.rlo[2] + A.tz * tz;
  const int ez_end = min(ez0 + A.tz, g.nez);
  const int ez_first = max(ez0 - 1, g.rlo[2]);
  const long long so = (long long)shot * A.shot_stride;
  const double* const in0 = A.in[0] + so;
  const double* const in1 = NF == 2 ? A.in[1] + so : nullptr;
  const unsigned NXY = (unsigned)(g.NX * g.NY);

  // load role: window position of one of the two new planes (regular-domain nodes only)
  const int lp = tid >= RWP ? 1 : 0;
  const int lpos = tid - lp * RWP;
  const int wi = 2 * ex0 - 2 + lpos % RW, wj = 2 * ey0 - 2 + lpos / RW;
  const bool ldr = tid < 2 * RWP && wi >= 2 * g.rlo[0] && wi <= 2 * g.rhi[0] && wj >= 2 * g.rlo[1] && wj <= 2 * g.rhi[1];
  const unsigned ln = ldr ? (unsigned)(wi + g.NX * wj) : 0u;
  // element role: z-line (lx, ly) of window element se; lane 63 and lanes without a
  // regular-domain element compute on zeros of the window corner and store nothing
  const int le = lane < 9 * REW ? lane / 9 : 0, sq = lane < 9 * REW ? lane - 9 * le : 0;
  const int se = REW * (tid >> 6) + le;
  const int slx = sq % 3, sly = sq / 3;
  const int sex = ex0 - 1 + se % (RT + 1), sey = ey0 - 1 + se / (RT + 1);
  const bool elm = lane < 9 * REW && se < RNE && sex >= g.rlo[0] && sex < g.rhi[0] && sey >= g.rlo[1] && sey < g.rhi[1];
  const int spc = elm ? 2 * (se % (RT + 1)) + slx + RW * (2 * (se / (RT + 1)) + sly) : slx + RW * sly;   // column in the window
  const unsigned sn = elm ? (unsigned)((2 * sex + slx) + g.NX * (2 * sey + sly)) : 0u;
  // the derivative of a, b, c at local point l is (c - a) / 2 + (l - 1) (a - 2 b + c);
  // transposed coefficients DM(a, l) for a = l, l + 1, l + 2 (mod 3) in physical units,
  // and the lanes of those lines
  const double px = slx - 1, py = sly - 1;
  double hx[3], hy[3];
  int nx[3], ny[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    auto dm = [](int a, int b) { return b == 0 ? (a - 1) - 0.5 : (b == 1 ? -2.0 * (a - 1) : (a - 1) + 0.5); };
    const int ax = (slx + c) % 3, ay = (sly + c) % 3;
    hx[c] = g.dxi[0] * dm(ax, slx);
    hy[c] = g.dxi[1] * dm(ay, sly);
    nx[c] = 9 * le + ax + 3 * sly;
    ny[c] = 9 * le + slx + 3 * ay;
  }
  const double swxy = g.detj * (slx == 1 ? 4.0 / 3.0 : 1.0 / 3.0) * (sly == 1 ? 4.0 / 3.0 : 1.0 / 3.0);
  const double dz = g.dxi[2];
  // owner role: column oc of the plane group P (planes k % 3 == P)
  const int P = tid / (RO * RO), oc = tid - P * (RO * RO);
  const int ix = oc % RO, iy = oc / RO;
  const int i = 2 * ex0 + ix, j = 2 * ey0 + iy;
  const bool owned = P < 3 && (ix < 2 * RT || tx == A.ntx - 1) && (iy < 2 * RT || ty == A.nty - 1) && i <= 2 * g.rhi[0] &&
                     j <= 2 * g.rhi[1];
  const int opos = (ix + 2) + RW * (iy + 2);
  const unsigned ecol = 24u * iface_column(g, i, j), rim = iface_rim(g);
  // the node's places in the forces of the up to four elements of a layer that hold it:
  // an odd coordinate has one element (local point 1), an even one the element below
  // (local point 2) and the one above (local point 0)
  int fq[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int a = q & 1, b = q >> 1;
    const int lx = (ix & 1) ? 1 : 2 - 2 * a, ly = (iy & 1) ? 1 : 2 - 2 * b;
    const int exi = (ix >> 1) + ((ix & 1) ? 1 : a), eyi = (iy >> 1) + ((iy & 1) ? 1 : b);
    const int ex = ex0 - 1 + exi, ey = ey0 - 1 + eyi;
    const bool ok = owned && !((ix & 1) && a) && !((iy & 1) && b) && ex >= g.rlo[0] && ex < g.rhi[0] && ey >= g.rlo[1] &&
                    ey < g.rhi[1];
    fq[q] = ok ? 27 * (exi + (RT + 1) * eyi) + lx + 3 * ly : -1;
  }

  auto load_plane = [&](int k, double* r0, double* r1) {
    if (ldr) {
      const unsigned o = (ln + NXY * (unsigned)k) * 24u;
      ld3(in0, o, r0[0], r0[1], r0[2]);
      if constexpr (NF == 2) ld3(in1, o, r1[0], r1[1], r1[2]);
    }
  };
  auto put_plane = [&](int k, const double* r0, const double* r1) {
    if (tid < 2 * RWP) {
      const int s = k % 3;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        sV[0][s][c][lpos] = r0[c];
        if constexpr (NF == 2) sV[NF - 1][s][c][lpos] = r1[c];
      }
    }
  };
  double r0[3] = {0.0, 0.0, 0.0}, r1[3] = {0.0, 0.0, 0.0};
  if (lp == 0) {
    load_plane(2 * ez_first, r0, r1);
    put_plane(2 * ez_first, r0, r1);
  }
  load_plane(2 * ez_first + 1 + lp, r0, r1);
  // lambda, mu of the line's three points: index 2 of a layer is index 0 of the next
  double lm[3][2];
#pragma unroll
  for (int z = 0; z < 3; ++z) ld2(A.node, (sn + NXY * (unsigned)(2 * ez_first + z)) * 16u, lm[z][0], lm[z][1]);

  double acc[NF][3];
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int c = 0; c < 3; ++c) acc[f][c] = 0.0;

  for (int ez = ez_first; ez < ez_end; ++ez) {
    const bool halo = ez < ez0;
    const int p = ((P - 2 * ez) % 3 + 3) % 3;       // this group's plane within the layer
    const int k = 2 * ez + p;
    put_plane(2 * ez + 1 + lp, r0, r1);
    // the nodes finished in this layer: two planes, the top one at the surface
    const bool fin = owned && !halo && (p < 2 || ez == g.nez - 1);
    const bool ifc = fin && pml3(g, i, j, k);       // interface node
    const unsigned n = fin ? (unsigned)i + (unsigned)g.NX * (unsigned)j + NXY * (unsigned)k : 0u;
    double minv = 0.0, x2[3], x3[3], own[2][3];
    __syncthreads();
    const int zs[3] = {(2 * ez) % 3, (2 * ez + 1) % 3, (2 * ez + 2) % 3};
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      double S[3][6];                               // W * stress at the line's points
      {
        double gz[3][3], u[3][3];                   // point, component
#pragma unroll
        for (int c = 0; c < 3; ++c) {
#pragma unroll
          for (int z = 0; z < 3; ++z) u[z][c] = sV[f][zs[z]][c][spc];
          gz[0][c] = dz * (-1.5 * u[0][c] + 2.0 * u[1][c] - 0.5 * u[2][c]);
          gz[1][c] = dz * (0.5 * u[2][c] - 0.5 * u[0][c]);
          gz[2][c] = dz * (0.5 * u[0][c] - 2.0 * u[1][c] + 1.5 * u[2][c]);
        }
#pragma unroll
        for (int z = 0; z < 3; ++z) {
          double gx[3], gy[3];
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            const double* U = sV[f][zs[z]][c];
            const int rx = spc - slx, ry = spc - RW * sly;
            const double a0 = U[rx], a1 = U[rx + 1], a2 = U[rx + 2];
            const double b0 = U[ry], b1 = U[ry + RW], b2 = U[ry + 2 * RW];
            gx[c] = g.dxi[0] * (0.5 * (a2 - a0) + px * ((a0 + a2) - 2.0 * a1));
            gy[c] = g.dxi[1] * (0.5 * (b2 - b0) + py * ((b0 + b2) - 2.0 * b1));
          }
          const double W = swxy * (z == 1 ? 4.0 / 3.0 : 1.0 / 3.0);
          const double lam = W * lm[z][0], mu = W * lm[z][1];
          const double tr = lam * (gx[0] + gy[1] + gz[z][2]), m2 = 2.0 * mu;
          S[z][0] = tr + m2 * gx[0];
          S[z][1] = tr + m2 * gy[1];
          S[z][2] = tr + m2 * gz[z][2];
          S[z][3] = mu * (gy[0] + gx[1]);
          S[z][4] = mu * (gz[z][0] + gx[2]);
          S[z][5] = mu * (gz[z][1] + gy[2]);
          __builtin_amdgcn_sched_barrier(0);        // one plane's reads at a time: no spills
        }
      }
      // nodal forces of the line: transposed derivatives along z in registers, along
      // x and y with the neighbouring lines' stresses
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const int cx = sym3(c, 0), cy = sym3(c, 1), cz = sym3(c, 2);
        double fz[3];
        fz[0] = dz * (-1.5 * S[0][cz] - 0.5 * S[1][cz] + 0.5 * S[2][cz]);
        fz[1] = dz * (2.0 * S[0][cz] - 2.0 * S[2][cz]);
        fz[2] = dz * (-0.5 * S[0][cz] + 0.5 * S[1][cz] + 1.5 * S[2][cz]);
        double t[3][2];                             // a direction's shuffles in flight
#pragma unroll
        for (int z = 0; z < 3; ++z)
#pragma unroll
          for (int d = 0; d < 2; ++d) t[z][d] = __shfl(S[z][cx], nx[d + 1]);
#pragma unroll
        for (int z = 0; z < 3; ++z) fz[z] += hx[0] * S[z][cx] + (hx[1] * t[z][0] + hx[2] * t[z][1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int z = 0; z < 3; ++z)
#pragma unroll
          for (int d = 0; d < 2; ++d) t[z][d] = __shfl(S[z][cy], ny[d + 1]);
#pragma unroll
        for (int z = 0; z < 3; ++z)
          sR[f][c][elm ? 27 * se + sq + 9 * z : RNE * 27] =
              fz[z] + (hy[0] * S[z][cy] + (hy[1] * t[z][0] + hy[2] * t[z][1]));
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // loads of the finish and of the next layer, once the stresses have freed their
    // registers
    if (fin) {
      if constexpr (NF == 2) minv = A.minvu[n];
      if constexpr (UPDATE) {
        ld3(A.x[0] + so, n * 24u, x2[0], x2[1], x2[2]);
        ld3(A.x[1] + so, n * 24u, x3[0], x3[1], x3[2]);
      }
    }
    if (ez + 1 < ez_end) {
      load_plane(2 * ez + 3 + lp, r0, r1);
      lm[0][0] = lm[2][0];
      lm[0][1] = lm[2][1];
#pragma unroll
      for (int z = 1; z < 3; ++z) ld2(A.node, (sn + NXY * (unsigned)(2 * ez + 2 + z)) * 16u, lm[z][0], lm[z][1]);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (UPDATE) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        own[0][c] = sV[0][k % 3][c][opos];
        own[1][c] = sV[1][k % 3][c][opos];
      }
    }
    __syncthreads();
    if (owned && (!halo || p == 2)) {
      // a plane starts afresh unless the layer below started it
      const bool fresh = p != 0 || ez == ez_first;
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          double s = fresh ? 0.0 : acc[f][c];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const double v = sR[f][c][(fq[q] >= 0 ? fq[q] : 0) + 9 * p];
            s += fq[q] >= 0 ? v : 0.0;
          }
          acc[f][c] = s;
        }
    }
    if (fin) {
      if (ifc) {
        const long long eo = (long long)shot * 3 * A.nif;
        const unsigned o = ecol + 24u * rim * (unsigned)(k - 2 * g.rlo[2]);
#pragma unroll
        for (int f = 0; f < NF; ++f) st3(A.E[f] + eo, o, acc[f][0], acc[f][1], acc[f][2]);
      } else if constexpr (NF == 1) {
        st3(A.out[0] + so, n * 24u, acc[0][0], acc[0][1], acc[0][2]);
      } else {
        double o0[3], o1[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const double s0 = -(minv * acc[0][c]), s1 = -(minv * acc[NF - 1][c]);
          if constexpr (UPDATE) {
            const double a1 = own[0][c], a2 = own[1][c];
            o0[c] = x2[c] + (A.h * x3[c] + (A.h2 * a1 + (A.h3 * a2 + A.h4 * s0)));
            o1[c] = x3[c] + (A.h * a1 + (A.h2 * a2 + (A.h3 * s0 + A.h4 * s1)));
          } else {
            o0[c] = s0;
            o1[c] = s1;
          }
        }
        st3(A.out[0] + so, n * 24u, o0[0], o0[1], o0[2]);
        st3(A.out[1] + so, n * 24u, o1[0], o1[1], o1[2]);
      }
    }
  }
}

// the element pass alone
template <bool UPDATE>
__global__ void __launch_bounds__(SPLIT_NT, 2) element_kernel(const RdArgs A) {
  __shared__ RdLds<2> sh;
  element_pass<2, UPDATE>(A, blockIdx.x, sh);
}

// The element pass (the first nrd blocks) and the nodal pass of stages 1 and 3 in one
// launch: the one is bound by LDS, the other by memory, and neither waits for the other,
// so they share the CUs without the events of two streams, which cost 15-20 us a
// stage.  The element blocks run longest and come first: mixed in with the nodal
// blocks, one in two or in proportion, the pair took 5-20 % longer.
// The traces and the history slice of the state that stage 1 reads are the last blocks.
// Against launches of their own (on two streams from 37x29x19 up), forward and adjoint
// step on average: 16x16x8 elements 84 -> 74 us,
// 37x29x19 150 -> 131, 4 shots of 32x32x16 341 -> 317, 64x64x32 equal.
// GRAD: the adjoint step's gradient sums as well, after the element blocks; their 240
// registers leave two blocks on a CU, so only where all blocks fit at once (see
// the launch's caller).
template <bool UPDATE, bool TR, bool GRAD>
__global__ void __launch_bounds__(SPLIT_NT, 2) stage_pair_kernel(const SplitArgs A, const RdArgs R, const OutArgs O,
                                                                const GradArgs G, int nrd, int nn) {
  static_assert(GNT == SPLIT_NT, "one block size");
  __shared__ union {
    NodalLds nodal;
    RdLds<2> element;
    GradLds grad;
  } sh;
  int b = blockIdx.x;
  if (b < nrd) {
    element_pass<2, UPDATE>(R, b, sh.element);
    return;
  }
  b -= nrd;
  if constexpr (GRAD) {
    const int ng = gradient_blocks(G);
    if (b < ng) {
      gradient_block(G, b, sh.grad);
      return;
    }
    b -= ng;
  }
  const int q = b - nn * A.nshot;
  if (q >= 0) {
    const int nb = output_blocks(O);
    output_block(O, q % nb, q / nb);
    return;
  }
  const int shot = b / nn;
  nodal_block<false, TR>(A, b - shot * nn, shot, sh.nodal);
}

// Operator product with G (set 0), K (1) or C (2) on A.v[0], in place of a stage: the nodal
// pass and, in the first nrd blocks, the element pass of K, or zeros at the
// regular-domain-only nodes, which G and C do not reach; then the pull.
// The tile classes of the fused stage kernel recompute each PML flux at up to five
// nodes and put the elements' work on their own CUs only: K on 64x64x32 elements with
// PML 6 took 130 us there against 64 + 35 us here, C^T on 45x37x22 45 against 14 + 12.
template <bool TR>
__global__ void __launch_bounds__(SPLIT_NT, 3) apply_pair_kernel(const SplitArgs A, const RdArgs R, int set, int nrd) {
  __shared__ union {
    NodalLds nodal;
    RdLds<1> element;
  } sh;
  const int b = blockIdx.x;
  if (b < nrd) {
    if (set == 1) {
      element_pass<1, false>(R, b, sh.element);
      return;
    }
    const Geo3& g = A.g;
    const int ni = 2 * (g.rhi[0] - g.rlo[0]) - 1, nj = 2 * (g.rhi[1] - g.rlo[1]) - 1, nk = g.NZ - 1 - 2 * g.rlo[2];
    const int q = b * SPLIT_NT + (int)threadIdx.x;
    if (q >= ni * nj * nk) return;
    const int i = 2 * g.rlo[0] + 1 + q % ni, j = 2 * g.rlo[1] + 1 + (q / ni) % nj, k = 2 * g.rlo[2] + 1 + q / (ni * nj);
    st3(A.out, 24u * (unsigned)(i + g.NX * (j + g.NY * k)), 0.0, 0.0, 0.0);
    return;
  }
  const int lb = split_block(b - nrd, A.pnbn);
  if (lb >= A.pnbn) return;
  const Entry E = list_entry(A.g, lb);
  const unsigned NN = (unsigned)A.g.NN;
  double x[9], V[3][9];
  ld_node(A.v[0], E.n * 24u, 8u * (3u * NN + (NN & 1u)) + E.n * 48u, x);
#pragma unroll
  for (int q = 0; q < 3; ++q)
#pragma unroll
    for (int m = 0; m < 9; ++m) V[q][m] = q == set ? x[m] : 0.0;
  nodal_pass<false, TR, true>(A, E, 0, V, sh.nodal);
}

template <bool TR>
__global__ void __launch_bounds__(SPLIT_NT, 2) apply_pull_kernel(const SplitArgs A) {
  __shared__ PullLds sh;
  const int lb = split_block(blockIdx.x, A.pnbn);
  if (lb >= A.pnbn) return;
  const Entry E = list_entry(A.g, lb);
  double out[9];
  pull_pass<TR, true>(A, E, lb, 0, sh, out);
  if (!E.own) return;
  const unsigned NN = (unsigned)A.g.NN;
  st_node(A.a, E.n * 24u, 8u * (3u * NN + (NN & 1u)) + E.n * 48u, u_act3(A.g, E.i, E.j, E.k),
          smask3(A.g, E.i, E.j, E.k), out);
}

}  // namespace

hipError_t launch_split_nodal(const SplitArgs& A, int last, int transpose, hipStream_t s) {
  if (A.nshot <= 0 || A.pnbn <= 0) return hipSuccess;
  const dim3 grid(8 * ((A.pnbn + 7) / 8), A.nshot);
  if (last) {
    if (transpose) pml_nodal_kernel<true, true><<<grid, SPLIT_NT, 0, s>>>(A);
    else pml_nodal_kernel<true, false><<<grid, SPLIT_NT, 0, s>>>(A);
  } else {
    if (transpose) pml_nodal_kernel<false, true><<<grid, SPLIT_NT, 0, s>>>(A);
    else pml_nodal_kernel<false, false><<<grid, SPLIT_NT, 0, s>>>(A);
  }
  return hipGetLastError();
}

namespace {
// blocks of the pull: the list's, and those of the sources at regular-domain-only nodes
dim3 pull_grid(const SplitArgs& A) {
  const int nsrc = A.src_mode ? (A.src.nrd + SPLIT_NT - 1) / SPLIT_NT : 0;
  return dim3(8 * ((A.pnbn + 7) / 8) + nsrc, A.nshot);
}
}  // namespace

hipError_t launch_split_pull(const SplitArgs& A, int transpose, hipStream_t s) {
  if (A.nshot <= 0 || pull_grid(A).x == 0) return hipSuccess;
  if (transpose) pml_pull_kernel<true><<<pull_grid(A), SPLIT_NT, 0, s>>>(A);
  else pml_pull_kernel<false><<<pull_grid(A), SPLIT_NT, 0, s>>>(A);
  return hipGetLastError();
}

hipError_t launch_pull_nodal(const SplitArgs& P, const SplitArgs& N, int last, int transpose, hipStream_t s) {
  const dim3 grid = pull_grid(P);
  if (P.nshot <= 0 || grid.x == 0) return hipSuccess;
  if (last) {
    if (transpose) pull_nodal_kernel<true, true><<<grid, SPLIT_NT, 0, s>>>(P, N);
    else pull_nodal_kernel<true, false><<<grid, SPLIT_NT, 0, s>>>(P, N);
  } else {
    if (transpose) pull_nodal_kernel<false, true><<<grid, SPLIT_NT, 0, s>>>(P, N);
    else pull_nodal_kernel<false, false><<<grid, SPLIT_NT, 0, s>>>(P, N);
  }
  return hipGetLastError();
}

void rd_tiles(const Geo& g, int tz, int t[3]) {
  t[0] = (g.rhi[0] - g.rlo[0] + RT - 1) / RT;
  t[1] = (g.rhi[1] - g.rlo[1] + RT - 1) / RT;
  t[2] = (g.nez - g.rlo[2] + tz - 1) / tz;
}

hipError_t launch_elements(const RdArgs& R, int update, hipStream_t s) {
  const long long n = (long long)R.ntx * R.nty * R.ntz * R.nshot;
  if (n <= 0) return hipSuccess;
  const unsigned nb = (unsigned)(8 * ((n + 7) / 8));
  if (update) element_kernel<true><<<nb, SPLIT_NT, 0, s>>>(R);
  else element_kernel<false><<<nb, SPLIT_NT, 0, s>>>(R);
  return hipGetLastError();
}

int stage_pair_blocks(const SplitArgs& A, const RdArgs& R) {
  const long long n = (long long)R.ntx * R.nty * R.ntz * R.nshot;
  return (int)(8 * ((n + 7) / 8)) + 8 * ((A.pnbn + 7) / 8) * A.nshot;
}

hipError_t launch_stage_pair(const SplitArgs& A, const RdArgs& R, const OutArgs& O, const GradArgs& G, int update,
                             int transpose, hipStream_t s) {
  if (A.nshot <= 0) return hipSuccess;
  const int nn = 8 * ((A.pnbn + 7) / 8), nrd = stage_pair_blocks(A, R) - nn * A.nshot, ng = gradient_blocks(G);
  if (ng > 0 && (update || !transpose)) return hipErrorInvalidValue;   // the gradient goes with the adjoint's stage 1
  const unsigned nb = (unsigned)(nrd + nn * A.nshot + ng + output_blocks(O) * O.nshot);
  if (nb == 0) return hipSuccess;
  if (ng > 0) stage_pair_kernel<false, true, true><<<nb, SPLIT_NT, 0, s>>>(A, R, O, G, nrd, nn);
  else if (update) {
    if (transpose) stage_pair_kernel<true, true, false><<<nb, SPLIT_NT, 0, s>>>(A, R, O, G, nrd, nn);
    else stage_pair_kernel<true, false, false><<<nb, SPLIT_NT, 0, s>>>(A, R, O, G, nrd, nn);
  } else {
    if (transpose) stage_pair_kernel<false, true, false><<<nb, SPLIT_NT, 0, s>>>(A, R, O, G, nrd, nn);
    else stage_pair_kernel<false, false, false><<<nb, SPLIT_NT, 0, s>>>(A, R, O, G, nrd, nn);
  }
  return hipGetLastError();
}

hipError_t launch_split_apply(const SplitArgs& A, const RdArgs& R, int set, int transpose, hipStream_t s) {
  const Geo3& g = A.g;
  long long n = (long long)R.ntx * R.nty * R.ntz;
  if (set != 1) {
    const long long only = (2ll * (g.rhi[0] - g.rlo[0]) - 1) * (2 * (g.rhi[1] - g.rlo[1]) - 1) * (g.NZ - 1 - 2 * g.rlo[2]);
    n = g.rhi[0] > g.rlo[0] && g.rhi[1] > g.rlo[1] && only > 0 ? (only + SPLIT_NT - 1) / SPLIT_NT : 0;
  }
  const int nrd = (int)(8 * ((n + 7) / 8)), nn = 8 * ((A.pnbn + 7) / 8);
  if (nrd + nn == 0) return hipSuccess;
  if (transpose) apply_pair_kernel<true><<<nrd + nn, SPLIT_NT, 0, s>>>(A, R, set, nrd);
  else apply_pair_kernel<false><<<nrd + nn, SPLIT_NT, 0, s>>>(A, R, set, nrd);
  if (nn > 0) {
    if (transpose) apply_pull_kernel<true><<<nn, SPLIT_NT, 0, s>>>(A);
    else apply_pull_kernel<false><<<nn, SPLIT_NT, 0, s>>>(A);
  }
  return hipGetLastError();
}

}  // namespace hr
