// The per-step lambda, mu gradient of one adjoint step (internal linkage, included by the
// kernels that run it).
#pragma once
#include <hip/hip_runtime.h>
#include "hr_lattice.h"

namespace hr {
namespace {

// Per-step gradient accumulation (Update_g + ELEMENT_g_3D, Assemble_PETSc_3D.F90:556-661,
// Element_Matrices_3D.F90:1725-1890): for every node of the regular-domain box,
// sum over the regular-domain elements containing it of W * div u * div p and
// W * [2 eps(u):eps(p) in the reference's component form], times dt.
// u comes from the history slice (3 x nbox), p from the adjoint x2 (lattice).
//
// Per axis a node has one element side (odd coordinate) or two (even: below and
// above), each with its own derivatives; the weight W = w_x w_y w_z is the same for all
// the elements of a node.  The sum over the up to eight elements of a product of
// derivatives along axes a and b then splits into sums over sides: of products
// for a = b, times the number of sides of the other two axes, and a product of sums
// for a != b, times that of the third axis.  A side outside the box enters with
// zero coefficients.
//
// A block owns GTX x GTY box columns and marches up a chunk of planes.  The thread of a
// column keeps the planes k-2..k+2 of its own u and p in registers (z stencils); plane k
// of the block's window, with a halo of two nodes, sits in LDS (x and y stencils).
// What plane k + 1 needs is loaded before plane k is worked on, and the two LDS
// planes alternate, so a plane costs one barrier and no load in its path.  All shots
// go in one launch, each with accumulators of its own: one small box alone has too
// few blocks for the GPU.
// One call alone: 64x64x32 elements with PML 6, 41 -> 19 us (47 MB, about half
// the copy rate); 32x32x16 with PML 4, 18 -> 6 us.
constexpr int GTX = 32, GTY = 8, GH = 2;
constexpr int GWX = GTX + 2 * GH, GWY = GTY + 2 * GH, GW = GWX * GWY;
constexpr int GNT = GTX * GTY;
// halo positions read by the stencils: rows 0, 1 and GWY-2, GWY-1 over the owned
// columns (y stencils), columns 0, 1 and GWX-2, GWX-1 over the owned rows (x stencils)
constexpr int GHALO = 2 * 2 * GTX + 2 * 2 * GTY;
static_assert(GHALO <= GNT, "one halo position per thread");
constexpr int GBLOCKS = 2;                     // blocks per CU: three spill 100 registers (79 us for 19)

// one axis' sides of u and p: sums over the sides of each component, and of the
// products of equal components
struct Sides {
  double u[3], p[3], d[3];
};

struct GradLds {
  double u[2][3][GW], p[2][3][GW];
};

// block `blk`
__device__ __forceinline__ void gradient_block(const GradArgs& A, int blk, GradLds& sh) {
#pragma clang fp contract(fast)
  double(&sU)[2][3][GW] = sh.u;
  double(&sP)[2][3][GW] = sh.p;
  const int bi0 = A.b0[0], bj0 = A.b0[1], bk0 = A.b0[2], bnx = A.bn[0], bny = A.bn[1], bnz = A.bn[2];
  const int ntx = A.ntx, nty = A.nty, tz = A.tz;
  const double* __restrict__ uh = A.uh;
  const double* __restrict__ p2 = A.p2;
  double* __restrict__ glam = A.glam;
  double* __restrict__ gmu = A.gmu;
  const int tid = threadIdx.x;
  const int tx = tid % GTX, ty = tid / GTX;
  const int ntile = ntx * nty * A.ntz, ntot = ntile * A.nshot;
  // XCD-aware order: XCD x = blk % 8 takes a contiguous run of the (shot, z, y, x) tiles
  const int C = (ntot + 7) / 8;
  const int li = (blk & 7) * C + (blk >> 3);
  if (li >= ntot) return;
  const int shot = li / ntile, t = li - shot * ntile;
  const int nbox = bnx * bny * bnz;              // and its byte offsets fit 32 bits (LATTICE_NODES)
  if (A.step) uh += (long long)(*A.step) * A.stride;
  uh += shot * A.ustride;
  p2 += shot * A.pstride;
  glam += (long long)shot * nbox;
  gmu += (long long)shot * nbox;
  const int ti0 = (t % ntx) * GTX, tj0 = ((t / ntx) % nty) * GTY;
  const int kc0 = (t / (ntx * nty)) * tz, kc1 = min(kc0 + tz, bnz);
  const int bi = ti0 + tx, bj = tj0 + ty;
  const bool own = bi < bnx && bj < bny;
  // u and p of a box column at plane k, both clamped to the box: a position outside it
  // meets zero coefficients only
  const double *const u0p = uh, *const u1p = uh + nbox, *const u2p = uh + 2 * nbox;
  auto fetch = [&](unsigned r0, unsigned n0, int k, double* u, double* p) {
    const int kk = min(max(k, 0), bnz - 1);
    const unsigned r = (r0 + (unsigned)(bnx * bny) * (unsigned)kk) * 8u;
    u[0] = ldo(u0p, r);
    u[1] = ldo(u1p, r);
    u[2] = ldo(u2p, r);
    ld3(p2 + plane_doubles(A.NX, A.NY, bk0 + kk), n0, p[0], p[1], p[2]);
  };
  const int ci = min(bi, bnx - 1), cj = min(bj, bny - 1);
  const unsigned r0 = (unsigned)(ci + bnx * cj), n0 = in_plane_bytes(A.NX, bi0 + ci, bj0 + cj);
  const int wo = (GH + tx) + GWX * (GH + ty);
  // halo position of this thread
  int hx = 0, hy = 0;
  if (tid < 4 * GTX) { hy = tid / GTX; hx = GH + (tid - hy * GTX); if (hy >= 2) hy += GTY; }
  else if (tid < GHALO) { const int q = tid - 4 * GTX; hy = GH + (q >> 2); hx = q & 3; if (hx >= 2) hx += GTX; }
  const bool halo = tid < GHALO;
  const int hi = min(max(ti0 + hx - GH, 0), bnx - 1), hj = min(max(tj0 + hy - GH, 0), bny - 1);
  const unsigned hr0 = (unsigned)(hi + bnx * hj), hn0 = in_plane_bytes(A.NX, bi0 + hi, bj0 + hj);
  const int hw = hx + GWX * hy;
  // x and y sides.  Side 0 is the element below (even node, its local point 2) or
  // the one element of an odd node (local point 1), side 1 the element above (local
  // point 0).  With a, b the side's other two values,
  //   even, below  (3 (f - a) + b - a) / 2     odd  (a - b) / 2
  //   above        (3 (a - f) + a - b) / 2
  int ox[4], oy[4];
  double cx[3], cy[3];
  int cnt[3];
  auto sides = [&](int q, int n, double dxi, int unit, int* o, double* c) {
    const bool odd = q & 1, below = q >= 2, above = !odd && q + 2 <= n - 1;
    o[0] = odd ? unit : -unit;
    o[1] = odd ? -unit : -2 * unit;
    o[2] = odd ? 0 : unit;
    o[3] = odd ? 0 : 2 * unit;
    c[0] = !odd && below ? 1.5 * dxi : 0.0;
    c[1] = odd ? 0.5 * dxi : (below ? -0.5 * dxi : 0.0);
    c[2] = above ? 0.5 * dxi : 0.0;
    return (odd || below ? 1 : 0) + (above ? 1 : 0);
  };
  cnt[0] = sides(bi, bnx, A.dxi[0], 1, ox, cx);
  cnt[1] = sides(bj, bny, A.dxi[1], GWX, oy, cy);
  const double wxy = A.wdt * (bi & 1 ? 1.0 : 0.25) * (bj & 1 ? 1.0 : 0.25);
  // own column: planes k-2 .. k+2 (index 0..4); halo of plane k
  double qu[5][3], qp[5][3], hu[3], hp[3];
#pragma unroll
  for (int d = 0; d < 5; ++d) fetch(r0, n0, kc0 - 2 + d, qu[d], qp[d]);
  fetch(hr0, hn0, kc0, hu, hp);
  for (int k = kc0; k < kc1; ++k) {
    double(*const U)[GW] = sU[(k - kc0) & 1];
    double(*const Q)[GW] = sP[(k - kc0) & 1];
#pragma unroll
    for (int c = 0; c < 3; ++c) { U[c][wo] = qu[2][c]; Q[c][wo] = qp[2][c]; }
    if (halo)
#pragma unroll
      for (int c = 0; c < 3; ++c) { U[c][hw] = hu[c]; Q[c][hw] = hp[c]; }
    Sides Z;
    if (k & 1) {
      const double c = 0.5 * A.dxi[2];
      cnt[2] = 1;
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        Z.u[m] = c * (qu[3][m] - qu[1][m]);
        Z.p[m] = c * (qp[3][m] - qp[1][m]);
        Z.d[m] = Z.u[m] * Z.p[m];
      }
    } else {
      const double c0 = k >= 2 ? 0.5 * A.dxi[2] : 0.0, c1 = k + 2 <= bnz - 1 ? 0.5 * A.dxi[2] : 0.0;
      cnt[2] = (k >= 2 ? 1 : 0) + (k + 2 <= bnz - 1 ? 1 : 0);
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        const double u0 = c0 * (3.0 * (qu[2][m] - qu[1][m]) + (qu[0][m] - qu[1][m]));
        const double u1 = c1 * (3.0 * (qu[3][m] - qu[2][m]) + (qu[3][m] - qu[4][m]));
        const double p0 = c0 * (3.0 * (qp[2][m] - qp[1][m]) + (qp[0][m] - qp[1][m]));
        const double p1 = c1 * (3.0 * (qp[3][m] - qp[2][m]) + (qp[3][m] - qp[4][m]));
        Z.u[m] = u0 + u1;
        Z.p[m] = p0 + p1;
        Z.d[m] = u0 * p0 + u1 * p1;
      }
    }
    // the window moves up (index 1 is now plane k); the next plane's inputs
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int c = 0; c < 3; ++c) { qu[d][c] = qu[d + 1][c]; qp[d][c] = qp[d + 1][c]; }
    if (k + 1 < kc1) {
      fetch(r0, n0, k + 3, qu[4], qp[4]);
      if (halo) fetch(hr0, hn0, k + 1, hu, hp);
    }
    const unsigned r = (r0 + (unsigned)(bnx * bny * k)) * 8u;
    const double gl0 = ldo(glam, r), gm0 = ldo(gmu, r);
    __syncthreads();
    Sides X, Y;
    auto line = [&](const int* o, const double* c, Sides& S) {
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        const double* fu = U[m] + wo;
        const double* fp = Q[m] + wo;
        const double ua = fu[o[0]], pa = fp[o[0]], ub = fu[o[2]], pb = fp[o[2]];
        const double u0 = c[0] * (qu[1][m] - ua) + c[1] * (ua - fu[o[1]]);
        const double u1 = c[2] * (3.0 * (ub - qu[1][m]) + (ub - fu[o[3]]));
        const double p0 = c[0] * (qp[1][m] - pa) + c[1] * (pa - fp[o[1]]);
        const double p1 = c[2] * (3.0 * (pb - qp[1][m]) + (pb - fp[o[3]]));
        S.u[m] = u0 + u1;
        S.p[m] = p0 + p1;
        S.d[m] = u0 * p0 + u1 * p1;
        __builtin_amdgcn_sched_barrier(0);         // one component's reads at a time: no spills
      }
    };
    const double nx = cnt[0], ny = cnt[1], nz = cnt[2];
    const double nyz = ny * nz, nxz = nx * nz, nxy = nx * ny;
    double sl = 0.0, dd = nxy * Z.d[2], sh = nxy * (Z.d[0] + Z.d[1]);
    line(ox, cx, X);
    dd += nyz * X.d[0];
    sh += nyz * (X.d[1] + X.d[2]) + ny * (Z.p[0] * X.u[2] + X.p[2] * Z.u[0]);
    sl += ny * (X.u[0] * Z.p[2] + Z.u[2] * X.p[0]);
    line(oy, cy, Y);
    dd += nxz * Y.d[1];
    sh += nxz * (Y.d[0] + Y.d[2]) + nz * (Y.p[0] * X.u[1] + X.p[1] * Y.u[0]) + nx * (Y.p[2] * Z.u[1] + Z.p[1] * Y.u[2]);
    sl += nz * (X.u[0] * Y.p[1] + Y.u[1] * X.p[0]) + nx * (Y.u[1] * Z.p[2] + Z.u[2] * Y.p[1]);
    if (own) {
      const double W = wxy * (k & 1 ? 1.0 : 0.25);
      sto(glam, r, gl0 + (dd + sl) * W);
      sto(gmu, r, gm0 + (2.0 * dd + sh) * W);
    }
  }
}

}  // namespace
}  // namespace hr
