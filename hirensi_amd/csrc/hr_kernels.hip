// Small HIP kernels around the stage kernel (hr_stage3.hip): reference
// numbering <-> lattice slots for the operator apply, receiver traces,
// regular-domain history slices, the per-step lambda/mu gradient, misfit.
//
// State layout: per state vector, the displacement block [3 * n + c]
// (c = u_x, u_y, u_z) followed by the stress block [SB + 6 * n + m]
// (m = s_xx s_yy s_zz s_xy s_xz s_yz; SB = 3 NN rounded up to an even count,
// so that a node's stress components are 16-byte aligned),
// n = i + NX * (j + NY * k): the components of a node are contiguous.
// Inactive entries are zero and never written.

#include <hip/hip_runtime.h>
#include "hr_lattice.h"

#pragma clang fp contract(off)

namespace hr {

// ----------------------------------------------------- small kernels
// lattice <- reference numbering (optionally scaled): out[slot[e]] = x[e] * r[e]
__global__ void gather_eq_kernel(long long neq, const unsigned* __restrict__ slot, const double* __restrict__ x,
                                 const double* __restrict__ r, double* __restrict__ out) {
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < neq; e += (long long)gridDim.x * blockDim.x) {
    const double v = x[e];
    out[slot[e]] = r ? v * r[e] : v;
  }
}

// reference numbering <- lattice: z[e] = y[e] + s * (l[e] * raw[slot[e]])
__global__ void scatter_eq_kernel(long long neq, const unsigned* __restrict__ slot, const double* __restrict__ raw,
                                  const double* __restrict__ y, double s, const double* __restrict__ l,
                                  double* __restrict__ z) {
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < neq; e += (long long)gridDim.x * blockDim.x) {
    double a = raw[slot[e]];
    if (l) a = l[e] * a;
    z[e] = y[e] + s * a;
  }
}

// device-side step index of a captured time loop
__global__ void step_set_kernel(int* __restrict__ step, int value) {
  if (threadIdx.x == 0) step[0] = value;
}
__global__ void step_advance_kernel(int* __restrict__ step, int delta) {
  if (threadIdx.x == 0) step[0] = step[0] + delta;
}

// The material's tables, a node per thread.  The sums over the elements that hold the
// node are taken in element order.  First the pairs and the arrays, then
// (material_quad_kernel) the quadruples, where host arrays may have been staged.
// On the host, as loops over the elements with an upload of each table, they
// took about 2 ms at 32x32x16 elements.
__global__ void __launch_bounds__(256) material_kernel(Geo g, const double* __restrict__ tab,
                                                       const double* __restrict__ lam, const double* __restrict__ mu,
                                                       const double* __restrict__ rho, double* __restrict__ pairs,
                                                       double* __restrict__ mrd, double* __restrict__ minvu,
                                                       double* __restrict__ rwp) {
  for (long long n = blockIdx.x * 256LL + threadIdx.x; n < g.NN; n += 256LL * gridDim.x) {
    const int i = (int)(n % g.NX), j = (int)((n / g.NX) % g.NY), k = (int)(n / ((long long)g.NX * g.NY));
    const int x0 = i >= 1 ? (i - 1) / 2 : 0, x1 = min(i / 2, g.nex - 1);
    const int y0 = j >= 1 ? (j - 1) / 2 : 0, y1 = min(j / 2, g.ney - 1);
    const int z0 = k >= 1 ? (k - 1) / 2 : 0, z1 = min(k / 2, g.nez - 1);
    double sr = 0.0, sp = 0.0;
    for (int ez = z0; ez <= z1; ++ez)
      for (int ey = y0; ey <= y1; ++ey)
        for (int ex = x0; ex <= x1; ++ex) {
          const double m = rho[ex + (long long)g.nex * (ey + (long long)g.ney * ez)] *
                           tab[(i - 2 * ex) + 3 * (j - 2 * ey) + 9 * (k - 2 * ez)];
          if (ex >= g.rlo[0] && ex < g.rhi[0] && ey >= g.rlo[1] && ey < g.rhi[1] && ez >= g.rlo[2]) sr += m;
          else sp += m;
        }
    const double a = tab[TAB_STRETCH + 2 * i] * tab[TAB_STRETCH + 2 * g.NX + 2 * j] *
                     tab[TAB_STRETCH + 2 * (g.NX + g.NY) + 2 * k];
    const double M = sr + a * sp;
    mrd[n] = sr;
    rwp[n] = sp;
    minvu[n] = M > 0.0 ? 1.0 / M : 0.0;
    pairs[2 * n] = lam[n];
    pairs[2 * n + 1] = mu[n];
  }
}

__global__ void __launch_bounds__(256) material_quad_kernel(Geo g, const double* __restrict__ tab,
                                                            const double* __restrict__ minvu,
                                                            const double* __restrict__ rwp,
                                                            double* __restrict__ quad) {
  for (long long n = blockIdx.x * 256LL + threadIdx.x; n < g.NN; n += 256LL * gridDim.x) {
    const int i = (int)(n % g.NX), j = (int)((n / g.NX) % g.NY), k = (int)(n / ((long long)g.NX * g.NY));
    const int x0 = i >= 1 ? (i - 1) / 2 : 0, x1 = min(i / 2, g.nex - 1);
    const int y0 = j >= 1 ? (j - 1) / 2 : 0, y1 = min(j / 2, g.ney - 1);
    const int z0 = k >= 1 ? (k - 1) / 2 : 0, z1 = min(k / 2, g.nez - 1);
    double w = 0.0;
    for (int ez = z0; ez <= z1; ++ez)
      for (int ey = y0; ey <= y1; ++ey)
        for (int ex = x0; ex <= x1; ++ex)
          if (!(ex >= g.rlo[0] && ex < g.rhi[0] && ey >= g.rlo[1] && ey < g.rhi[1] && ez >= g.rlo[2]))
            w += tab[(i - 2 * ex) + 3 * (j - 2 * ey) + 9 * (k - 2 * ez)];
    const double a = tab[TAB_STRETCH + 2 * i] * tab[TAB_STRETCH + 2 * g.NX + 2 * j] *
                     tab[TAB_STRETCH + 2 * (g.NX + g.NY) + 2 * k];
    quad[4 * n] = minvu[n];
    quad[4 * n + 1] = w > 0.0 ? 1.0 / (a * w) : 0.0;
    quad[4 * n + 2] = rwp[n];
    quad[4 * n + 3] = w;
  }
}

// traces and history slice of a state (hr_lattice.h)
__global__ void __launch_bounds__(OUT_NT) output_kernel(const OutArgs O) { output_block(O, blockIdx.x, blockIdx.y); }

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

__global__ void __launch_bounds__(GNT, GBLOCKS) gradient_tile_kernel(
    Geo g, int bi0, int bj0, int bk0, int bnx, int bny, int bnz, int ntx, int nty, int ntz, int tz, int nshot,
    const double* __restrict__ uh, long long ustride, const double* __restrict__ p2, long long pstride, double dt,
    double* __restrict__ glam, double* __restrict__ gmu, const int* __restrict__ step, long long stride) {
#pragma clang fp contract(fast)
  __shared__ double sU[2][3][GW], sP[2][3][GW];
  const int tid = threadIdx.x;
  const int tx = tid % GTX, ty = tid / GTX;
  const int ntile = ntx * nty * ntz, ntot = ntile * nshot;
  // XCD-aware order: XCD x = blockIdx % 8 takes a contiguous run of the (shot, z, y, x) tiles
  const int C = (ntot + 7) / 8;
  const int li = (blockIdx.x & 7) * C + (blockIdx.x >> 3);
  if (li >= ntot) return;
  const int shot = li / ntile, t = li - shot * ntile;
  const int nbox = bnx * bny * bnz;              // 32-bit: 9 NN < 2^31 (checked by the host)
  if (step) uh += (long long)(*step) * stride;
  uh += shot * ustride;
  p2 += shot * pstride;
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
    const unsigned kk = (unsigned)min(max(k, 0), bnz - 1);
    const unsigned r = (r0 + (unsigned)(bnx * bny) * kk) * 8u;
    const unsigned n = (n0 + (unsigned)(g.NX * g.NY) * kk) * 24u;
    u[0] = ldo(u0p, r);
    u[1] = ldo(u1p, r);
    u[2] = ldo(u2p, r);
    ld3(p2, n, p[0], p[1], p[2]);
  };
  const int ci = min(bi, bnx - 1), cj = min(bj, bny - 1);
  const unsigned r0 = (unsigned)(ci + bnx * cj), n0 = (unsigned)((bi0 + ci) + g.NX * ((bj0 + cj) + g.NY * bk0));
  const int wo = (GH + tx) + GWX * (GH + ty);
  // halo position of this thread
  int hx = 0, hy = 0;
  if (tid < 4 * GTX) { hy = tid / GTX; hx = GH + (tid - hy * GTX); if (hy >= 2) hy += GTY; }
  else if (tid < GHALO) { const int q = tid - 4 * GTX; hy = GH + (q >> 2); hx = q & 3; if (hx >= 2) hx += GTX; }
  const bool halo = tid < GHALO;
  const int hi = min(max(ti0 + hx - GH, 0), bnx - 1), hj = min(max(tj0 + hy - GH, 0), bny - 1);
  const unsigned hr0 = (unsigned)(hi + bnx * hj), hn0 = (unsigned)((bi0 + hi) + g.NX * ((bj0 + hj) + g.NY * bk0));
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
  cnt[0] = sides(bi, bnx, g.dxi[0], 1, ox, cx);
  cnt[1] = sides(bj, bny, g.dxi[1], GWX, oy, cy);
  const double wxy = g.wq[1 + 3 * 1 + 9 * 1] * (bi & 1 ? 1.0 : 0.25) * (bj & 1 ? 1.0 : 0.25) * dt;
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
      const double c = 0.5 * g.dxi[2];
      cnt[2] = 1;
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        Z.u[m] = c * (qu[3][m] - qu[1][m]);
        Z.p[m] = c * (qp[3][m] - qp[1][m]);
        Z.d[m] = Z.u[m] * Z.p[m];
      }
    } else {
      const double c0 = k >= 2 ? 0.5 * g.dxi[2] : 0.0, c1 = k + 2 <= bnz - 1 ? 0.5 * g.dxi[2] : 0.0;
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

// dst[n][q] = src[n][perm[q]]: receiver columns in source-entry order
__global__ void permute_cols_kernel(long long nrows, int ncols, const long long* __restrict__ perm,
                                    const double* __restrict__ src, double* __restrict__ dst) {
  const long long tot = nrows * ncols;
  for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < tot; t += (long long)gridDim.x * blockDim.x) {
    const long long n = t / ncols;
    const int q = (int)(t - n * ncols);
    dst[t] = src[n * ncols + perm[q]];
  }
}

// Misfit partial sums per step (Compute_Misfit, Solver_PETSc_Inverse.F90:633-650):
// the residuals of receivers that share an equation are added first (VecSetValues
// with ADD_VALUES), then the squares are summed in equation order (VecDot).
// Group g holds the receivers gidx[gptr[g] .. gptr[g+1]), groups in ascending
// equation order.
__global__ void __launch_bounds__(256) misfit_rows_kernel(int nstep, int ngrp, const int* __restrict__ gptr,
                                                          const int* __restrict__ gidx, int nrec,
                                                          const double* __restrict__ tr,
                                                          const double* __restrict__ ob, double* __restrict__ part) {
  // one wavefront per time row: lane l takes groups l, l + 64, ... (neighbouring
  // receivers of the row, coalesced), then a fixed butterfly sums the lanes
  const int lane = threadIdx.x & 63;
  const int nstp = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (nstp > nstep) return;                       // whole wavefront (uniform)
  const long long row = (long long)nstp * nrec;
  double c = 0.0;
  for (int g = lane; g < ngrp; g += 64) {
    double b = 0.0;
    for (int j = gptr[g]; j < gptr[g + 1]; ++j) {
      const int r = gidx[j];
      b += tr[row + r] - ob[row + r];
    }
    c += b * b;
  }
  for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
  if (lane == 0) part[nstp] = c;
}

// J = sum_{n = NSTEP..1} 0.5 * part[n] * dt  (Compute_Misfit order)
__global__ void misfit_sum_kernel(int nstep, const double* __restrict__ part, double dt, double* __restrict__ out) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    double cost = 0.0;
    for (int n = nstep; n >= 1; --n) cost = cost + 0.5 * part[n] * dt;
    out[0] = cost;
  }
}

// out = in[0] + in[1] + ... + in[n-1], in that order (per-shot misfits)
__global__ void sum_kernel(int n, const double* __restrict__ in, double* __restrict__ out) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    double c = 0.0;
    for (int q = 0; q < n; ++q) c = c + in[q];
    out[0] = c;
  }
}

// g <- -(sum over the shots of g) for the regular-domain box, scattered to the nodal output
__global__ void gradient_finish_kernel(Geo g, int bi0, int bj0, int bk0, int bnx, int bny, int bnz, int nshot,
                                       const double* __restrict__ gl_box, const double* __restrict__ gm_box,
                                       double* __restrict__ gl, double* __restrict__ gm) {
  const long long nbox = (long long)bnx * bny * bnz;
  for (long long r = blockIdx.x * (long long)blockDim.x + threadIdx.x; r < nbox; r += (long long)gridDim.x * blockDim.x) {
    const int bi = (int)(r % bnx), bj = (int)((r / bnx) % bny), bk = (int)(r / ((long long)bnx * bny));
    const long long n = (long long)(bi0 + bi) + (long long)g.NX * ((long long)(bj0 + bj) + (long long)g.NY * (bk0 + bk));
    double sl = 0.0, sm = 0.0;
    for (int q = 0; q < nshot; ++q) {
      sl += gl_box[q * nbox + r];
      sm += gm_box[q * nbox + r];
    }
    gl[n] = sl * -1.0;
    gm[n] = sm * -1.0;
  }
}

// g[n] += box[r] over the regular-domain node box (one Update_g step into the
// caller's nodal gradients)
__global__ void box_add_kernel(Geo g, int bi0, int bj0, int bk0, int bnx, int bny, int bnz,
                               const double* __restrict__ gl_box, const double* __restrict__ gm_box,
                               double* __restrict__ gl, double* __restrict__ gm) {
  const long long nbox = (long long)bnx * bny * bnz;
  for (long long r = blockIdx.x * (long long)blockDim.x + threadIdx.x; r < nbox; r += (long long)gridDim.x * blockDim.x) {
    const int bi = (int)(r % bnx), bj = (int)((r / bnx) % bny), bk = (int)(r / ((long long)bnx * bny));
    const long long n = (long long)(bi0 + bi) + (long long)g.NX * ((long long)(bj0 + bj) + (long long)g.NY * (bk0 + bk));
    gl[n] = gl[n] + gl_box[r];
    gm[n] = gm[n] + gm_box[r];
  }
}

// Regular-domain energy (TOTAL_ENERGY_RD_PETSC_EXPLICIT, Obsolete.F90:108-150):
// 0.5 (u . AK_RD u + (M_RD x3) . x3); AK_RD is never assembled (the insertion is
// commented out, Assemble_PETSc_3D.F90:163), so only the kinetic term remains.
// Fixed grid of ENERGY_BLOCKS blocks, partial sums in block order: deterministic.
constexpr int ENERGY_BLOCKS = 256;
__global__ void __launch_bounds__(256) energy_partial_kernel(long long nn, const double* __restrict__ mrd,
                                                             const double* __restrict__ x3,
                                                             double* __restrict__ part) {
  __shared__ double red[256];
  double acc = 0.0;
  for (long long n = blockIdx.x * 256LL + threadIdx.x; n < nn; n += 256LL * gridDim.x) {
    const double m = mrd[n];
    const double a = x3[3 * n], b = x3[3 * n + 1], c = x3[3 * n + 2];
    acc += (m * a) * a + (m * b) * b + (m * c) * c;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}
__global__ void energy_finish_kernel(const double* __restrict__ part, double* __restrict__ out) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    double c = 0.0;
    for (int b = 0; b < ENERGY_BLOCKS; ++b) c += part[b];
    out[0] = 0.50 * (0.0 + c);
  }
}

}  // namespace hr

// ------------------------------------------------------------ launchers
namespace hr {
namespace {
int grid_for(long long n) {
  long long b = (n + 255) / 256;
  if (b < 1) b = 1;
  return (int)(b < 65535 ? b : 65535);
}
}  // namespace

hipError_t launch_gather_eq(long long neq, const unsigned* slot, const double* x, const double* r, double* out,
                            hipStream_t s) {
  hipLaunchKernelGGL(gather_eq_kernel, dim3(grid_for(neq)), dim3(256), 0, s, neq, slot, x, r, out);
  return hipGetLastError();
}
hipError_t launch_scatter_eq(long long neq, const unsigned* slot, const double* raw, const double* y, double sc,
                             const double* l, double* z, hipStream_t s) {
  hipLaunchKernelGGL(scatter_eq_kernel, dim3(grid_for(neq)), dim3(256), 0, s, neq, slot, raw, y, sc, l, z);
  return hipGetLastError();
}
hipError_t launch_material(const Geo& g, const double* tab, const double* lam, const double* mu, const double* rho,
                           double* node, double* mrd, double* minvu, double* rwp, hipStream_t s) {
  material_kernel<<<grid_for(g.NN), 256, 0, s>>>(g, tab, lam, mu, rho, node, mrd, minvu, rwp);
  material_quad_kernel<<<grid_for(g.NN), 256, 0, s>>>(g, tab, minvu, rwp, node + NT_PAIR * g.NN);
  return hipGetLastError();
}

hipError_t launch_outputs(const OutArgs& O, hipStream_t s) {
  if (output_blocks(O) <= 0) return hipSuccess;
  output_kernel<<<dim3(output_blocks(O), O.nshot), OUT_NT, 0, s>>>(O);
  return hipGetLastError();
}
hipError_t launch_step_set(int* step, int value, hipStream_t s) {
  hipLaunchKernelGGL(step_set_kernel, dim3(1), dim3(64), 0, s, step, value);
  return hipGetLastError();
}
hipError_t launch_step_advance(int* step, int delta, hipStream_t s) {
  hipLaunchKernelGGL(step_advance_kernel, dim3(1), dim3(64), 0, s, step, delta);
  return hipGetLastError();
}
hipError_t launch_gradient(const Geo& g, const int* b0, const int* bn, int nshot, const double* uh, long long ustride,
                           const double* p2, long long pstride, double dt, double* glam, double* gmu, hipStream_t s,
                           StepRef sr) {
  // planes per chunk: the fewest planes in sequence, rounds of blocks times planes
  // with the two that a chunk's start costs; of equals the longest
  const int ntx = (bn[0] + GTX - 1) / GTX, nty = (bn[1] + GTY - 1) / GTY;
  const long long slots = 256 * GBLOCKS;
  long long best = -1;
  int tz = bn[2];
  for (int c = bn[2]; c >= 1; --c) {
    const long long n = (long long)ntx * nty * ((bn[2] + c - 1) / c) * nshot;
    const long long cost = (n + slots - 1) / slots * (c + 2);
    if (best < 0 || cost < best) { best = cost; tz = c; }
  }
  const int ntz = (bn[2] + tz - 1) / tz;
  const long long n = (long long)ntx * nty * ntz * nshot;
  if (n <= 0) return hipSuccess;
  gradient_tile_kernel<<<(unsigned)(8 * ((n + 7) / 8)), GNT, 0, s>>>(g, b0[0], b0[1], b0[2], bn[0], bn[1], bn[2], ntx,
                                                                     nty, ntz, tz, nshot, uh, ustride, p2, pstride, dt,
                                                                     glam, gmu, sr.step, sr.stride);
  return hipGetLastError();
}
hipError_t launch_gradient_finish(const Geo& g, const int* b0, const int* bn, int nshot, const double* glb, const double* gmb,
                                  double* gl, double* gm, hipStream_t s) {
  const long long tot = (long long)bn[0] * bn[1] * bn[2];
  hipLaunchKernelGGL(gradient_finish_kernel, dim3(grid_for(tot)), dim3(256), 0, s, g, b0[0], b0[1], b0[2], bn[0],
                     bn[1], bn[2], nshot, glb, gmb, gl, gm);
  return hipGetLastError();
}
hipError_t launch_box_add(const Geo& g, const int* b0, const int* bn, const double* glb, const double* gmb, double* gl,
                          double* gm, hipStream_t s) {
  const long long tot = (long long)bn[0] * bn[1] * bn[2];
  hipLaunchKernelGGL(box_add_kernel, dim3(grid_for(tot)), dim3(256), 0, s, g, b0[0], b0[1], b0[2], bn[0], bn[1],
                     bn[2], glb, gmb, gl, gm);
  return hipGetLastError();
}
int energy_partials_size() { return ENERGY_BLOCKS; }
hipError_t launch_energy(long long nn, const double* mrd, const double* x3, double* part, double* out, hipStream_t s) {
  hipLaunchKernelGGL(energy_partial_kernel, dim3(ENERGY_BLOCKS), dim3(256), 0, s, nn, mrd, x3, part);
  hipLaunchKernelGGL(energy_finish_kernel, dim3(1), dim3(64), 0, s, part, out);
  return hipGetLastError();
}
hipError_t launch_permute_cols(long long nrows, int ncols, const long long* perm, const double* src, double* dst,
                               hipStream_t s) {
  hipLaunchKernelGGL(permute_cols_kernel, dim3(grid_for(nrows * ncols)), dim3(256), 0, s, nrows, ncols, perm, src, dst);
  return hipGetLastError();
}
hipError_t launch_sum(int n, const double* in, double* out, hipStream_t s) {
  hipLaunchKernelGGL(sum_kernel, dim3(1), dim3(64), 0, s, n, in, out);
  return hipGetLastError();
}
hipError_t launch_misfit(int nstep, int ngrp, const int* gptr, const int* gidx, int nrec, const double* tr,
                         const double* ob, double dt, double* part, double* out, hipStream_t s) {
  hipLaunchKernelGGL(misfit_rows_kernel, dim3((nstep + 1 + 3) / 4), dim3(256), 0, s, nstep, ngrp, gptr, gidx, nrec,
                     tr, ob, part);
  hipLaunchKernelGGL(misfit_sum_kernel, dim3(1), dim3(64), 0, s, nstep, part, dt, out);
  return hipGetLastError();
}
}  // namespace hr
