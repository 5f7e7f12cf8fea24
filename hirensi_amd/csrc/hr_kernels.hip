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
#include "hr_gradient.h"
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

__global__ void __launch_bounds__(GNT, GBLOCKS) gradient_tile_kernel(const GradArgs G) {
  __shared__ GradLds sh;
  gradient_block(G, blockIdx.x, sh);
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
GradArgs gradient_args(const Geo& g, const int* b0, const int* bn, int nshot, const double* uh, long long ustride,
                       const double* p2, long long pstride, double dt, double* glam, double* gmu, StepRef sr) {
  // planes per chunk: the fewest planes in sequence, rounds of blocks times planes
  // with the two that a chunk's start costs; of equals the longest
  GradArgs G{};
  G.ntx = (bn[0] + GTX - 1) / GTX;
  G.nty = (bn[1] + GTY - 1) / GTY;
  const long long slots = 256 * GBLOCKS;
  long long best = -1;
  G.tz = bn[2];
  for (int c = bn[2]; c >= 1; --c) {
    const long long n = (long long)G.ntx * G.nty * ((bn[2] + c - 1) / c) * nshot;
    const long long cost = (n + slots - 1) / slots * (c + 2);
    if (best < 0 || cost < best) { best = cost; G.tz = c; }
  }
  G.ntz = (bn[2] + G.tz - 1) / G.tz;
  G.nshot = nshot;
  G.NX = g.NX; G.NY = g.NY;
  for (int d = 0; d < 3; ++d) { G.b0[d] = b0[d]; G.bn[d] = bn[d]; G.dxi[d] = g.dxi[d]; }
  G.wdt = g.wq[13] * dt;
  G.uh = uh; G.ustride = ustride;
  G.p2 = p2; G.pstride = pstride;
  G.glam = glam; G.gmu = gmu;
  G.step = sr.step; G.stride = sr.stride;
  return G;
}

hipError_t launch_gradient(const GradArgs& G, hipStream_t s) {
  const int n = gradient_blocks(G);
  if (n <= 0) return hipSuccess;
  gradient_tile_kernel<<<n, GNT, 0, s>>>(G);
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
