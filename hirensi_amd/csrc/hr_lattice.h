// Device helpers of the lattice kernels: accesses to a node's contiguous
// components and the DOF rules of the box (internal linkage, included by the
// stage kernels).
#pragma once
#include <hip/hip_runtime.h>
#include "hr_device.h"
#include "hr_index.h"

namespace hr {
namespace {

// one double at a byte offset from a uniform base
__device__ __forceinline__ double ldo(const double* p, unsigned off) {
  return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(p) + off);
}
__device__ __forceinline__ void sto(double* p, unsigned off, double v) {
  *reinterpret_cast<double*>(reinterpret_cast<char*>(p) + off) = v;
}
// two consecutive doubles at a 16-byte aligned offset
__device__ __forceinline__ void ld2(const double* p, unsigned off, double& a, double& b) {
  const double2 t = *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(p) + off);
  a = t.x;
  b = t.y;
}
// three consecutive components of a node (8-byte aligned): one 16-byte and one
// 8-byte access instead of three 8-byte ones
struct alignas(8) D3 {
  double v[3];
};
__device__ __forceinline__ void ld3(const double* p, unsigned off, double& a, double& b, double& c) {
  const D3 t = *reinterpret_cast<const D3*>(reinterpret_cast<const char*>(p) + off);
  a = t.v[0];
  b = t.v[1];
  c = t.v[2];
}
__device__ __forceinline__ void st3(double* p, unsigned off, double a, double b, double c) {
  D3 t;
  t.v[0] = a;
  t.v[1] = b;
  t.v[2] = c;
  *reinterpret_cast<D3*>(reinterpret_cast<char*>(p) + off) = t;
}
// six consecutive components at a 16-byte aligned offset: three 16-byte stores
__device__ __forceinline__ void st6(double* p, unsigned off, const double* v) {
  char* q = reinterpret_cast<char*>(p) + off;
#pragma unroll
  for (int a = 0; a < 3; ++a) *reinterpret_cast<double2*>(q + 16 * a) = make_double2(v[2 * a], v[2 * a + 1]);
}
// stores of three consecutive components, each only where its bit of act is set
__device__ __forceinline__ void st3m(double* p, unsigned off, int act, double a, double b, double c) {
  if (act == 7) {
    st3(p, off, a, b, c);
  } else {
    if (act & 1) sto(p, off, a);
    if (act & 2) sto(p, off + 8u, b);
    if (act & 4) sto(p, off + 16u, c);
  }
}

__device__ __forceinline__ bool in_dom3(const Geo3& g, int i, int j, int k) {
  return i >= 0 && j >= 0 && k >= 0 && i < g.NX && j < g.NY && k < g.NZ;
}
__device__ __forceinline__ bool u_act3(const Geo3& g, int i, int j, int k) {
  return !(i == 0 || j == 0 || k == 0 || i == g.NX - 1 || j == g.NY - 1);
}
// node touched by at least one PML element
__device__ __forceinline__ bool pml3(const Geo3& g, int i, int j, int k) {
  return !(i > 2 * g.rlo[0] && i < 2 * g.rhi[0] && j > 2 * g.rlo[1] && j < 2 * g.rhi[1] && k > 2 * g.rlo[2]);
}
// active stress components (bit m) of a PML node
__device__ __forceinline__ int smask3(const Geo3& g, int i, int j, int k) {
  if (g.top_rule && k == g.NZ - 1 && !((i & 1) && (j & 1))) return 0x3f & ~((1 << 2) | (1 << 4) | (1 << 5));
  return 0x3f;
}
__device__ __forceinline__ bool rd3(const Geo3& g, int ex, int ey, int ez) {
  return ex >= g.rlo[0] && ex < g.rhi[0] && ey >= g.rlo[1] && ey < g.rhi[1] && ez >= g.rlo[2];
}
__device__ __forceinline__ int sym3(int i, int k) { return i == k ? i : i + k + 2; }

__device__ __forceinline__ void st2(double* p, unsigned off, double a, double b) {
  *reinterpret_cast<double2*>(reinterpret_cast<char*>(p) + off) = make_double2(a, b);
}

// The last stage's update of one component from X = a1, a2, a3, x1, x2, x3 and
// the weights h, h^2/2, h^3/6, h^4/24: the new x1 and x2, and the part c3 of the
// new x3 that does not need a4 (x3 + ... + h^4/24 a4)
__device__ __forceinline__ void rk4_update(const double* X, double h, double h2, double h3, double h4, double& xn0,
                                           double& xn1, double& c3) {
  xn0 = X[3] + (h * X[4] + (h2 * X[5] + (h3 * X[0] + h4 * X[1])));
  xn1 = X[4] + (h * X[5] + (h2 * X[0] + (h3 * X[1] + h4 * X[2])));
  c3 = X[5] + (h * X[0] + (h2 * X[1] + h3 * X[2]));
}

// Value of source entry jj of a shot: forward f(row) B M^-1, adjoint the weighted
// residual rows times M^-1 (sdyn: offset of a captured step)
template <class Args>
__device__ __forceinline__ double src_value(const Args& A, int jj, int shot, int sdyn) {
  const Src3& sp = A.src;
  const double mm = sp.m[jj];
  if (A.src_mode == 1) {
    const double f = sp.ftab[((size_t)shot * sp.nstep + (A.step + sdyn)) * 3 + A.fcol];
    return f * (sp.val[jj] * mm);
  }
  const size_t nr = (size_t)sp.nrec;
  const size_t base = (size_t)shot * ((size_t)sp.nstep + 1) * nr + ((size_t)jj - (size_t)shot * nr);
  const size_t ra = (size_t)(A.ra + sdyn);
  double val = A.ca * ((sp.tr[base + ra * nr] - sp.obs[base + ra * nr]) * mm);
  if (A.rb_on) {
    const size_t rb = (size_t)(A.rb + sdyn);
    val = val + A.cb * ((sp.tr[base + rb * nr] - sp.obs[base + rb * nr]) * mm);
  }
  return val;
}

// Block `blk` of a step's outputs of one shot: receiver traces row[r] = x2[slot[r]], then
// the displacement of the regular-domain node box into the history slice (3 x
// nbox, component-major): a thread reads one node's three contiguous components and
// writes them to the three component planes (each plane coalesced across lanes).
__device__ __forceinline__ void output_block(const OutArgs& O, int blk, int shot) {
  const double* __restrict__ x2 = O.x2 + shot * O.xstride;
  const int nrb = (O.nrec + OUT_NT - 1) / OUT_NT;
  if (blk < nrb) {
    const int r = blk * OUT_NT + (int)threadIdx.x;
    double* row = O.row + shot * O.rstride;
    if (O.step) row += (long long)(*O.step) * O.nrec;
    if (r < O.nrec) row[r] = x2[O.slot[r]];
    return;
  }
  const int r = (blk - nrb) * OUT_NT + (int)threadIdx.x;
  if (r >= O.nbox) return;
  double* hist = O.hist + shot * O.hstride;
  if (O.step) hist += (long long)(*O.step) * 3 * O.nbox;
  const int bi = r % O.bn[0], bj = (r / O.bn[0]) % O.bn[1], bk = r / (O.bn[0] * O.bn[1]);
  double u0, u1, u2;
  ld3(x2 + plane_doubles(O.NX, O.NY, O.b0[2] + bk), in_plane_bytes(O.NX, O.b0[0] + bi, O.b0[1] + bj), u0, u1, u2);
  hist[r] = u0;
  hist[O.nbox + r] = u1;
  hist[2 * (long long)O.nbox + r] = u2;
}

}  // namespace
}  // namespace hr
