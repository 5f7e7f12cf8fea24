// Gradient post-processing on the regular-domain box: the gradient mass
// (Assem_R_Mg_3D, Assemble_PETSc_3D.F90:670-748, inverted as in
// Control_Problem_Operators.F90:12-24), the TV and TN regularisation vectors
// (ELEMENT_TV_TN_Reg_3D / ELEMENT_R_Mg_3D, Element_Matrices_3D.F90:1555-1718,
// 1899-2075, assembled by Assemble_PETSc_3D.F90:670-860) and the update of the
// misfit gradient of Program_Main.F90:431-455.
//
// All elements of the box share one affine geometry, so at a GLL point q =
// (i, j, k) of an element the derivative of the shape function of local node
// (a, b, c) is dxi_x L_a'(xi_i) [b == j][c == k] (and likewise along y, z):
// the gradient of a nodal field at q is three 3-term sums along the lattice
// lines through q, and the element vector scatters back along the same lines.
//
// Sums over nodes and elements are taken per block in a fixed order and added by
// one block in block order, so that a repeated call gives the same bits.
#include <hip/hip_runtime.h>

#include "hr_device.h"

namespace hr {
namespace {

// L_a'(xi_q) of the quadratic Lagrange basis on the GLL points (-1, 0, 1)
__device__ __forceinline__ double dl(int q, int a) {
  constexpr double D[3][3] = {{-1.5, 2.0, -0.5}, {-0.5, 0.0, 0.5}, {0.5, -2.0, 1.5}};
  return D[q][a];
}

// Fortran REAL -> default INTEGER as flang compiles it (truncation, saturation
// at the int32 range, NaN -> 0): the reference's TV cost takes its
// `numerator` through an implicitly INTEGER variable.
__device__ __forceinline__ double f90_int4(double x) {
  if (x != x) return 0.0;
  const double t = trunc(x);
  return t < -2147483648.0 ? -2147483648.0 : (t > 2147483647.0 ? 2147483647.0 : t);
}

struct RegArgs {
  Geo g;
  const double* zc;          // lattice z coordinates
  int ntx, nty, ntz, tz;     // tiles, element layers per z-chunk
  int weighted;              // Weighted_Regularization
  double w_top, w_bot, w_len;
  const double* m[2];        // lambda, mu (nodal)
  const double* gr[2];       // misfit gradients (null: their norms are not taken)
  double* r[2];              // regularisation vectors (nodal)
  double* part;              // per-block sums, columns as reg_tail_kernel reads them
};

constexpr int REG_THREADS = 256;
constexpr int REG_BLOCKS = 4;                    // blocks per CU (128 VGPRs without spills)
constexpr int REG_STREAM = 1024;                 // blocks that clear the rest of the lattice
constexpr int RT = 4, RO = 2 * RT + 1, RNE = (RT + 1) * (RT + 1);
constexpr int REW = 7;                           // elements per wavefront (9 lanes each)
static_assert(4 * REW >= RNE && 3 * RO * RO <= REG_THREADS, "one block of four wavefronts");

// sum of v over the block (every thread calls it; the result is thread 0's)
__device__ double block_sum(double v, double* sh) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) v += __shfl_down(v, w);
  if ((tid & 63) == 0) sh[tid >> 6] = v;
  __syncthreads();
  const double s = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  __syncthreads();
  return s;
}

// TV: reg_I = sum_q W_q F_q (grad N_I . grad m) / sqrt(|grad m|^2 + 0.01), cost =
// sum_q W_q F_q int(|grad m|^2) / sqrt(...); TN: reg = ER m, cost = 1/2 m.ER m.
//
// Tile blocks: a block owns the nodes of 4 x 4 elements in x-y and of a chunk of element
// layers and marches up the chunk; the elements on the low side of the tile and
// the layer below the chunk are computed again.  Nine lanes take an element,
// each a z-line of three GLL points: the line's nodal values come from memory
// once, the neighbouring lines' values and fluxes by lane shuffles, and the
// element vectors go through LDS to the nodes' owners (at most four elements of a layer).
// So each node is written once, with its share of ||reg||^2 taken on the way.
// Stream blocks: zeros outside the box and ||g||^2 over the lattice.
//
// The instructions bound it (700 per layer and wavefront, a fifth of them shuffles): 57
// us at 64x64x32 elements with PML 6, for 75 MB of traffic.  One launch per element
// colour, which read and wrote every vector entry 3.4 times, with separate passes for
// the zeros and the sums, took 250 us there.  The point's |grad m|^2 keeps its separate
// multiplies and adds, as the cost truncates it.
template <bool TV>
__global__ __launch_bounds__(REG_THREADS, REG_BLOCKS) void reg_kernel(const RegArgs A) {
  __shared__ double sR[2][RNE * 27 + 1];         // element vectors, and a spare
  __shared__ double sh[4];
  const Geo& g = A.g;
  const int tid = threadIdx.x, lane = tid & 63;
  const int ntile = A.ntx * A.nty * A.ntz;
  const unsigned NXY = (unsigned)(g.NX * g.NY);
  if ((int)blockIdx.x >= ntile) {
    const int b = blockIdx.x - ntile;
    double s0 = 0.0, s1 = 0.0;
    for (long long n = b * (long long)REG_THREADS + tid; n < g.NN; n += (long long)REG_STREAM * REG_THREADS) {
      const unsigned u = (unsigned)n, k = u / NXY, jk = u / (unsigned)g.NX;
      const int i = (int)(u - jk * (unsigned)g.NX), j = (int)(jk - k * (unsigned)g.NY);
      const bool box = i >= 2 * g.rlo[0] && i <= 2 * g.rhi[0] && j >= 2 * g.rlo[1] && j <= 2 * g.rhi[1] &&
                       (int)k >= 2 * g.rlo[2] && (int)k <= 2 * g.rhi[2];
      if (!box || ntile == 0) A.r[0][n] = A.r[1][n] = 0.0;
      if (A.gr[0]) {
        const double a = A.gr[0][n], c = A.gr[1][n];
        s0 += a * a;
        s1 += c * c;
      }
    }
    if (A.gr[0]) {
      s0 = block_sum(s0, sh);
      s1 = block_sum(s1, sh);
      if (tid == 0) {
        A.part[b] = s0;
        A.part[REG_STREAM + b] = s1;
      }
    }
    return;
  }
  // XCD-aware order: XCD x = blockIdx % 8 takes a contiguous run of the tiles (the
  // first ntile / 8 of each; the rest of the blocks follow in order)
  const int C = ntile / 8;
  const int t = (int)blockIdx.x < 8 * C ? (blockIdx.x & 7) * C + (blockIdx.x >> 3) : (int)blockIdx.x;
  const int tx = t % A.ntx, tz = (t / A.ntx) % A.ntz, ty = t / (A.ntx * A.ntz);
  const int ex0 = g.rlo[0] + RT * tx, ey0 = g.rlo[1] + RT * ty, ez0 = g.rlo[2] + A.tz * tz;
  const int ez_end = min(ez0 + A.tz, g.rhi[2]);
  const int ez_first = max(ez0 - 1, g.rlo[2]);
  // element role: z-line (slx, sly) of window element se (lanes without an element
  // compute on a node that is there and store nothing)
  const int le = lane < 9 * REW ? lane / 9 : 0, sq = lane < 9 * REW ? lane - 9 * le : 0;
  const int se = REW * (tid >> 6) + le;
  const int slx = sq % 3, sly = sq / 3;
  const int sex = ex0 - 1 + se % (RT + 1), sey = ey0 - 1 + se / (RT + 1);
  const bool elm = lane < 9 * REW && se < RNE && sex >= g.rlo[0] && sex < g.rhi[0] && sey >= g.rlo[1] && sey < g.rhi[1];
  const bool mine = elm && sex >= ex0 && sey >= ey0;      // the tile's own elements: their cost
  const unsigned sn = elm ? (unsigned)((2 * sex + slx) + g.NX * (2 * sey + sly))
                          : (unsigned)(2 * g.rlo[0] + g.NX * (2 * g.rlo[1]));
  auto dm = [](int q, int a) { return a == 0 ? (q - 1) - 0.5 : (a == 1 ? -2.0 * (q - 1) : (q - 1) + 0.5); };
  double fx[3], fy[3], hx[3], hy[3];     // L_a' at this line's point, L' of this line's point at point a (x, y)
  int nx[3], ny[3];                      // and the lanes of those lines
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    fx[a] = dm(slx, a);
    fy[a] = dm(sly, a);
    hx[a] = g.dxi[0] * dm(a, slx);
    hy[a] = g.dxi[1] * dm(a, sly);
    nx[a] = 9 * le + a + 3 * sly;
    ny[a] = 9 * le + slx + 3 * a;
  }
  const double d0 = g.dxi[0], d1 = g.dxi[1], d2 = g.dxi[2];
  // owner role: column oc of the plane group P (planes k % 3 == P)
  const int P = tid / (RO * RO), oc = tid - P * (RO * RO);
  const int ix = oc % RO, iy = oc / RO;
  const int i = 2 * ex0 + ix, j = 2 * ey0 + iy;
  const bool owned = P < 3 && (ix < 2 * RT || tx == A.ntx - 1) && (iy < 2 * RT || ty == A.nty - 1) && i <= 2 * g.rhi[0] &&
                     j <= 2 * g.rhi[1];
  int fq[4];                             // the node's places in its elements' vectors
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
  double m[2][3], acc[2] = {0.0, 0.0}, cost[2] = {0.0, 0.0}, rr[2] = {0.0, 0.0};
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int z = 0; z < 3; ++z) m[f][z] = A.m[f][sn + NXY * (unsigned)(2 * ez_first + z)];
  for (int ez = ez_first; ez < ez_end; ++ez) {
    const bool halo = ez < ez0;
    const int p = ((P - 2 * ez) % 3 + 3) % 3;    // this group's plane within the layer
    const int k = 2 * ez + p;
    const bool next = ez + 1 < ez_end;
    double w3[3], mn[2][2];
#pragma unroll
    for (int z = 0; z < 3; ++z) {
      w3[z] = g.wq[sq + 9 * z];
      if (A.weighted) {
        const double f2 = fabs(A.zc[2 * ez + z] / A.w_len);
        w3[z] *= (1.0 - f2) * A.w_top + f2 * A.w_bot;
      }
    }
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int z = 0; z < 2; ++z) mn[f][z] = next ? A.m[f][sn + NXY * (unsigned)(2 * ez + 3 + z)] : 0.0;
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      double X[3], Y[3], Z[3];
#pragma unroll
      for (int z = 0; z < 3; ++z) {
        double gx = 0.0, gy = 0.0, gz = 0.0;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          gx += fx[a] * __shfl(m[f][z], nx[a]);
          gy += fy[a] * __shfl(m[f][z], ny[a]);
          gz += dl(z, a) * m[f][a];
        }
        gx *= d0;
        gy *= d1;
        gz *= d2;
        const double s = (gx * gx + gy * gy) + gz * gz;
        double w = w3[z], c;
        if (TV) {
          w = w * rsqrt(s + 0.01);
          c = f90_int4(s) * w;
        } else {
          c = s * w;
        }
        if (mine && !halo) cost[f] += c;
        X[z] = w * gx;
        Y[z] = w * gy;
        Z[z] = w * gz * d2;
      }
#pragma unroll
      for (int z = 0; z < 3; ++z) {
        double r = 0.0;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          r = fma(hx[a], __shfl(X[z], nx[a]), r);
          r = fma(hy[a], __shfl(Y[z], ny[a]), r);
          r = fma(dl(a, z), Z[a], r);
        }
        sR[f][elm ? 27 * se + sq + 9 * z : RNE * 27] = r;
      }
      m[f][0] = m[f][2];
      m[f][1] = mn[f][0];
      m[f][2] = mn[f][1];
    }
    __syncthreads();
    if (owned && (!halo || p == 2)) {
      // a plane starts afresh unless the layer below started it
      const bool fresh = p != 0 || ez == ez_first;
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        double s = fresh ? 0.0 : acc[f];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double v = sR[f][(fq[q] >= 0 ? fq[q] : 0) + 9 * p];
          s += fq[q] >= 0 ? v : 0.0;
        }
        acc[f] = s;
      }
      if (!halo && (p < 2 || ez == g.rhi[2] - 1)) {
        const unsigned n = (unsigned)i + (unsigned)g.NX * (unsigned)j + NXY * (unsigned)k;
#pragma unroll
        for (int f = 0; f < 2; ++f) {
          A.r[f][n] = acc[f];
          rr[f] += acc[f] * acc[f];
        }
      }
    }
    __syncthreads();
  }
  double* const part = A.part + 2 * REG_STREAM;
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    const double a = block_sum(rr[f], sh), c = block_sum(cost[f], sh);
    if (tid == 0) {
      part[f * ntile + blockIdx.x] = a;
      part[(2 + f) * ntile + blockIdx.x] = TV ? c : 0.5 * c;
    }
  }
}

// out = [||g_l||^2, ||g_m||^2 (when taken), ||r_l||^2, ||r_m||^2, cost_l, cost_m]: one
// wavefront per sum
__global__ __launch_bounds__(384) void reg_tail_kernel(int ntile, int norms, const double* __restrict__ part,
                                                       double* __restrict__ out) {
  const int v = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (v < 2 && !norms) return;
  const double* const p = v < 2 ? part + v * REG_STREAM : part + 2 * REG_STREAM + (long long)(v - 2) * ntile;
  const int n = v < 2 ? REG_STREAM : ntile;
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  int q = lane;
  for (; q + 192 < n; q += 256)
#pragma unroll
    for (int u = 0; u < 4; ++u) s[u] += p[q + 64 * u];
  for (; q < n; q += 64) s[0] += p[q];
  double a = (s[0] + s[1]) + (s[2] + s[3]);
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) a += __shfl_down(a, w);
  if (lane == 0) out[v] = a;
}

// Gradient mass at a lattice node: the GLL weights x det J of the box elements
// that hold it, summed in element order; 1/Mg where Mg > 1e-10 (else 0) and
// the 0/1 restriction.
__global__ __launch_bounds__(256) void gradient_mass_kernel(Geo g, double* __restrict__ img,
                                                            double* __restrict__ restr) {
  const long long NN = g.NN;
  for (long long n = blockIdx.x * (long long)blockDim.x + threadIdx.x; n < NN;
       n += (long long)gridDim.x * blockDim.x) {
    const int i = (int)(n % g.NX), j = (int)((n / g.NX) % g.NY), k = (int)(n / ((long long)g.NX * g.NY));
    const int idx[3] = {i, j, k};
    int e_lo[3], e_hi[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      // elements along axis d holding lattice index idx[d]: (idx-1)/2 .. idx/2
      e_lo[d] = idx[d] >= 1 ? (idx[d] - 1) / 2 : 0;
      e_hi[d] = idx[d] / 2;
      const int ne = d == 0 ? g.nex : (d == 1 ? g.ney : g.nez);
      if (e_hi[d] > ne - 1) e_hi[d] = ne - 1;
      if (e_lo[d] < g.rlo[d]) e_lo[d] = g.rlo[d];
      if (e_hi[d] > g.rhi[d] - 1) e_hi[d] = g.rhi[d] - 1;
    }
    double mg = 0.0;
    for (int ez = e_lo[2]; ez <= e_hi[2]; ++ez)
      for (int ey = e_lo[1]; ey <= e_hi[1]; ++ey)
        for (int ex = e_lo[0]; ex <= e_hi[0]; ++ex)
          mg += g.wq[(i - 2 * ex) + 3 * (j - 2 * ey) + 9 * (k - 2 * ez)];
    const bool on = mg > 1.0e-10;
    img[n] = on ? 1.0 / mg : 0.0;
    if (restr) restr[n] = on ? 1.0 : 0.0;
  }
}

// The adaptive factors f = factor ||g|| / ||reg|| (0 when ||reg|| = 0, a homogeneous
// field, where the reference divides by zero) from the sums in red, then
// g <- (g + f reg) img (add = 1), g <- g img (add = 0); red[6..9] = the scaled costs
// and the factors.  One pass at copy speed; the factors are two divides a
// thread, where reading the sums back first made the host wait between the passes.
__global__ __launch_bounds__(256) void reg_update_kernel(long long n, int add, double factor,
                                                         const double* __restrict__ rl, const double* __restrict__ rm,
                                                         const double* __restrict__ img, double* __restrict__ gl,
                                                         double* __restrict__ gm, double* red) {
  const double fl = red[2] > 0.0 ? factor * sqrt(red[0]) / sqrt(red[2]) : 0.0;
  const double fm = red[3] > 0.0 ? factor * sqrt(red[1]) / sqrt(red[3]) : 0.0;
  for (long long q = blockIdx.x * (long long)blockDim.x + threadIdx.x; q < n; q += (long long)gridDim.x * blockDim.x) {
    double a = gl[q], b = gm[q];
    if (add) {
      a = a + fl * rl[q];
      b = b + fm * rm[q];
    }
    gl[q] = a * img[q];
    gm[q] = b * img[q];
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    red[6] = add ? red[4] * fl : 0.0;
    red[7] = add ? red[5] * fm : 0.0;
    red[8] = fl;
    red[9] = fm;
  }
}

int grid_for(long long n, int threads) {
  long long b = (n + threads - 1) / threads;
  if (b > 8192) b = 8192;
  if (b < 1) b = 1;
  return (int)b;
}

}  // namespace

namespace {

// Tiles and z-chunks of the regularisation kernel: the chunk with the fewest element
// layers in sequence, rounds of blocks (REG_BLOCKS per CU run at once) times layers
// per block, the halo layer with them; of equals the longest.  At 64x64x32 elements
// (13 x 13 tiles) five layers, 1014 blocks: 57 us; four layers, 1183 blocks, 67 us.
void reg_tiles(const Geo& g, int t[3], int& tz) {
  const int R[3] = {g.rhi[0] - g.rlo[0], g.rhi[1] - g.rlo[1], g.rhi[2] - g.rlo[2]};
  for (int d = 0; d < 2; ++d) t[d] = R[d] > 0 ? (R[d] + RT - 1) / RT : 0;
  tz = R[2];
  t[2] = R[2] > 0 ? 1 : 0;
  const long long slots = 256 * REG_BLOCKS;
  long long best = -1;
  for (int c = R[2]; c >= 1; --c) {
    const int n = (R[2] + c - 1) / c;
    const long long cost = ((long long)t[0] * t[1] * n + slots - 1) / slots * (c + (n > 1));
    if (best < 0 || cost < best) { best = cost; tz = c; t[2] = n; }
  }
}

}  // namespace

size_t reg_partials_size(const Geo& g) {
  int t[3], tz;
  reg_tiles(g, t, tz);
  return 2 * REG_STREAM + 4 * (size_t)t[0] * t[1] * t[2];
}

hipError_t launch_gradient_mass(const Geo& g, double* img, double* restr, hipStream_t s) {
  hipLaunchKernelGGL(gradient_mass_kernel, dim3(grid_for(g.NN, 256)), dim3(256), 0, s, g, img, restr);
  return hipGetLastError();
}

hipError_t launch_regularization(const Geo& g, const double* zc, int tv, const double* wreg, const double* lam,
                                 const double* mu, const double* gl, const double* gm, double* rl, double* rm,
                                 double* part, double* red, hipStream_t s) {
  RegArgs A{};
  A.g = g;
  A.zc = zc;
  A.weighted = wreg != nullptr;
  if (wreg) {
    A.w_top = wreg[0];
    A.w_bot = wreg[1];
    A.w_len = wreg[2];
  }
  A.m[0] = lam;
  A.m[1] = mu;
  A.gr[0] = gl;
  A.gr[1] = gm;
  A.r[0] = rl;
  A.r[1] = rm;
  A.part = part;
  int t[3];
  reg_tiles(g, t, A.tz);
  A.ntx = t[0];
  A.nty = t[1];
  A.ntz = t[2];
  const int ntile = t[0] * t[1] * t[2];
  if (tv) reg_kernel<true><<<ntile + REG_STREAM, REG_THREADS, 0, s>>>(A);
  else reg_kernel<false><<<ntile + REG_STREAM, REG_THREADS, 0, s>>>(A);
  reg_tail_kernel<<<1, 384, 0, s>>>(ntile, gl != nullptr, part, red);
  return hipGetLastError();
}

hipError_t launch_reg_update(long long n, int add, double factor, const double* rl, const double* rm,
                             const double* img, double* gl, double* gm, double* red, hipStream_t s) {
  hipLaunchKernelGGL(reg_update_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, n, add, factor, rl, rm, img, gl, gm,
                     red);
  return hipGetLastError();
}

}  // namespace hr
