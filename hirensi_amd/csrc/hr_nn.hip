// Kernels of the learned gradient preconditioner: a 3D convolutional
// encoder-decoder evaluated and trained on the GPU.  Activations are FP32
// volumes [sample][channel][z][y][x]; convolution weights are BF16
// [cout][cin * 27] (3x3x3 taps, zero padding, tap t = 9 (dz+1) + 3 (dy+1) +
// (dx+1)) with FP32 accumulation on the matrix cores
// (v_mfma_f32_16x16x16_bf16); FP32 master weights for the optimiser.
//
// A convolution is the GEMM out[co][v] = sum_k W[co][k] X[k][v] over the
// columns v = (sample, voxel), with k = (ci, tap) and X[k][v] = in[ci][voxel +
// offset(tap)] gathered on the fly (no im2col buffer).  One wavefront computes
// 16 (co) x 16 (column) tiles; its lanes hold the MFMA operands: A row
// co0 + lane % 16, B column v0 + lane % 16, four K values 4 (lane / 16) .. +3
// each; D column lane % 16, rows 4 (lane / 16) .. +3.  Operands are rounded
// to BF16 (nearest even) as they are gathered.
//
// The tiled kernels stage the input of a block's columns in LDS, as BF16 and
// zero-padded, and read all 27 taps from there; the gather kernels read every
// tap from memory, for volumes whose rows are too long for the staging and for convolutions of
// too few channels to pay for it.  Both accumulate the same products in the same order (K
// ascending in steps of 16 for a convolution, the columns of a slice in steps of 16
// for the weight gradient), so their results agree bit for bit.

#include <hip/hip_runtime.h>
#include <cstdint>
#include <algorithm>
#include "../../include/hirensi_nn.h"
#include "hr_nn_fused.h"

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even (finite inputs)
__device__ __forceinline__ short to_bf16(float f) {
  unsigned int u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (short)(u >> 16);
}

struct Vol {
  int D, H, W;   // one sample's volume
  int NB;        // samples
  __device__ __host__ __forceinline__ int n() const { return D * H * W; }
};

// a column's voxel coordinates (fixed for a lane across the K loop)
struct Col {
  int b, x, y, z, v;   // sample, coordinates, voxel index; b < 0: padding column
};

__device__ __forceinline__ Col column(const Vol& g, int c) {
  Col r;
  const int V = g.n();
  if (c >= V * g.NB) { r.b = -1; r.x = r.y = r.z = r.v = 0; return r; }
  r.b = c / V;
  r.v = c - r.b * V;
  r.x = r.v % g.W;
  r.y = (r.v / g.W) % g.H;
  r.z = r.v / (g.W * g.H);
  return r;
}

// X[k][column] for k = ci * 27 + tap of sample c.b, zero outside the volume
__device__ __forceinline__ float gather(const float* __restrict__ in, const Vol& g, int cin, int k, const Col& c) {
  if (c.b < 0 || k >= cin * 27) return 0.0f;
  const int ci = k / 27, t = k - 27 * ci;
  const int dz = t / 9 - 1, dy = (t / 3) % 3 - 1, dx = t % 3 - 1;
  const int xx = c.x + dx, yy = c.y + dy, zz = c.z + dz;
  if (xx < 0 || yy < 0 || zz < 0 || xx >= g.W || yy >= g.H || zz >= g.D) return 0.0f;
  return in[((size_t)c.b * cin + ci) * g.n() + (xx + g.W * (yy + g.H * zz))];
}

// What follows a sum on its way out: + add, leaky ReLU, or the leaky ReLU's
// backward at its output y (null pointers, slope 1: nothing)
struct Epilogue {
  const float* add;
  const float* gate;
  float slope;
  __device__ __forceinline__ float apply(float s, size_t o) const {
    if (add) s += add[o];
    if (gate) return gate[o] > 0.0f ? s : slope * s;
    return slope == 1.0f ? s : (s > 0.0f ? s : slope * s);
  }
};

// out[b][co][v] = epilogue(bias[co] + sum_k w[co][k] X[k][(b, v)])
__global__ void __launch_bounds__(256) conv3d_gather_kernel(const float* __restrict__ in, const unsigned short* __restrict__ w,
                                                     const float* __restrict__ bias, Epilogue ep,
                                                     float* __restrict__ out, int cin, int cout, Vol g) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int V = g.n(), K = cin * 27;
  const int v0 = (blockIdx.x * 4 + wave) * 16;
  const int co0 = blockIdx.y * 16;
  if (v0 >= V * g.NB) return;                 // whole wavefront past the last column (uniform)
  const int r = lane & 15, kq = lane >> 4;
  const Col c = column(g, v0 + r);
  const int co_a = co0 + r;
  const unsigned short* __restrict__ wrow = w + (size_t)(co_a < cout ? co_a : 0) * K;
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int k0 = 0; k0 < K; k0 += 16) {
    bf16x4 a, b;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = k0 + 4 * kq + j;
      a[j] = (short)((co_a < cout && k < K) ? wrow[k] : 0);
      b[j] = to_bf16(gather(in, g, cin, k, c));
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
  }
  if (c.b >= 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int co = co0 + 4 * kq + j;
      if (co < cout) {
        const size_t o = ((size_t)c.b * cout + co) * V + c.v;
        out[o] = ep.apply(acc[j] + (bias ? bias[co] : 0.0f), o);
      }
    }
  }
}

// Weight gradient over a slice of the columns:
// part[s][co][k] = sum_{columns in slice s} dy[co][col] X[k][col]
__global__ void __launch_bounds__(256) conv3d_wgrad_gather_kernel(const float* __restrict__ in, const float* __restrict__ dy,
                                                           float* __restrict__ part, int cin, int cout, Vol g,
                                                           int cslice) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int V = g.n(), K = cin * 27, NC = V * g.NB;
  const int n0 = (blockIdx.x * 4 + wave) * 16;   // k columns of the tile
  const int co0 = blockIdx.y * 16;
  const int s = blockIdx.z;
  if (n0 >= K) return;
  const int r = lane & 15, kq = lane >> 4;
  const int cb = s * cslice, ce = min(cb + cslice, NC);
  const int co_a = co0 + r;
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int u0 = cb; u0 < ce; u0 += 16) {
    bf16x4 a, b;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int u = u0 + 4 * kq + j;
      const Col c = column(g, u < ce ? u : NC);
      a[j] = to_bf16((co_a < cout && c.b >= 0) ? dy[((size_t)c.b * cout + co_a) * V + c.v] : 0.0f);
      b[j] = to_bf16(gather(in, g, cin, n0 + r, c));
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
  }
  const int n = n0 + r;
  if (n < K) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int co = co0 + 4 * kq + j;
      if (co < cout) part[((size_t)s * cout + co) * K + n] = acc[j];
    }
  }
}

// ---------------------------------------------------------------- tiled kernels
// Columns in a padded index: voxel (b, z, y, x) of NB volumes with one zero voxel
// around each has the place P = ((b (D+2) + z + 1) (H+2) + y + 1) (W+2) + x + 1, so a tap
// is a constant offset and the padding needs no test.  A range of columns is
// staged as three segments per channel (dz = -1, 0, 1), each the range's places
// and W + 3 more on both sides; tap (dz, dy, dx) of the column at place q of the middle
// segment is element (dz + 1) seg + q + dy (W+2) + dx.
struct Div {                               // n / d for 0 <= n < 2^24 (float quotient, corrected)
  int d;
  float inv;
  __device__ __host__ explicit Div(int d_) : d(d_), inv(1.0f / (float)d_) {}
  __device__ __forceinline__ int operator()(int n) const {
    int q = (int)((float)n * inv);
    const int r = n - q * d;
    q += r >= d ? 1 : (r < 0 ? -1 : 0);
    return q;
  }
};
struct Pad {
  int D, H, W, NB, V, row, plane, vol;     // padded row, plane and volume
  Div dW, dWH, dV, drow, dplane, dvol;
  __host__ explicit Pad(const Vol& g)
      : D(g.D), H(g.H), W(g.W), NB(g.NB), V(g.n()), row(g.W + 2), plane((g.H + 2) * (g.W + 2)),
        vol((g.D + 2) * (g.H + 2) * (g.W + 2)), dW(g.W), dWH(g.W * g.H), dV(g.n()), drow(g.W + 2), dplane(plane),
        dvol(vol) {}
  // place of voxel index v counted from the first voxel of a sample (v >= V: in the
  // samples after it), relative to that sample
  __device__ __forceinline__ int place(int v) const {
    const int b = dV(v), u = v - b * V;
    const int z = dWH(u), w = u - z * W * H, y = dW(w);
    return b * vol + (z + 1) * plane + (y + 1) * row + (w - y * W) + 1;
  }
  // index of the voxel at a place relative to sample b0 within [b - b0][ch][voxel]
  // of nch channels, -1 in the padding
  __device__ __forceinline__ int voxel(int p, int b0, int nch) const {
    if (p < 0) return -1;
    const int b = dvol(p), r = p - b * vol;
    const int z = dplane(r), t = r - z * plane, y = drow(t), x = t - y * row;
    if (b0 + b >= NB || z < 1 || z > D || y < 1 || y > H || x < 1 || x > W) return -1;
    return b * nch * V + (x - 1) + W * ((y - 1) + H * (z - 1));
  }
  // bound of the places that n columns span, ranges starting at multiples of
  // `from` columns of a sample: rows, planes and (cross) samples entered inside one
  __host__ long long span(int n, int from, bool cross) const {
    auto inside = [&](int m) -> long long {
      if (from == n && m % n == 0) return 0;
      return from % m == 0 ? (n - 1) / m : (n - 1) / m + 1;
    };
    long long s = n + 2 * inside(W) + 2ll * row * inside(W * H);
    if (cross) s += 2ll * plane * ((n - 1) / V + 1);
    return s;
  }
};

constexpr int CCH = 16;                    // input channels staged at a time: 27 K steps of 16
constexpr int CK = CCH * 27;

__device__ __forceinline__ bf16x4 read4(const unsigned short* p, const int o[4]) {
  bf16x4 b;
#pragma unroll
  for (int j = 0; j < 4; ++j) b[j] = (short)p[o[j]];
  return b;
}

// One convolution: a block takes ncb columns (a range inside one sample, or whole
// samples where they are smaller) and 16 MT WM output channels; its four
// wavefronts are WM groups along the channels and 4 / WM along the columns, MT x NT
// tiles each.  K runs in steps of 16 over (channel, tap) as in the weights'
// rows; the places of a step's operands come from a table over the CK entries of
// a channel chunk.  Bounded by the staging's latency and, per step, five LDS reads a
// lane (four of two bytes); the matrix cores are 3-8 % busy (counters).  16 -> 16 channels on 8 x
// 16 x 32 x 32 voxels: 95 -> 23 us against the gather kernel, 128 -> 128 on 8 x 2 x 4 x
// 4: 91 -> 23 us (216 dependent steps in 8 chunks); with weights read 16 bytes a lane, the
// 64 -> 64 layers of a 32 x 64 x 64 volume's third level 22 -> 18 us (without any weight
// reads 16).  Operands of several steps read at once, or their places kept in
// registers, cost the second block of a CU: 20-30 % slower over a network.
template <int MT, int NT, int WM>
__global__ void __launch_bounds__(256) conv3d_tile_kernel(const float* __restrict__ in,
                                                          const unsigned short* __restrict__ w,
                                                          const float* __restrict__ bias, Epilogue ep,
                                                          float* __restrict__ out, int cin, int cout, Pad pd, int ncb,
                                                          int segmax) {
  constexpr int WN = 4 / WM;
  extern __shared__ int smem[];
  int* const sOff = smem;                                    // [CK] element offset of a K entry
  int* const sPos = smem + CK;                               // [3 segmax] voxel of a staged place, -1: zero
  unsigned short* const sX = (unsigned short*)(sPos + 3 * segmax);   // [CCH][3 seg]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave % WM, wn = wave / WM;
  const int V = pd.V, K = cin * 27;
  // nc columns from voxel v0 of sample b0 on
  int b0, v0, nc;
  if (V >= ncb) {
    const int bps = (V + ncb - 1) / ncb;
    b0 = blockIdx.x / bps;
    v0 = (blockIdx.x - b0 * bps) * ncb;
    nc = min(ncb, V - v0);
  } else {
    const int spb = ncb / V;
    b0 = (int)blockIdx.x * spb;
    v0 = 0;
    nc = min(spb, pd.NB - b0) * V;
  }
  const int p0 = pd.place(v0), seg = pd.place(v0 + nc - 1) - p0 + 1 + 2 * (pd.row + 1);
  for (int t = tid; t < 3 * seg; t += 256) {
    const int dz = t >= 2 * seg ? 2 : (t >= seg ? 1 : 0), q = t - dz * seg;
    sPos[t] = pd.voxel(p0 + q - (pd.row + 1) + (dz - 1) * pd.plane, b0, cin);
  }
  for (int k = tid; k < CK; k += 256) {
    const int ci = k / 27, t = k - 27 * ci;
    sOff[k] = (3 * ci + t / 9) * seg + ((t / 3) % 3 - 1) * pd.row + t % 3 - 1;
  }
  const int r = lane & 15, kq = lane >> 4;
  int q[NT];                               // place of the lane's columns in the middle segment
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int c = (wn * NT + n) * 16 + r;
    q[n] = pd.place(v0 + (c < nc ? c : 0)) - p0 + pd.row + 1;
  }
  const int co0 = ((int)blockIdx.y * WM + wm) * 16 * MT;
  const unsigned short* wrow[MT];
  bool wok[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int co = co0 + 16 * m + r;
    wok[m] = co < cout;
    wrow[m] = w + (size_t)(wok[m] ? co : 0) * K;
  }
  const bool aligned = (K & 3) == 0 && ((size_t)w & 7) == 0;   // four weights of a lane: one 8-byte load
  f32x4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // the chunk's channels of one staged place, and their store
  auto fetch = [&](int t, int ci0, float* f) {
    const int v = sPos[t], nch = min(CCH, cin - ci0);
    const float* __restrict__ src = in + ((size_t)b0 * cin + ci0) * V + (v < 0 ? 0 : v);
#pragma unroll
    for (int c = 0; c < CCH; ++c) f[c] = (v >= 0 && c < nch) ? src[(size_t)c * V] : 0.0f;
  };
  auto stage = [&](int t, const float* f) {
#pragma unroll
    for (int c = 0; c < CCH; ++c) sX[c * 3 * seg + t] = (unsigned short)to_bf16(f[c]);
  };
  // one place a thread: the next chunk's values are in flight while this one is computed
  const bool ahead = 3 * seg <= 256;
  float f0[CCH];
  // the weights of a whole chunk are loaded before they are needed: a chunk ahead
  // with one channel tile, else before the staging
  constexpr int WU2 = (CK / 16 + 1) / 2;
  bf16x4 a[2 * WU2][MT];
  // rows that start at 16 bytes are read 16 bytes a lane, the four lanes of a row 64 in
  // a row, for two steps at a time (half the requests, each a whole sector pair); `deal`
  // then hands every lane the four weights of each step
  const bool wide = MT == 1 && (cin & 7) == 0 && ((size_t)w & 15) == 0;
  auto weights = [&](int ci0) {
    if (wide) {
#pragma unroll
      for (int u = 0; u < WU2; ++u) {
        // the last pair is one step: its upper lanes read the lower ones' piece again
        const int piece = 4 * u + (2 * u + 1 < CK / 16 ? kq : (kq & 1));
        const uint4 q = *reinterpret_cast<const uint4*>(wrow[0] + ci0 * 27 + 8 * piece);
        a[2 * u][0] = __builtin_bit_cast(bf16x4, make_uint2(q.x, q.y));
        a[2 * u + 1][0] = __builtin_bit_cast(bf16x4, make_uint2(q.z, q.w));
      }
      return;
    }
#pragma unroll
    for (int s = 0; s < CK / 16; ++s)
#pragma unroll
      for (int m = 0; m < MT; ++m) a[s][m] = *reinterpret_cast<const bf16x4*>(wrow[m] + ci0 * 27 + 16 * s + 4 * kq);
  };
  // lane group kq holds weights 32 u + 8 kq .. + 7 and needs 32 u + 4 kq .. + 3 (step 2 u)
  // and 32 u + 16 + 4 kq .. + 3 (step 2 u + 1): exchange the piece's halves with
  // lane bit 4, then with lane bit 5
  auto deal = [&](bf16x4* an) {
    if constexpr (MT == 1) {
#pragma unroll
      for (int u = 0; u < WU2; ++u) {
        const uint2 lo = __builtin_bit_cast(uint2, an[2 * u]), hi = __builtin_bit_cast(uint2, an[2 * u + 1]);
        unsigned x[2] = {lo.x, lo.y}, y[2] = {hi.x, hi.y};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          auto t = __builtin_amdgcn_permlane16_swap(x[h], y[h], false, false);
          t = __builtin_amdgcn_permlane32_swap(t[0], t[1], false, false);
          x[h] = t[0];
          y[h] = t[1];
        }
        an[2 * u] = __builtin_bit_cast(bf16x4, make_uint2(x[0], x[1]));
        an[2 * u + 1] = __builtin_bit_cast(bf16x4, make_uint2(y[0], y[1]));
      }
    }
  };
  if (MT == 1 && aligned && cin >= CCH) weights(0);
  __syncthreads();
  if (ahead && tid < 3 * seg) fetch(tid, 0, f0);
  for (int ci0 = 0; ci0 < cin; ci0 += CCH) {
    const int nch = min(CCH, cin - ci0), kc = nch * 27, kbase = ci0 * 27;
    const bool full = nch == CCH && aligned;
    if (MT > 1 && full) weights(ci0);
    if (ahead) {
      if (tid < 3 * seg) stage(tid, f0);
    } else {
      int t = tid;
      for (; t + 256 < 3 * seg; t += 512) {
        float f[2][CCH];
        fetch(t, ci0, f[0]);
        fetch(t + 256, ci0, f[1]);
        stage(t, f[0]);
        stage(t + 256, f[1]);
      }
      if (t < 3 * seg) {
        float f[CCH];
        fetch(t, ci0, f);
        stage(t, f);
      }
    }
    __syncthreads();
    if (ahead && ci0 + CCH < cin && tid < 3 * seg) fetch(tid, ci0 + CCH, f0);
    if (full) {
      bf16x4 an[2 * WU2];                    // this chunk's weights, the next one's on their way
      if constexpr (MT == 1) {
#pragma unroll
        for (int s = 0; s < 2 * WU2; ++s) an[s] = a[s][0];
        if (wide) deal(an);
        if (ci0 + 2 * CCH <= cin) weights(ci0 + CCH);
      }
#pragma unroll
      for (int s = 0; s < CK / 16; ++s) {
        int o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = sOff[16 * s + 4 * kq + j];
        bf16x4 am[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) am[m] = wok[m] ? (MT == 1 ? an[s] : a[s][m]) : bf16x4{0, 0, 0, 0};
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const bf16x4 b = read4(sX + q[n], o);
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(am[m], b, acc[m][n], 0, 0, 0);
        }
      }
    } else {
      for (int k0 = 0; k0 < kc; k0 += 16) {
        const int kk = k0 + 4 * kq;
        bf16x4 am[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int j = 0; j < 4; ++j) am[m][j] = (short)((wok[m] && kk + j < kc) ? wrow[m][kbase + kk + j] : 0);
        int o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = sOff[min(kk + j, kc - 1)];
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          bf16x4 b = read4(sX + q[n], o);
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (kk + j >= kc) b[j] = 0;      // entries past the last channel are zero
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(am[m], b, acc[m][n], 0, 0, 0);
        }
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int c = (wn * NT + n) * 16 + r;
    if (c >= nc) continue;
    const int b = pd.dV(v0 + c), v = v0 + c - b * V;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int co = co0 + 16 * m + 4 * kq + j;
        if (co < cout) {
          const size_t o = ((size_t)(b0 + b) * cout + co) * V + v;
          out[o] = ep.apply(acc[m][n][j] + (bias ? bias[co] : 0.0f), o);
        }
      }
  }
}

// db[co] = sum over samples and voxels of dy[b][co][v]: 256 chains over the voxels,
// sixteen loads in flight each, then a tree
__device__ __forceinline__ void bias_grad(const float* __restrict__ dy, int co, int cout, const Vol& g,
                                          float* __restrict__ db, float* __restrict__ red) {
  const int V = g.n(), tid = threadIdx.x;
  float c = 0.0f;
  for (int b = 0; b < g.NB; ++b) {
    const float* __restrict__ p = dy + ((size_t)b * cout + co) * V;
    int v = tid;
    for (; v + 15 * 256 < V; v += 16 * 256) {
      float f[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) f[u] = p[v + 256 * u];
#pragma unroll
      for (int u = 0; u < 16; ++u) c += f[u];
    }
    for (; v < V; v += 256) c += p[v];
  }
  red[tid] = c;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (tid < s) red[tid] += red[tid + s];
    __syncthreads();
  }
  if (tid == 0) db[co] = red[0];
}

// Weight gradient over a slice of the columns (the K dimension, in steps of 16):
// a wavefront takes one input channel, whose 27 taps are two 16-wide column
// tiles, against all output channels (16 MT of them); a block's four channels and the
// output gradient's rows are staged together, WU columns at a time.  The blocks
// past the first nx of a row sum the bias gradient, beside the others.  16 -> 16
// channels on 8 x 16 x 32 x 32 voxels: 95 -> 35 us against the gather kernel.
constexpr int WU = 256, WCH = 4, WROW = WU + 8;   // row stride: 16 rows on different banks
template <int MT>
__global__ void __launch_bounds__(256) conv3d_wgrad_tile_kernel(const float* __restrict__ in,
                                                                const float* __restrict__ dy,
                                                                float* __restrict__ part, float* __restrict__ db,
                                                                int cin, int cout, Vol g, Pad pd, int cslice, int nx,
                                                                int segmax) {
  extern __shared__ int smem[];
  if ((int)blockIdx.x >= nx) {
    const int co = ((int)blockIdx.x - nx) + ((int)gridDim.x - nx) * ((int)blockIdx.y + (int)gridDim.y * (int)blockIdx.z);
    if (co < cout) bias_grad(dy, co, cout, g, db, (float*)smem);
    return;
  }
  unsigned short* const sY = (unsigned short*)smem;           // [16 MT][WROW]
  unsigned short* const sQ = sY + 16 * MT * WROW;             // [WU] place of a column
  unsigned short* const sX = sQ + WU;                         // [WCH][3 seg]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int V = pd.V, K = cin * 27, NC = V * g.NB;
  const int ci0 = blockIdx.x * WCH, ci = ci0 + wave;
  const int co0 = blockIdx.y * 16 * MT;
  const int s = blockIdx.z;
  const int cb = s * cslice, ce = min(cb + cslice, NC);
  const int r = lane & 15, kq = lane >> 4;
  f32x4 acc[MT][2];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m][0] = acc[m][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int u0 = cb; u0 < ce;) {
    // a chunk ends with its sample where a step of 16 columns cannot straddle two
    int n = min(WU, ce - u0);
    const int b0 = u0 / V, v0 = u0 - b0 * V;
    if ((V & 15) == 0) n = min(n, V - v0);
    const int p0 = pd.place(v0), seg = pd.place(v0 + n - 1) - p0 + 1 + 2 * (pd.row + 1);
    __syncthreads();
    // the output gradient's rows, one column a thread
    const bool ok = tid < n;
    const int cbs = pd.dV(v0 + (ok ? tid : 0)), cv = v0 + (ok ? tid : 0) - cbs * V;
    sQ[tid] = (unsigned short)(pd.place(v0 + (ok ? tid : 0)) - p0 + pd.row + 1);
    const float* __restrict__ ysrc = dy + ((size_t)(b0 + cbs) * cout + co0) * V + cv;
#pragma unroll
    for (int m0 = 0; m0 < 16 * MT; m0 += 16) {
      float f[16];
#pragma unroll
      for (int m = 0; m < 16; ++m) f[m] = (ok && co0 + m0 + m < cout) ? ysrc[(size_t)(m0 + m) * V] : 0.0f;
#pragma unroll
      for (int m = 0; m < 16; ++m) sY[(m0 + m) * WROW + tid] = (unsigned short)to_bf16(f[m]);
    }
    for (int t0 = tid; t0 < 3 * seg; t0 += 4 * 256) {   // four places, sixteen loads in flight
      float f[4][WCH];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = t0 + 256 * u;
        const int dz = t >= 2 * seg ? 2 : (t >= seg ? 1 : 0), q = t - dz * seg;
        const int v = t < 3 * seg ? pd.voxel(p0 + q - (pd.row + 1) + (dz - 1) * pd.plane, b0, cin) : -1;
#pragma unroll
        for (int c = 0; c < WCH; ++c)
          f[u][c] = (v >= 0 && ci0 + c < cin) ? in[((size_t)b0 * cin + ci0 + c) * V + v] : 0.0f;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = t0 + 256 * u;
        if (t < 3 * seg) {
#pragma unroll
          for (int c = 0; c < WCH; ++c) sX[c * 3 * segmax + t] = (unsigned short)to_bf16(f[u][c]);
        }
      }
    }
    __syncthreads();
    if (ci < cin) {
      const unsigned short* const X = sX + wave * 3 * segmax;
      int off[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int t = min(16 * h + r, 26);
        off[h] = (t / 9) * seg + ((t / 3) % 3 - 1) * pd.row + t % 3 - 1;
      }
      // four whole steps at a time: their places, then their operands in flight together
      constexpr int G = 4;
      int k0 = 0;
      for (; k0 + 16 * G <= n; k0 += 16 * G) {
        bf16x4 a[G][MT];
        ushort4 q4[G];
        short x[G][2][4];
#pragma unroll
        for (int s = 0; s < G; ++s) q4[s] = *reinterpret_cast<const ushort4*>(sQ + k0 + 16 * s + 4 * kq);
#pragma unroll
        for (int s = 0; s < G; ++s)
#pragma unroll
          for (int m = 0; m < MT; ++m)
            a[s][m] = *reinterpret_cast<const bf16x4*>(sY + (16 * m + r) * WROW + k0 + 16 * s + 4 * kq);
#pragma unroll
        for (int s = 0; s < G; ++s)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const unsigned short* const Xh = X + off[h];
            x[s][h][0] = (short)Xh[q4[s].x];
            x[s][h][1] = (short)Xh[q4[s].y];
            x[s][h][2] = (short)Xh[q4[s].z];
            x[s][h][3] = (short)Xh[q4[s].w];
          }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < G; ++s)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const bf16x4 b = {x[s][h][0], x[s][h][1], x[s][h][2], x[s][h][3]};
#pragma unroll
            for (int m = 0; m < MT; ++m)
              acc[m][h] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[s][m], b, acc[m][h], 0, 0, 0);
          }
      }
      for (; k0 < n; k0 += 16) {
        const int kk = k0 + 4 * kq;
        bf16x4 a[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) a[m] = *reinterpret_cast<const bf16x4*>(sY + (16 * m + r) * WROW + kk);
        const ushort4 q4 = *reinterpret_cast<const ushort4*>(sQ + kk);
        const int o[4] = {q4.x, q4.y, q4.z, q4.w};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          bf16x4 b = read4(X + off[h], o);
          if (k0 + 16 > n) {                // columns past the slice are zero
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (kk + j >= n) b[j] = 0;
          }
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[m][h] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[m], b, acc[m][h], 0, 0, 0);
        }
      }
    }
    u0 += n;
  }
  if (ci >= cin) return;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int t = 16 * h + r;
    if (t >= 27) continue;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int co = co0 + 16 * m + 4 * kq + j;
        if (co < cout) part[((size_t)s * cout + co) * K + ci * 27 + t] = acc[m][h][j];
      }
  }
}

// dw[i] = sum_s part[s][i], in slice order
__global__ void __launch_bounds__(64) reduce_slices_kernel(const float* __restrict__ part, int nslice, int n,
                                                           float* __restrict__ dw) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  if (i >= n) return;
  float c = 0.0f;
  int s = 0;
  for (; s + 16 <= nslice; s += 16) {       // sixteen loads in flight, added in order
    float f[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) f[u] = part[(size_t)(s + u) * n + i];
#pragma unroll
    for (int u = 0; u < 16; ++u) c += f[u];
  }
  for (; s < nslice; ++s) c += part[(size_t)s * n + i];
  dw[i] = c;
}

__global__ void __launch_bounds__(256) bias_grad_kernel(const float* __restrict__ dy, int cout, Vol g,
                                                        float* __restrict__ db) {
  __shared__ float red[256];
  bias_grad(dy, blockIdx.x, cout, g, db, red);
}

// wt[ci][co * 27 + (26 - t)] = w[co][ci * 27 + t]: the weights of the adjoint
// (input-gradient) convolution, whose taps are the mirrored offsets
__global__ void transpose_weights_kernel(const unsigned short* __restrict__ w, unsigned short* __restrict__ wt, int cin,
                                         int cout) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= cin * cout * 27) return;
  const int t = i % 27, ci = (i / 27) % cin, co = i / (27 * cin);
  wt[((size_t)ci * cout + co) * 27 + (26 - t)] = w[i];
}

// the same for every layer of a network in one launch
constexpr int TL_MAX = 32;
struct LayerTable {
  int n, cin[TL_MAX], cout[TL_MAX], start[TL_MAX + 1];    // weights of layer l: [start[l], start[l + 1])
};
__global__ void transpose_layers_kernel(const unsigned short* __restrict__ w, unsigned short* __restrict__ wt,
                                        LayerTable T) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= T.start[T.n]) return;
  int l = 0;
  while (g >= T.start[l + 1]) ++l;
  const int i = g - T.start[l], cin = T.cin[l], cout = T.cout[l];
  const int t = i % 27, ci = (i / 27) % cin, co = i / (27 * cin);
  wt[T.start[l] + (ci * cout + co) * 27 + (26 - t)] = w[g];
}

__global__ void leaky_relu_kernel(float* __restrict__ x, size_t n, float slope) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i < n) {
    const float v = x[i];
    x[i] = v > 0.0f ? v : slope * v;
  }
}

// dy *= f'(x) for y = f(x) the activation output (y > 0 exactly when x > 0)
__global__ void leaky_relu_grad_kernel(const float* __restrict__ y, float* __restrict__ dy, size_t n, float slope) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i < n) dy[i] = y[i] > 0.0f ? dy[i] : slope * dy[i];
}

// 2x2x2 average pooling of C volumes (D, H, W) (even sizes)
__global__ void avgpool2_kernel(const float* __restrict__ in, float* __restrict__ out, long long C, int D, int H,
                                int W) {
  const int Ho = H / 2, Wo = W / 2, Vo = (D / 2) * Ho * Wo;
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i >= (size_t)C * Vo) return;
  const size_t c = i / Vo;
  const int v = (int)(i - c * Vo);
  const int x = v % Wo, y = (v / Wo) % Ho, z = v / (Wo * Ho);
  const float* __restrict__ p = in + c * (size_t)(D * H * W);
  float s = 0.0f;
  for (int d = 0; d < 8; ++d) s += p[(2 * x + (d & 1)) + W * ((2 * y + ((d >> 1) & 1)) + H * (2 * z + (d >> 2)))];
  out[i] = 0.125f * s;
}

// pooling backward: dx[fine] = dy[coarse] / 8 (added to dx when accumulate)
// gate: the activation output whose backward follows (null: none)
__global__ void avgpool2_grad_kernel(const float* __restrict__ dy, float* __restrict__ dx, long long C, int D, int H,
                                     int W, int accumulate, const float* __restrict__ gate, float slope) {
  const int V = D * H * W, Ho = H / 2, Wo = W / 2, Vo = V / 8;
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i >= (size_t)C * V) return;
  const size_t c = i / V;
  const int v = (int)(i - c * V);
  const int x = v % W, y = (v / W) % H, z = v / (W * H);
  const float d = 0.125f * dy[c * Vo + (x / 2) + Wo * ((y / 2) + Ho * (z / 2))];
  const float s = accumulate ? dx[i] + d : d;
  dx[i] = gate && !(gate[i] > 0.0f) ? slope * s : s;
}

// nearest 2x upsampling of C coarse volumes to (D, H, W)
__global__ void upsample2_kernel(const float* __restrict__ in, float* __restrict__ out, long long C, int D, int H,
                                 int W) {
  const int V = D * H * W, Ho = H / 2, Wo = W / 2, Vo = V / 8;
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i >= (size_t)C * V) return;
  const size_t c = i / V;
  const int v = (int)(i - c * V);
  const int x = v % W, y = (v / W) % H, z = v / (W * H);
  out[i] = in[c * Vo + (x / 2) + Wo * ((y / 2) + Ho * (z / 2))];
}

// upsampling backward: dcoarse = sum of the 8 fine values
__global__ void upsample2_grad_kernel(const float* __restrict__ dy, float* __restrict__ dx, long long C, int D, int H,
                                      int W, const float* __restrict__ gate, float slope) {
  const int Ho = H / 2, Wo = W / 2, Vo = (D / 2) * Ho * Wo;
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i >= (size_t)C * Vo) return;
  const size_t c = i / Vo;
  const int v = (int)(i - c * Vo);
  const int x = v % Wo, y = (v / Wo) % Ho, z = v / (Wo * Ho);
  const float* __restrict__ p = dy + c * (size_t)(D * H * W);
  float s = 0.0f;
  for (int d = 0; d < 8; ++d) s += p[(2 * x + (d & 1)) + W * ((2 * y + ((d >> 1) & 1)) + H * (2 * z + (d >> 2)))];
  dx[i] = gate && !(gate[i] > 0.0f) ? slope * s : s;
}

constexpr int MSE_BLOCKS = 256;

// squared-error partial sums per block; grad = 2 (y - t) / n
__global__ void __launch_bounds__(256) mse_kernel(const float* __restrict__ y, const float* __restrict__ t, size_t n,
                                                  float* __restrict__ grad, float* __restrict__ part) {
  __shared__ float red[256];
  float c = 0.0f;
  for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += (size_t)256 * gridDim.x) {
    const float d = y[i] - t[i];
    if (grad) grad[i] = 2.0f * d / (float)n;
    c += d * d;
  }
  red[threadIdx.x] = c;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// loss = sum of the block partials (in block order) / n
__global__ void loss_finish_kernel(const float* __restrict__ part, int nb, size_t n, float* __restrict__ loss) {
  __shared__ float p[MSE_BLOCKS];
  for (int b = threadIdx.x; b < nb; b += 64) p[b] = part[b];
  __syncthreads();
  if (threadIdx.x == 0) {
    float c = 0.0f;
    for (int b = 0; b < nb; ++b) c += p[b];
    loss[0] = c / (float)n;
  }
}

// Adam step on FP32 master weights, then their BF16 copy (wb null: biases)
__global__ void adam_kernel(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                            float* __restrict__ v, unsigned short* __restrict__ wb, size_t n, float lr, float b1,
                            float b2, float eps, float c1, float c2) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
  if (wb) wb[i] = (unsigned short)to_bf16(wi);
}

__global__ void to_bf16_kernel(const float* __restrict__ w, unsigned short* __restrict__ wb, size_t n) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i < n) wb[i] = (unsigned short)to_bf16(w[i]);
}

inline unsigned nblocks(size_t n, unsigned b = 256) { return (unsigned)((n + b - 1) / b); }

bool bad_vol(int D, int H, int W, int NB) { return D < 1 || H < 1 || W < 1 || NB < 1; }
bool odd(int D, int H, int W) { return (D | H | W) & 1; }

// ------------------------------------------------------------ tiled launches
constexpr size_t LDS_LIMIT = 64 * 1024;

// What became of a tile: launched, its rows too long for the staging, or the gather
// kernel is the faster one, or the only one whose blocks (64 columns each) one launch holds
enum class Tile { DONE, TOO_LONG, GATHER };

// Whether a tile beats the gather kernel.  With whole chunks of 16 channels and four
// weights a load it always does (714 random shapes: 1.1-10 times).  A chunk of fewer
// channels is staged at the cost of a whole one, and rows of weights that are no multiple
// of 8 bytes are read weight by weight; what the tile saves is K's gathers.  So the K
// steps that a chunk brings are held against a bound that grows with the places staged per
// column, less where the blocks do not fill the GPU twice and the staging's loads are
// hidden worse by others of their kind than the gathers' chain.  1318 random shapes of such
// channels, rows of 2-280: the tile runs at 0.22-3.4 times the gather kernel's rate, where it
// is taken at 0.80-3.4, nine in ten above 1; where it is not, at most 1.2.  One channel on
// 2 x 32 x 64 x 64 voxels, the network's first layer: 20 us gathered, 29 tiled; 12 -> 24
// channels there 227 and 89; 8 -> 16 on 2 x 8 x 33 x 100 26 and 28.
bool tile_pays(int cin, int cout, const unsigned short* w, double places, long long blocks, double least, double slope) {
  if (cin >= CCH && (cin & 3) == 0 && ((size_t)w & 7) == 0) return true;
  const int steps = (27 * cin + 15) / 16, chunks = (cin + CCH - 1) / CCH;
  if (blocks < 512) slope *= 0.3;
  if (cout <= 4) slope *= 0.5;             // most lanes have no weights to read
  return steps >= chunks * (least + slope * std::max(0.0, places - 10.0));
}

template <int MT, int NT, int WM>
Tile launch_conv(const float* in, const unsigned short* w, const float* bias, const Epilogue& ep, float* out, int cin,
                 int cout, const Vol& g, hipStream_t st, double least, double slope) {
  constexpr int NCB = 16 * NT * (4 / WM), COB = 16 * MT * WM;
  const Pad pd(g);
  const bool whole = pd.V < NCB;             // blocks of whole samples
  const int spb = whole ? NCB / pd.V : 1;
  long long span = whole ? (long long)spb * pd.vol : pd.span(NCB, NCB, false);
  const long long seg = span + 2 * (pd.row + 1);
  const size_t lds = CK * sizeof(int) + 3 * (size_t)seg * (sizeof(int) + CCH * sizeof(short));
  if (lds > LDS_LIMIT) return Tile::TOO_LONG;
  const long long nblk = whole ? (g.NB + spb - 1) / spb : (long long)g.NB * ((pd.V + NCB - 1) / NCB);
  const int ny = (cout + COB - 1) / COB;
  // 2^24 blocks are 2^32 threads, where a launch wraps without an error
  if (nblk >= 1 << 24 || !tile_pays(cin, cout, w, 3.0 * seg / (whole ? spb * pd.V : NCB), nblk * ny, least, slope))
    return Tile::GATHER;
  const dim3 grid((unsigned)nblk, (unsigned)ny);
  conv3d_tile_kernel<MT, NT, WM><<<grid, 256, lds, st>>>(in, w, bias, ep, out, cin, cout, pd, NCB, (int)seg);
  return Tile::DONE;
}

// The tile by output channels, then by whether the larger column range still
// gives every CU a block (256).  Wider tiles reuse a lane's LDS reads: more output
// channels per wavefront first (each read feeds MT matrix operations), more
// columns where there are few.  False: the gather kernel's.
bool conv_tiled(const float* in, const unsigned short* w, const float* bias, const Epilogue& ep, float* out, int cin,
                int cout, const Vol& g, hipStream_t st) {
  if (cin < 2) return false;               // fewer K steps than any tile's bound below
  const Pad pd(g);
  const long long V = g.n(), ncol = V * g.NB;
  if (V * cin * 2 >= (1ll << 31) || pd.vol >= 1 << 23) return false;   // 32-bit voxel offsets, 24-bit places
  const int cot = (cout + 15) / 16;
  const long long y = (cot + 3) / 4;
  Tile t = Tile::TOO_LONG;
  if (cot <= 2) {
    const double least = cout <= 4 ? 4.0 : (cot == 1 ? 7.0 : 6.0);
    if (ncol >= (cot == 1 ? 256 * 256 : 256 * 128)) t = launch_conv<1, 4, 1>(in, w, bias, ep, out, cin, cout, g, st, least, 1.0);
    if (t != Tile::TOO_LONG) return t == Tile::DONE;
    if (cot == 1) return launch_conv<1, 1, 1>(in, w, bias, ep, out, cin, cout, g, st, 8.0, 1.0) == Tile::DONE;
    return launch_conv<1, 1, 2>(in, w, bias, ep, out, cin, cout, g, st, 7.0, 0.8) == Tile::DONE;
  }
  if (ncol * y >= 64 * 256) t = launch_conv<4, 1, 1>(in, w, bias, ep, out, cin, cout, g, st, 22.0, 0.5);
  if (t == Tile::TOO_LONG && ncol * y >= 32 * 256) t = launch_conv<2, 1, 2>(in, w, bias, ep, out, cin, cout, g, st, 9.0, 1.2);
  if (t == Tile::TOO_LONG) t = launch_conv<1, 1, 4>(in, w, bias, ep, out, cin, cout, g, st, 6.0, 0.1);
  return t == Tile::DONE;
}

bool wgrad_tiled(const float* in, const float* dy, float* part, float* db, int cin, int cout, const Vol& g, int cslice,
                 int ns, hipStream_t st) {
  const Pad pd(g);
  const long long V = pd.V;
  if (V * std::max(cin, cout) * 2 >= (1ll << 31) || pd.vol >= 1 << 23) return false;
  // a step of 16 columns straddles samples where their size is no multiple of 16
  const bool cross = (V & 15) != 0 && g.NB > 1;
  const long long seg = pd.span(WU, cross ? 1 : 16, cross) + 2 * (pd.row + 1);
  const int MT = cout > 32 ? 4 : (cout > 16 ? 2 : 1);
  const size_t lds = sizeof(short) * ((size_t)16 * MT * WROW + WU + (size_t)WCH * 3 * seg);
  if (lds > LDS_LIMIT || seg >= 65536) return false;
  const unsigned nx = (unsigned)((cin + WCH - 1) / WCH), ny = (unsigned)((cout + 16 * MT - 1) / (16 * MT));
  // While few blocks are at work a slice's chunks come one after another, each as long as
  // five steps of the gather kernel (three with half the rows of the output gradient, where
  // a single chunk is as fast), so those that short slices or samples of few voxels
  // cut shorter are left to it: 24 -> 64 channels on 8 x 48 voxels 37 us gathered, 49 tiled;
  // 5 -> 64 on 32 voxels 7.0 and 10.8; 40 -> 32 on 8 x 16 15 and 30; but with 30 x 42
  // blocks, 120 -> 64 on 8 x 336, 116 and 40.
  const long long most = (V & 15) == 0 ? std::min<long long>(V, WU) : WU;
  const long long chunks = (cslice + most - 1) / most + ((V & 15) == 0 && g.NB > 1 && cslice % V && V % cslice ? 1 : 0);
  const long long steps = cslice / 16;
  if ((long long)nx * ny * ns < 32 && (MT == 4 ? steps < 5 * chunks : MT == 2 && chunks > 1 && steps < 3 * chunks)) return false;
  const unsigned rows = ny * (unsigned)ns;
  const dim3 grid(nx + (db ? ((unsigned)cout + rows - 1) / rows : 0), ny, (unsigned)ns);
  if (ns > 65535) return false;
  const size_t l = std::max(lds, (size_t)1024);
#define HR_WGRAD(M) conv3d_wgrad_tile_kernel<M><<<grid, 256, l, st>>>(in, dy, part, db, cin, cout, g, pd, cslice, (int)nx, (int)seg)
  if (MT == 4) HR_WGRAD(4);
  else if (MT == 2) HR_WGRAD(2);
  else HR_WGRAD(1);
#undef HR_WGRAD
  return true;
}

}  // namespace

// ------------------------------------------------------------------ C ABI
// Every entry point queues its kernels on `stream` (a hipStream_t, 0 for the
// null stream) and returns 0 or a nonzero error code; pointers are device
// pointers.  Volumes are NB samples of (D, H, W), x fastest.
extern "C" {

int hr_nn_conv3d(const float* in, const unsigned short* w, const float* bias, float* out, int cin, int cout, int NB,
                 int D, int H, int W, int accumulate, void* stream) {
  return hr_nn_conv3d_fused(in, w, bias, accumulate ? out : nullptr, nullptr, 1.0f, out, cin, cout, NB, D, H, W, stream);
}

int hr_nn_conv3d_fused(const float* in, const unsigned short* w, const float* bias, const float* add,
                       const float* gate, float slope, float* out, int cin, int cout, int NB, int D, int H, int W,
                       void* stream) {
  if (!in || !w || !out || cin < 1 || cout < 1 || bad_vol(D, H, W, NB)) return 1;
  const Vol g{D, H, W, NB};
  const long long ncol = (long long)g.n() * NB;
  if (ncol >= (1ll << 31) - 64) return 1;
  const Epilogue ep{add, gate, slope};
  const hipStream_t st = (hipStream_t)stream;
  if (conv_tiled(in, w, bias, ep, out, cin, cout, g, st)) return (int)hipGetLastError();
  const dim3 grid((unsigned)((ncol + 63) / 64), (unsigned)((cout + 15) / 16));
  hipLaunchKernelGGL(conv3d_gather_kernel, grid, dim3(256), 0, st, in, w, bias, ep, out, cin, cout, g);
  return (int)hipGetLastError();
}

// part: nslice * cout * cin * 27 floats of scratch; db may be null
int hr_nn_conv3d_wgrad(const float* in, const float* dy, float* part, int nslice, float* dw, float* db, int cin,
                       int cout, int NB, int D, int H, int W, void* stream) {
  if (!in || !dy || !part || !dw || nslice < 1 || cin < 1 || cout < 1 || bad_vol(D, H, W, NB)) return 1;
  const Vol g{D, H, W, NB};
  const long long ncol = (long long)g.n() * NB;
  if (ncol >= (1ll << 31) - 64) return 1;
  const int K = cin * 27;
  const int cslice = (int)(((ncol + nslice - 1) / nslice + 15) / 16 * 16);
  const int ns = (int)((ncol + cslice - 1) / cslice);
  const hipStream_t st = (hipStream_t)stream;
  if (!wgrad_tiled(in, dy, part, db, cin, cout, g, cslice, ns, st)) {
    const dim3 grid((unsigned)((K + 63) / 64), (unsigned)((cout + 15) / 16), (unsigned)ns);
    hipLaunchKernelGGL(conv3d_wgrad_gather_kernel, grid, dim3(256), 0, st, in, dy, part, cin, cout, g, cslice);
    if (db) hipLaunchKernelGGL(bias_grad_kernel, dim3(cout), dim3(256), 0, st, dy, cout, g, db);
  }
  hipLaunchKernelGGL(reduce_slices_kernel, dim3(nblocks((size_t)cout * K, 64)), dim3(64), 0, st, part, ns, cout * K, dw);
  return (int)hipGetLastError();
}

int hr_nn_transpose_weights(const unsigned short* w, unsigned short* wt, int cin, int cout, void* stream) {
  if (!w || !wt || cin < 1 || cout < 1) return 1;
  hipLaunchKernelGGL(transpose_weights_kernel, dim3(nblocks((size_t)cin * cout * 27)), dim3(256), 0,
                     (hipStream_t)stream, w, wt, cin, cout);
  return (int)hipGetLastError();
}

int hr_nn_transpose_layers(const unsigned short* w, unsigned short* wt, int nlayer, const int* cin, const int* cout,
                           void* stream) {
  if (!w || !wt || !cin || !cout || nlayer < 1 || nlayer > TL_MAX) return 1;
  LayerTable T;
  T.n = nlayer;
  long long tot = 0;
  for (int l = 0; l < nlayer; ++l) {
    if (cin[l] < 1 || cout[l] < 1) return 1;
    T.cin[l] = cin[l];
    T.cout[l] = cout[l];
    T.start[l] = (int)tot;
    tot += 27ll * cin[l] * cout[l];
    if (tot >= (1ll << 31) - 256) return 1;
  }
  T.start[nlayer] = (int)tot;
  hipLaunchKernelGGL(transpose_layers_kernel, dim3(nblocks((size_t)tot)), dim3(256), 0, (hipStream_t)stream, w, wt, T);
  return (int)hipGetLastError();
}

int hr_nn_leaky_relu(float* x, long long n, float slope, void* stream) {
  if (!x || n < 0) return 1;
  if (n == 0) return 0;
  hipLaunchKernelGGL(leaky_relu_kernel, dim3(nblocks((size_t)n)), dim3(256), 0, (hipStream_t)stream, x, (size_t)n,
                     slope);
  return (int)hipGetLastError();
}

int hr_nn_leaky_relu_grad(const float* y, float* dy, long long n, float slope, void* stream) {
  if (!y || !dy || n < 0) return 1;
  if (n == 0) return 0;
  hipLaunchKernelGGL(leaky_relu_grad_kernel, dim3(nblocks((size_t)n)), dim3(256), 0, (hipStream_t)stream, y, dy,
                     (size_t)n, slope);
  return (int)hipGetLastError();
}

// C = samples x channels volumes of the fine size (D, H, W)
int hr_nn_avgpool2(const float* in, float* out, long long C, int D, int H, int W, void* stream) {
  if (!in || !out || C < 1 || bad_vol(D, H, W, 1) || odd(D, H, W)) return 1;
  hipLaunchKernelGGL(avgpool2_kernel, dim3(nblocks((size_t)C * D * H * W / 8)), dim3(256), 0, (hipStream_t)stream, in,
                     out, C, D, H, W);
  return (int)hipGetLastError();
}

int hr_nn_avgpool2_grad(const float* dy, float* dx, long long C, int D, int H, int W, int accumulate, void* stream) {
  if (!dy || !dx || C < 1 || bad_vol(D, H, W, 1) || odd(D, H, W)) return 1;
  hipLaunchKernelGGL(avgpool2_grad_kernel, dim3(nblocks((size_t)C * D * H * W)), dim3(256), 0, (hipStream_t)stream,
                     dy, dx, C, D, H, W, accumulate, (const float*)nullptr, 1.0f);
  return (int)hipGetLastError();
}

int hr_nn_avgpool2_grad_act(const float* dy, const float* y, float* dx, long long C, int D, int H, int W, float slope,
                            void* stream) {
  if (!dy || !y || !dx || C < 1 || bad_vol(D, H, W, 1) || odd(D, H, W)) return 1;
  hipLaunchKernelGGL(avgpool2_grad_kernel, dim3(nblocks((size_t)C * D * H * W)), dim3(256), 0, (hipStream_t)stream,
                     dy, dx, C, D, H, W, 1, y, slope);
  return (int)hipGetLastError();
}

int hr_nn_upsample2(const float* in, float* out, long long C, int D, int H, int W, void* stream) {
  if (!in || !out || C < 1 || bad_vol(D, H, W, 1) || odd(D, H, W)) return 1;
  hipLaunchKernelGGL(upsample2_kernel, dim3(nblocks((size_t)C * D * H * W)), dim3(256), 0, (hipStream_t)stream, in,
                     out, C, D, H, W);
  return (int)hipGetLastError();
}

int hr_nn_upsample2_grad(const float* dy, float* dx, long long C, int D, int H, int W, void* stream) {
  return hr_nn_upsample2_grad_act(dy, nullptr, dx, C, D, H, W, 1.0f, stream);
}

int hr_nn_upsample2_grad_act(const float* dy, const float* y, float* dx, long long C, int D, int H, int W, float slope,
                             void* stream) {
  if (!dy || !dx || C < 1 || bad_vol(D, H, W, 1) || odd(D, H, W)) return 1;
  hipLaunchKernelGGL(upsample2_grad_kernel, dim3(nblocks((size_t)C * D * H * W / 8)), dim3(256), 0,
                     (hipStream_t)stream, dy, dx, C, D, H, W, y, slope);
  return (int)hipGetLastError();
}

// loss[0] = mean (y - t)^2 over n; grad (may be null) = 2 (y - t) / n; part: 256 floats of scratch
int hr_nn_mse(const float* y, const float* t, long long n, float* grad, float* part, float* loss, void* stream) {
  if (!y || !t || !part || !loss || n < 1) return 1;
  hipLaunchKernelGGL(mse_kernel, dim3(MSE_BLOCKS), dim3(256), 0, (hipStream_t)stream, y, t, (size_t)n, grad, part);
  hipLaunchKernelGGL(loss_finish_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, part, MSE_BLOCKS, (size_t)n, loss);
  return (int)hipGetLastError();
}

// step >= 1: bias corrections 1 - b1^step, 1 - b2^step; wb (may be null) gets the BF16 copy
int hr_nn_adam(float* w, const float* g, float* m, float* v, unsigned short* wb, long long n, float lr, float b1,
               float b2, float eps, int step, void* stream) {
  if (!w || !g || !m || !v || n < 1 || step < 1) return 1;
  const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
  hipLaunchKernelGGL(adam_kernel, dim3(nblocks((size_t)n)), dim3(256), 0, (hipStream_t)stream, w, g, m, v, wb,
                     (size_t)n, lr, b1, b2, eps, c1, c2);
  return (int)hipGetLastError();
}

int hr_nn_to_bf16(const float* w, unsigned short* wb, long long n, void* stream) {
  if (!w || !wb || n < 1) return 1;
  hipLaunchKernelGGL(to_bf16_kernel, dim3(nblocks((size_t)n)), dim3(256), 0, (hipStream_t)stream, w, wb, (size_t)n);
  return (int)hipGetLastError();
}

}  // extern "C"
