// Device-side data structures shared by the HIP kernels and the host API.
#pragma once
#include <cstdint>

namespace hr {

constexpr int NCOMP = 9;           // u_x u_y u_z s_xx s_yy s_zz s_xy s_xz s_yz

// Structured box geometry and the per-element constants (all elements of the
// box share one geometry: edges hx, hy, hz).
struct Geo {
  int nex, ney, nez;               // elements per axis (PML included)
  int NX, NY, NZ;                  // lattice nodes per axis (2*ne + 1)
  long long NN;                    // lattice nodes
  int rlo[3], rhi[3];              // regular-domain element box [lo, hi)
  int top_rule;                    // 1: original top PML nodes lose s_zz, s_xz, s_yz
  int tiles[3];                    // stage-kernel tiles per axis
  int tx, ty;                      // elements per tile in x and y
  int tz;                          // elements per z-chunk of a tile
  double dxi[3];                   // dxi/dx = DJI(k,k) of the affine element
  double detj;                     // det J of the affine element
  double wq[27];                   // GLL weight * det J at local point a + 3b + 9c
  double pml[24];                  // PML_PARAM(6,4), column-major
};

struct StageArgs {
  Geo g;
  const double* in[6];             // as Stage3Args
  int stage;                       // 0 = apply (raw operator), 1..4 = RK4 stage, 5 = central difference
  int set_mask;                    // bit0: G on v1, bit1: K on v2, bit2: C on v3
  int transpose;                   // 1: apply the transposed operator
  double sgn[3];                   // multipliers on v1, v2, v3 (the kernels fix them by the transpose)
  double h, hh, h6, h4;            // as Stage3Args
  double* out;                     // stage 1-3: a_s; apply: raw result
  double* xnew[3];                 // stage 4: updated x1, x2, x3; stage 5: u_{n+1}, u_his
  int nsrc_tiles;                  // 0: no source
};

}  // namespace hr

#include <hip/hip_runtime.h>
namespace hr {
// Host launchers (defined with the kernels).
hipError_t launch_gather_eq(long long neq, const unsigned* slot, const double* x, const double* r, double* out,
                            hipStream_t s);
hipError_t launch_scatter_eq(long long neq, const unsigned* slot, const double* raw, const double* y, double sc,
                             const double* l, double* z, hipStream_t s);
// Device-side step index of a captured time loop: the kernel reads *step once and
// offsets its per-step pointer by (*step) * stride elements (step null: no offset).
struct StepRef {
  const int* step = nullptr;
  long long stride = 0;
};
// node table, regular-domain mass, M^-1 of the u rows and PML rho W sums of a material;
// tab: the small table; lam, mu, rho (device) may lie where the quadruples go
hipError_t launch_material(const Geo& g, const double* tab, const double* lam, const double* mu, const double* rho,
                           double* node, double* mrd, double* minvu, double* rwp, hipStream_t s);
// A step's outputs of all shots: receiver traces (nrec 0: none) and the displacement of
// the regular-domain node box as a history slice (nbox 0: none)
struct OutArgs {
  int nshot;
  const double* x2;                // state vector, shots xstride apart
  long long xstride;
  int nrec;
  const long long* slot;
  double* row;                     // trace row, shots rstride apart
  long long rstride;
  int nbox, b0[3], bn[3], NX, NY;  // node box
  double* hist;                    // slice, shots hstride apart
  long long hstride;
  const int* step;                 // captured loops: row and hist are those of step 0
};
constexpr int OUT_NT = 256;
__host__ __device__ inline int output_blocks(const OutArgs& O) { return (O.nrec + OUT_NT - 1) / OUT_NT + (O.nbox + OUT_NT - 1) / OUT_NT; }
hipError_t launch_outputs(const OutArgs& O, hipStream_t s);
// One adjoint step's gradient sums of all shots
struct GradArgs {
  int ntx, nty, ntz, tz, nshot;    // tiles, planes per z-chunk (gradient_args)
  int NX, NY, b0[3], bn[3];        // node box
  double dxi[3], wdt;              // centre point's weight x dt
  const double* uh;                // history slice (3 x box), shots ustride apart
  long long ustride;
  const double* p2;                // adjoint x2, shots pstride apart
  long long pstride;
  double *glam, *gmu;              // a block of box sums per shot
  const int* step;                 // captured loops: uh is the slice of step 0, stride elements a step
  long long stride;
};
GradArgs gradient_args(const Geo& g, const int* box0, const int* boxn, int nshot, const double* uh, long long ustride,
                       const double* p2, long long pstride, double dt, double* glam, double* gmu,
                       StepRef sr = StepRef());
// whole eights of blocks (0: none)
__host__ __device__ inline int gradient_blocks(const GradArgs& G) {
  return (int)(8 * (((long long)G.ntx * G.nty * G.ntz * G.nshot + 7) / 8));
}
hipError_t launch_gradient(const GradArgs& G, hipStream_t s);
// *step = value; *step += delta (one lane, a vector store)
hipError_t launch_step_set(int* step, int value, hipStream_t s);
hipError_t launch_step_advance(int* step, int delta, hipStream_t s);
hipError_t launch_gradient_finish(const Geo& g, const int* box0, const int* boxn, int nshot, const double* glb,
                                  const double* gmb, double* gl, double* gm, hipStream_t s);
hipError_t launch_permute_cols(long long nrows, int ncols, const long long* perm, const double* src, double* dst,
                               hipStream_t s);
// g += box sums on the regular-domain node box
hipError_t launch_box_add(const Geo& g, const int* box0, const int* boxn, const double* glb, const double* gmb,
                          double* gl, double* gm, hipStream_t s);
// out = 0.5 sum_n mrd[n] |x3 of node n|^2 (displacement block); part: energy_partials_size() doubles
int energy_partials_size();
hipError_t launch_energy(long long nn, const double* mrd, const double* x3, double* part, double* out, hipStream_t s);
hipError_t launch_sum(int n, const double* in, double* out, hipStream_t s);
// receivers grouped by equation: group g = receivers gidx[gptr[g] .. gptr[g+1])
hipError_t launch_misfit(int nstep, int ngrp, const int* gptr, const int* gidx, int nrec, const double* tr,
                         const double* ob, double dt, double* part, double* out, hipStream_t s);
// gradient post-processing (hr_reg.hip)
size_t reg_partials_size(const Geo& g);      // doubles of part below
hipError_t launch_gradient_mass(const Geo& g, double* img, double* restr, hipStream_t s);
// tv: 1 total variation, 0 TN; wreg: host (w_top, w_bot, w_Length) or nullptr; gl, gm:
// gradients whose norms are wanted too, or nullptr; red (RED_SUMS doubles): ||gl||^2,
// ||gm||^2, ||rl||^2, ||rm||^2, the two unscaled costs, then launch_reg_update's scaled
// costs and factors
constexpr int RED_SUMS = 10, RED_COST = 4, RED_SCALED = 6, RED_FACTOR = 8;
hipError_t launch_regularization(const Geo& g, const double* zc, int tv, const double* wreg, const double* lam,
                                 const double* mu, const double* gl, const double* gm, double* rl, double* rm,
                                 double* part, double* red, hipStream_t s);
hipError_t launch_reg_update(long long n, int add, double factor, const double* rl, const double* rm,
                             const double* img, double* gl, double* gm, double* red, hipStream_t s);
}  // namespace hr

namespace hr {
// ----------------------------------------------------------- stage kernel v3
constexpr int HR_MAX_ZCHUNKS = 64;
// Compact launch arguments: per-node and per-axis coefficients live in device
// tables, source lists behind a device pointer.
struct Geo3 {
  int NX, NY, NZ, NN;              // lattice (9 * NN < 2^31)
  int nex, ney, nez;
  int rlo[3], rhi[2];              // regular-domain element box; it extends to the top in z
  int top_rule;
  int tiles0, tiles1, tz;
  double dxi[3];
  double detj;
  int zb[HR_MAX_ZCHUNKS + 1];      // z-chunk c spans element layers [zb[c], zb[c+1])
};

// Node table: pairs (lam, mu) per node (2 NN doubles), then quadruples
// (minv_u, minv_s, rwp, wps) per node (4 NN doubles); each node's entries are
// one or two 16-byte loads.
constexpr int NT_PAIR = 2, NT_QUAD = 4, NT_COUNT = 6;
// Small table: [wq (27) | pad | (a_x, b_x) pairs (NX) | (a_y, b_y) (NY) | (a_z, b_z) (NZ)].
constexpr int TAB_STRETCH = 28;

struct Src3 {                      // device-resident source entries of one solve, grouped by shot and tile
  const int* tile_ptr;             // (nshot * ntiles + 1): entries of (shot, tile) at [ptr[s*ntiles+t], ptr[..+1])
  const long long* node;           // lattice node
  const int* comp;                 // component 0..2
  const double* m;                 // M^-1 of that DOF
  const double* val;               // forward: B entries
  const double* ftab;              // forward: source factors of stages 1, 2 and 4 (f0, 2 (fm - f0) / dt, (f0 - 2 fm + f1) / 6): nshot x nstep x 3
  const double* tr;                // adjoint: traces per shot, (nstep+1) rows of nrec, columns in entry order
  const double* obs;               // adjoint: observations, same layout
  int nrec;                        // adjoint: entries per shot (shared receivers)
  int nstep;
  int ntiles;
  // the same entries at PML nodes, by block of the PML node list: entries of
  // (shot, block) are pblk_idx[pblk_ptr[s*pnblk+b] .. pblk_ptr[s*pnblk+b+1]), in node
  // order, pblk_slot their node's thread in the block (an entry at a block's edge is
  // in two blocks, which both form that node's a)
  const int* pblk_ptr;
  const int* pblk_idx;
  const int* pblk_slot;
  int pnblk;
  // and those at regular-domain-only nodes, in (shot, node) order
  const int* rd_idx;
  const int* rd_shot;
  int nrd;
};

struct Stage3Args {
  Geo3 g;
  // RK4 stage: the operator inputs v1, v2, v3 (stage 1 x1 x2 x3, 2 x2 x3 a1, 3 x3 a1
  // a2, 4 a1 a2 a3; hr_split.hip gives the scheme), stage 4 then x1, x2, x3;
  // apply: in[0] = x; stage 5: u_n, u_{n-1}, u_his
  const double* in[6];
  double* out;                     // stage 1-3: a_s; apply: raw result
  double* xnew[3];                 // stage 4: updated x1, x2, x3; stage 5: u_{n+1}, u_his
  const double* node;              // node table
  const double* tab;               // small table
  Src3 src;                        // source entries, used when src_mode != 0
  int set_mask;                    // apply: bit0 G, bit1 K, bit2 C
  int src_mode;                    // 0 none, 1 forward: f * B * m, 2 adjoint misfit
  int step, fcol;                  // forward: f = ftab[(shot * nstep + step) * 3 + fcol]
  int ra, rb, rb_on;               // adjoint source rows (rb used when rb_on)
  double ca, cb;                   // adjoint row weights
  const int* step_dev;             // captured loops: step, ra, rb are offsets from *step_dev
  int nshot;                       // shots in the launch; state vectors are shot-major
  long long shot_stride;           // elements per shot of a state vector (9 NN)
  double h, hh, h6, h4;            // stage 4: h, h^2/2, h^3/6, h^4/24 (h = +-dt); stage 5: h, hh, h6 = dt, dt^2, dt^3
};

// Split stage path (hr_split.hip): the nodal kernels of one RK4 stage
struct SplitArgs {
  Geo3 g;
  const double* v[3];              // operator inputs
  const double* x[3];              // last stage: the state
  double* xn[2];                   // last stage: updated x1, x2
  double* out;                     // node-local terms, from the nodal pass to the pull
  double* a;                       // the pull's result: a_s (null: not kept); last stage: updated x3
  const double *node, *tab;        // node table (lambda, mu pairs), small table
  const double *minvu, *rwp;       // M^-1 of the displacement rows, sum of rho W over the PML elements per node (NN each)
  Src3 src;                        // as in Stage3Args
  int src_mode, step, fcol, ra, rb, rb_on;
  double ca, cb;
  const int* step_dev;
  int nshot;
  long long shot_stride;
  double h, h2, h3, h4;            // h, h^2/2, h^3/6, h^4/24
  double sc, ss;                   // scales of the stage's a in its output and of its source: 1, last stage h^4/24, h
  int pnbn;                        // blocks of the PML node list (SPLIT_OWN nodes each)
  double* D;                       // y- and z-line flux records, 12 NN doubles per shot
  const double* E;                 // regular-domain K sums of the interface nodes (sp_iface_column), 3 nif doubles per shot
  int nif;                         // interface nodes
};

// and its regular-domain element pass over two fields
struct RdArgs {
  Geo3 g;
  int ntx, nty, ntz, tz;           // tiles, element layers per z-chunk
  const double* in[2];             // x2, x3 (update: a1, a2)
  const double* x[2];              // update: x2, x3
  double* out[2];                  // a1, a2 (update: new x2, x3)
  double* E[2];                    // K sums of the interface nodes per field (sp_iface_column)
  int nif;                         // interface nodes
  const double *node, *minvu;
  int nshot;
  long long shot_stride;
  double h, h2, h3, h4;
};

// stage 0 = apply; transposed stages 1..4 carry the adjoint signs (-G, +K, -C)
hipError_t launch_stage3(const Stage3Args& A, int stage, int transpose, int tile_class, const int* tiles, int ntiles,
                         hipStream_t s);
// split stage path: the nodal pass over the PML nodes, the nodal pull, and the
// regular-domain element pass
constexpr int SPLIT_NT = 256;
// list entries a block of the nodal kernels owns: it also computes two entries on each
// side, for the x flux records of its own entries' x-lines
constexpr int SPLIT_OWN = SPLIT_NT - 4;      // nodes (threads) per block of the nodal kernels
hipError_t launch_split_nodal(const SplitArgs& A, int last, int transpose, hipStream_t s);
hipError_t launch_pull_nodal(const SplitArgs& P, const SplitArgs& N, int last, int transpose, hipStream_t s);
hipError_t launch_split_pull(const SplitArgs& A, int transpose, hipStream_t s);
void rd_tiles(const Geo& g, int tz, int t[3]);   // element pass tiles per axis (x, y, z-chunks)
// operator product: A.v[0] = x, A.out = A.a = result, one shot; set 0 G, 1 K, 2 C
hipError_t launch_split_apply(const SplitArgs& A, const RdArgs& R, int set, int transpose, hipStream_t s);
hipError_t launch_elements(const RdArgs& R, int update, hipStream_t s);
// both passes of stages 1 and 3, and the step's outputs
int stage_pair_blocks(const SplitArgs& A, const RdArgs& R);   // of the two passes
hipError_t launch_stage_pair(const SplitArgs& A, const RdArgs& R, const OutArgs& O, const GradArgs& G, int update,
                             int transpose, hipStream_t s);
}  // namespace hr
