// lepic_internal.h -- shared device helpers and the context of liblepic_hip.so.
//
// All arithmetic on the FP64 path keeps the reference's operation order and
// is compiled with -ffp-contract=off, so each product and sum rounds once as
// in a strict build of the reference.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/lepic.h"
#include "lepic_qdiv.h"

#define LEPIC_WAVE 64

struct lepic_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  // generic growable device scratch (sort keys, look-back status, ...)
  void *scratch = nullptr;
  size_t scratch_bytes = 0;
  void *scratch2 = nullptr;
  size_t scratch2_bytes = 0;
  size_t scratch_limit = 0;           // most bytes of either (0: no bound)
  // small device control block: counters, flags, partial sums
  int64_t *d_ctrl = nullptr;          // 4096 int64 words
  int64_t *h_pinned = nullptr;        // 4096 pinned host words for readbacks
  uint32_t epoch = 0;                 // look-back epoch (16 bits used)
  uint64_t *d_status = nullptr;       // look-back status words
  int64_t status_len = 0;
  // multigrid level storage
  void *mg_mem = nullptr;
  size_t mg_bytes = 0;
  int32_t mg_n[3] = {0, 0, 0};
  int32_t mg_ng = 0;
  // captured V-cycles (first and later ones) and the solve they belong to
  hipGraphExec_t mg_exec[2] = {nullptr, nullptr};
  std::vector<unsigned char> mg_key;
  hipStream_t capture_stream = nullptr;
  // mixed-precision solve: FP32 correction levels, and the captured inner
  // V-cycles + correction of one refinement step with the solve they belong to
  void *mgx_mem = nullptr;
  size_t mgx_bytes = 0;
  hipGraphExec_t mgx_exec = nullptr;
  std::vector<unsigned char> mgx_key;
  // the captured iteration of the preconditioned conjugate-gradient solve
  hipGraphExec_t pcg_exec = nullptr;
  std::vector<unsigned char> pcg_key;
  // per-XCD deposit replicas (LEPIC_XCDS x nodes doubles, kept zeroed)
  double *rep = nullptr;
  int64_t rep_nodes = 0;
  // per-XCD wall-diagnostic replicas (kept zeroed)
  double *wdiag = nullptr;
};

// MI355X has 8 XCDs, each with its own L2.  Deposition accumulates into one
// node-array replica per XCD with L2-resident (workgroup-scope) atomics; the
// replicas are summed afterwards.  The XCD of a running wave comes from the
// XCC_ID hardware register, so the replica choice never depends on how the
// dispatcher spreads workgroups.
#define LEPIC_XCDS 8
// electrode labels whose wall diagnostics the production pushes sum per
// block (lepic_partutil.h); the context keeps LEPIC_XCDS replicas of
// 2 LEPIC_WD_LABELS + 1 doubles for them
#define LEPIC_WD_LABELS 16

__device__ inline int xcc_id() {
  // s_getreg_b32 hwreg(HW_REG_XCC_ID=20, offset 0, size 4)
  return (int)(__builtin_amdgcn_s_getreg((3 << 11) | 20) & (LEPIC_XCDS - 1));
}

// Atomic add performed in this XCD's L2 (no cross-XCD coherence): valid only
// on memory that no other XCD touches during the kernel.
__device__ inline void l2_atomic_add(double *p, double v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

double *lepic_replicas(lepic_ctx *ctx, int64_t nodes);
int lepic_replica_flush(lepic_ctx *ctx, int64_t nodes, double *np_local, const double *kq);

// control block word offsets (int64 units)
enum : int {
  CTRL_TILE_COUNTER = 0,   // int32 used
  CTRL_COUNT_OUT = 8,      // compaction output count
  CTRL_SPIN_FAIL = 16,     // set when a bounded wait gives up
  CTRL_MCC = 64,           // MCC counters (256 words)
  CTRL_HEAT = 384,         // electron heating: count, energy sum, vt, seed (8 words)
  CTRL_MG = 512,           // MG per-level control (12 levels x 16 words)
  CTRL_PARTIALS = 1024,    // reduction partials (3072 words)
  CTRL_WORDS = 4096
};

int lepic_fail(lepic_ctx *ctx, int code, const std::string &msg);
int lepic_hip_check(lepic_ctx *ctx, hipError_t e, const char *what);
void *lepic_scratch(lepic_ctx *ctx, size_t bytes, int which);
// Particle indices ordered by cell (lepic_particles32.hip), on scratch 0 until
// its next use: first slots and counts per cell, the indices, their number.
struct CellOrder {
  int32_t *count, *start, *cursor, *bsum, *idx;
  int32_t *extra;    // the words asked for besides
  const int32_t *gate = nullptr;   // order_open (lepic_partutil.h): the kernels that form it
                                   // do so only then; count cleared by the caller
  int64_t *total;
  int32_t big = 0;                 // > 0: the cells of more go to list, *nlist of them
  int32_t *list, *nlist;           // (n / big at most)
};
// false: the scratch cannot be had
bool lepic_order_alloc(lepic_ctx *ctx, const int32_t dims[3], int64_t n, int64_t extra,
                       int32_t big, CellOrder &o);
int lepic_order_run(lepic_ctx *ctx, const int32_t dims[3], const int32_t *cell, int64_t n,
                    const CellOrder &o);
// The same of an FP64 set by its stencils' lower nodes (n + 2 per axis), which go
// to cell (16-byte aligned).
int lepic_order_run_set(lepic_ctx *ctx, const lepic_grid *g, const lepic_pset *set, int32_t *cell,
                        const CellOrder &o);
// Resolves, once per device, the static scratch lepic_efield_noalloc uses
// (lepic_fields.hip); the device must be current.
void lepic_efield_scratch_setup(int device);
uint32_t lepic_next_epoch(lepic_ctx *ctx, int64_t ntiles);

#define LEPIC_HIP(ctx, call)                                    \
  do {                                                          \
    hipError_t e__ = (call);                                    \
    if (e__ != hipSuccess) return lepic_hip_check(ctx, e__, #call); \
  } while (0)

#define LEPIC_LAUNCH_CHECK(ctx, what)                           \
  do {                                                          \
    hipError_t e__ = hipGetLastError();                         \
    if (e__ != hipSuccess) return lepic_hip_check(ctx, e__, what); \
  } while (0)

// ---------------------------------------------------------------------------
// Grid geometry handed to kernels by value.
// ---------------------------------------------------------------------------
struct KGrid {
  int n1, n2, n3;
  int64_t sy, sz;   // strides of j and k (x stride is 1)
  double h1, h2, h3;
  QDiv q1, q2, q3;  // x/h1, y/h2, z/h3 correctly rounded (lepic_qdiv.h)
};

static inline KGrid make_kgrid(const lepic_grid *g) {
  KGrid k;
  k.n1 = g->n[0]; k.n2 = g->n[1]; k.n3 = g->n[2];
  k.sy = (int64_t)g->n[0] + 3;
  k.sz = ((int64_t)g->n[0] + 3) * ((int64_t)g->n[1] + 3);
  k.h1 = g->h[0]; k.h2 = g->h[1]; k.h3 = g->h[2];
  k.q1 = qdiv_make(g->h[0]); k.q2 = qdiv_make(g->h[1]); k.q3 = qdiv_make(g->h[2]);
  return k;
}

static inline int64_t grid_nodes(const lepic_grid *g) {
  return ((int64_t)g->n[0] + 3) * ((int64_t)g->n[1] + 3) * ((int64_t)g->n[2] + 3);
}

__host__ __device__ inline int64_t gidx(const KGrid &g, int i, int j, int k) {
  return (int64_t)i + g.sy * (int64_t)j + g.sz * (int64_t)k;
}

__device__ inline int imin(int a, int b) { return a < b ? a : b; }
__device__ inline int imax(int a, int b) { return a > b ? a : b; }

// Trilinear stencil of mod_particleMover.f90:104-127: lower node clamped to
// [0, n+1], weights w1..w8 over nodes (ix,iy,iz), (ix+1,iy,iz), (ix+1,iy+1,iz),
// (ix,iy+1,iz) and the same at iz+1.
struct Stencil {
  int64_t base;      // node (ix,iy,iz)
  double w[8];
};

__device__ inline void make_stencil(const KGrid &g, double xp, double yp, double zp,
                                    Stencil &s) {
  int ix = (int)qdiv(xp, g.q1) + 1;
  int iy = (int)qdiv(yp, g.q2) + 1;
  int iz = (int)qdiv(zp, g.q3) + 1;
  ix = imax(0, imin(g.n1 + 1, ix));
  iy = imax(0, imin(g.n2 + 1, iy));
  iz = imax(0, imin(g.n3 + 1, iz));
  double px = qdiv((double)ix * g.h1 - xp, g.q1);
  double py = qdiv((double)iy * g.h2 - yp, g.q2);
  double pz = qdiv((double)iz * g.h3 - zp, g.q3);
  double wx2 = 1.0 - px, wy2 = 1.0 - py, wz2 = 1.0 - pz;
  s.w[0] = px * py * pz;
  s.w[1] = wx2 * py * pz;
  s.w[2] = wx2 * wy2 * pz;
  s.w[3] = px * wy2 * pz;
  s.w[4] = px * py * wz2;
  s.w[5] = wx2 * py * wz2;
  s.w[6] = wx2 * wy2 * wz2;
  s.w[7] = px * wy2 * wz2;
  s.base = gidx(g, ix, iy, iz);
}

// Lower node and fractions of deposit_weights (mod_charge_weights.f90:9-33:
// same range guard, same arithmetic); false: no deposit.
__device__ inline bool deposit_fracs(const KGrid &g, double x, double y, double z, int &ix,
                                     int &iy, int &iz, double &px, double &py, double &pz) {
  const double xmax = (double)g.n1 * g.h1, ymax = (double)g.n2 * g.h2,
               zmax = (double)g.n3 * g.h3;
  if (!(x >= -1.0e-12 && x <= xmax + 1.0e-12)) return false;
  if (!(y >= -1.0e-12 && y <= ymax + 1.0e-12)) return false;
  if (!(z >= -1.0e-12 && z <= zmax + 1.0e-12)) return false;
  ix = (int)qdiv(x, g.q1) + 1;
  iy = (int)qdiv(y, g.q2) + 1;
  iz = (int)qdiv(z, g.q3) + 1;
  px = qdiv((double)ix * g.h1 - x, g.q1);
  py = qdiv((double)iy * g.h2 - y, g.q2);
  pz = qdiv((double)iz * g.h3 - z, g.q3);
  return true;
}

// One particle's deposit, sign * kq[node] * k1 * w per node, by device-scope
// atomics (k1 = Nm / (h1 h2 h3)); the node order and weights of the run
// deposit in the particle kernels.
__device__ inline void deposit_one(const KGrid &g, double *np, const double *__restrict__ kq,
                                   double k1, double x, double y, double z, double sign) {
  int ix, iy, iz;
  double px, py, pz;
  if (!deposit_fracs(g, x, y, z, ix, iy, iz, px, py, pz)) return;
  const double wx2 = 1.0 - px, wy2 = 1.0 - py, wz2 = 1.0 - pz;
  const double w[8] = {px * py * pz,  wx2 * py * pz,  wx2 * wy2 * pz,  px * wy2 * pz,
                       px * py * wz2, wx2 * py * wz2, wx2 * wy2 * wz2, px * wy2 * wz2};
  const int64_t b = gidx(g, ix, iy, iz);
  const int64_t nd[8] = {b, b + 1, b + g.sy + 1, b + g.sy, b + g.sz, b + g.sz + 1,
                         b + g.sz + g.sy + 1, b + g.sz + g.sy};
#pragma unroll
  for (int q = 0; q < 8; ++q) atomicAdd(&np[nd[q]], sign * (kq[nd[q]] * (k1 * w[q])));
}

// Fixed-point deposit: one particle's full weight U (an integer number of
// units of 2^-S, held in a double below 2^53) split over its 8 stencil nodes
// in the order w1..w8 of the trilinear stencil (lower corner, +x, +x+y, +y,
// then the same at +z).  The weight is divided along x, then y, then z: at
// each division the upper node takes rint(parent * share) and the lower node
// the rest, so the 8 parts are integers that sum to U exactly -- charge is
// conserved bit for bit -- and each part is within 1.5 units of U times its
// trilinear weight.  ux, uy, uz are the upper nodes' shares (1 - px of the
// FP64 stencil, the in-cell offset of the FP32 layout).
__host__ __device__ inline void fixed_split(double U, double ux, double uy, double uz,
                                            long long a[8]) {
  const double x1 = rint(U * ux), x0 = U - x1;
  const double x0y1 = rint(x0 * uy), x0y0 = x0 - x0y1;
  const double x1y1 = rint(x1 * uy), x1y0 = x1 - x1y1;
  const double c[4] = {x0y0, x1y0, x1y1, x0y1};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const double z1 = rint(c[q] * uz);
    a[q] = (long long)(c[q] - z1);
    a[q + 4] = (long long)z1;
  }
}

// The same split in FP32 for the FP32 particle phase, whose full weight U is
// an integer of at most 2^22 units: every product U*u (< 2^22) rounds to
// FP32 with two fraction bits to spare, rint makes it an integer, and every
// difference of integers below 2^23 is exact, so the 8 parts are integers
// (int32) that sum to U exactly, at a fraction of the FP64 split's cost.
// The FP32 kernels take U up to 2^21 units, so that one block's sums at a node
// (1024 particles at most) fit the uint32 of their LDS box.
#define LEPIC_FIXED32_MAX 2097152.0   // 2^21 units per full weight
__host__ __device__ inline void fixed_split32(float U, float ux, float uy, float uz, int a[8]) {
  const float x1 = rintf(U * ux), x0 = U - x1;
  const float x0y1 = rintf(x0 * uy), x0y0 = x0 - x0y1;
  const float x1y1 = rintf(x1 * uy), x1y0 = x1 - x1y1;
  const float c[4] = {x0y0, x1y0, x1y1, x0y1};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float z1 = rintf(c[q] * uz);
    a[q] = (int)(c[q] - z1);
    a[q + 4] = (int)z1;
  }
}

// make_stencil with the quotient range test taken once for the particle
// (ok = qdiv_coord_ok of x, y and z): the same stencil for every input.
__device__ inline void make_stencil_pre(const KGrid &g, double xp, double yp, double zp, bool ok,
                                        Stencil &s) {
  int ix = (int)qdiv_pre(xp, g.q1, ok) + 1;
  int iy = (int)qdiv_pre(yp, g.q2, ok) + 1;
  int iz = (int)qdiv_pre(zp, g.q3, ok) + 1;
  ix = imax(0, imin(g.n1 + 1, ix));
  iy = imax(0, imin(g.n2 + 1, iy));
  iz = imax(0, imin(g.n3 + 1, iz));
  double px = qdiv_pre((double)ix * g.h1 - xp, g.q1, ok);
  double py = qdiv_pre((double)iy * g.h2 - yp, g.q2, ok);
  double pz = qdiv_pre((double)iz * g.h3 - zp, g.q3, ok);
  double wx2 = 1.0 - px, wy2 = 1.0 - py, wz2 = 1.0 - pz;
  s.w[0] = px * py * pz;
  s.w[1] = wx2 * py * pz;
  s.w[2] = wx2 * wy2 * pz;
  s.w[3] = px * wy2 * pz;
  s.w[4] = px * py * wz2;
  s.w[5] = wx2 * py * wz2;
  s.w[6] = wx2 * wy2 * wz2;
  s.w[7] = px * wy2 * wz2;
  s.base = gidx(g, ix, iy, iz);
}

// Gather of a 4-wide node field (E or B map) in the reference's summation order.
__device__ inline void gather3(const double4 *__restrict__ F, const KGrid &g, const Stencil &s,
                               double &ox, double &oy, double &oz) {
  const int64_t b0 = s.base, b1 = s.base + g.sy, b2 = s.base + g.sz, b3 = s.base + g.sz + g.sy;
  const double4 f1 = F[b0], f2 = F[b0 + 1], f3 = F[b1 + 1], f4 = F[b1];
  const double4 f5 = F[b2], f6 = F[b2 + 1], f7 = F[b3 + 1], f8 = F[b3];
  ox = s.w[0] * f1.x + s.w[1] * f2.x + s.w[2] * f3.x + s.w[3] * f4.x + s.w[4] * f5.x +
       s.w[5] * f6.x + s.w[6] * f7.x + s.w[7] * f8.x;
  oy = s.w[0] * f1.y + s.w[1] * f2.y + s.w[2] * f3.y + s.w[3] * f4.y + s.w[4] * f5.y +
       s.w[5] * f6.y + s.w[6] * f7.y + s.w[7] * f8.y;
  oz = s.w[0] * f1.z + s.w[1] * f2.z + s.w[2] * f3.z + s.w[3] * f4.z + s.w[4] * f5.z +
       s.w[5] * f6.z + s.w[6] * f7.z + s.w[7] * f8.z;
}

// Velocity update of part_mover (Src/part_expmover.f90:139-240) given the
// gathered E; bmode 0 leapfrog, 1 uniform B, 2 map gated at the lower node.
struct KBField {
  int mode;
  int magnetized;
  double bx, by, bz;
  const double4 *B4;
  double k2u;   // uniform B: k1*2/(1+(k1*|B|)^2), the same for every particle
  // map on its own grid (lepic_bfield mode 3, run as mode 2 with own_grid)
  int own_grid;
  int nB1, nB2, nB3;
  int64_t sBy, sBz;
  double hB1, hB2, hB3;
  QDiv qB1, qB2, qB3;
};

// The map's stencil at (x, y, z) when it lives on its own grid
// (Src/part_expmover.f90:149-175, flag_gridB = 1): lower node
// int(x/hB) + 1, kept inside the map's nodes 0..nB+1 so that the stencil
// stays in the array (positions inside the domain never need it).
__device__ inline void b_stencil(const KBField &bf, double xp, double yp, double zp, Stencil &s) {
  int ix = (int)fmax(fmin(qdiv(xp, bf.qB1), 2.0e9), -2.0e9) + 1;
  int iy = (int)fmax(fmin(qdiv(yp, bf.qB2), 2.0e9), -2.0e9) + 1;
  int iz = (int)fmax(fmin(qdiv(zp, bf.qB3), 2.0e9), -2.0e9) + 1;
  ix = imax(0, imin(bf.nB1 + 1, ix));
  iy = imax(0, imin(bf.nB2 + 1, iy));
  iz = imax(0, imin(bf.nB3 + 1, iz));
  const double px = qdiv((double)ix * bf.hB1 - xp, bf.qB1);
  const double py = qdiv((double)iy * bf.hB2 - yp, bf.qB2);
  const double pz = qdiv((double)iz * bf.hB3 - zp, bf.qB3);
  const double wx2 = 1.0 - px, wy2 = 1.0 - py, wz2 = 1.0 - pz;
  s.w[0] = px * py * pz;
  s.w[1] = wx2 * py * pz;
  s.w[2] = wx2 * wy2 * pz;
  s.w[3] = px * wy2 * pz;
  s.w[4] = px * py * wz2;
  s.w[5] = wx2 * py * wz2;
  s.w[6] = wx2 * wy2 * wz2;
  s.w[7] = px * wy2 * wz2;
  s.base = ix + bf.sBy * iy + bf.sBz * iz;
}

// BM is the B mode when known at compile time (the kernels are instantiated
// per mode, so a run with uniform B carries no registers for the map
// gather), -1 to read it from bf.
// xp, yp, zp: the position the fields are gathered at (the map on its own
// grid takes its stencil from it).
template <int BM>
__device__ inline void velocity_update(const KGrid &g, const KBField &bf, const Stencil &s,
                                       double k1, double Ex, double Ey, double Ez, double &vx,
                                       double &vy, double &vz, double xp, double yp, double zp) {
  const int mode = BM >= 0 ? BM : bf.mode;
  int use_b = 0;
  double Bx = 0.0, By = 0.0, Bz = 0.0;
  if (mode == 1) {
    Bx = bf.bx; By = bf.by; Bz = bf.bz;
    use_b = 1;
  } else if (mode == 2) {
    if (bf.own_grid) {
      Stencil sb;
      b_stencil(bf, xp, yp, zp, sb);
      if (bf.B4[sb.base].w > 1.0e-5) {
        const int64_t b0 = sb.base, b1 = sb.base + bf.sBy, b2 = sb.base + bf.sBz,
                      b3 = sb.base + bf.sBz + bf.sBy;
        const double4 f1 = bf.B4[b0], f2 = bf.B4[b0 + 1], f3 = bf.B4[b1 + 1], f4 = bf.B4[b1];
        const double4 f5 = bf.B4[b2], f6 = bf.B4[b2 + 1], f7 = bf.B4[b3 + 1], f8 = bf.B4[b3];
        Bx = sb.w[0] * f1.x + sb.w[1] * f2.x + sb.w[2] * f3.x + sb.w[3] * f4.x +
             sb.w[4] * f5.x + sb.w[5] * f6.x + sb.w[6] * f7.x + sb.w[7] * f8.x;
        By = sb.w[0] * f1.y + sb.w[1] * f2.y + sb.w[2] * f3.y + sb.w[3] * f4.y +
             sb.w[4] * f5.y + sb.w[5] * f6.y + sb.w[6] * f7.y + sb.w[7] * f8.y;
        Bz = sb.w[0] * f1.z + sb.w[1] * f2.z + sb.w[2] * f3.z + sb.w[3] * f4.z +
             sb.w[4] * f5.z + sb.w[5] * f6.z + sb.w[6] * f7.z + sb.w[7] * f8.z;
        use_b = 1;
      }
    } else if (bf.B4[s.base].w > 1.0e-5) {
      gather3(bf.B4, g, s, Bx, By, Bz);
      use_b = 1;
    }
  }
  if (!bf.magnetized) use_b = 0;
  if (use_b) {
    double k2;
    if (mode == 1) {
      k2 = bf.k2u;
    } else {
      double Bt = sqrt(Bx * Bx + By * By + Bz * Bz);
      k2 = k1 * (2.0 / (1.0 + (k1 * Bt) * (k1 * Bt)));
    }
    double v1x = vx + k1 * Ex, v1y = vy + k1 * Ey, v1z = vz + k1 * Ez;
    double v3x = v1x + k1 * (v1y * Bz - v1z * By);
    double v3y = v1y + k1 * (v1z * Bx - v1x * Bz);
    double v3z = v1z + k1 * (v1x * By - v1y * Bx);
    double v2x = v1x + k2 * (v3y * Bz - v3z * By);
    double v2y = v1y + k2 * (v3z * Bx - v3x * Bz);
    double v2z = v1z + k2 * (v3x * By - v3y * Bx);
    vx = v2x + k1 * Ex; vy = v2y + k1 * Ey; vz = v2z + k1 * Ez;
  } else {
    vx = vx + 2.0 * k1 * Ex; vy = vy + 2.0 * k1 * Ey; vz = vz + 2.0 * k1 * Ez;
  }
}

// k1 = dt*q/(2m) of the launch; the uniform-B k2 is evaluated here with the
// same operations the per-particle path performs.
static inline KBField make_kbfield(const lepic_bfield *bf, double k1) {
  KBField k;
  k.mode = bf ? bf->mode : 0;
  k.own_grid = 0;
  k.nB1 = k.nB2 = k.nB3 = 0;
  k.sBy = k.sBz = 0;
  k.hB1 = k.hB2 = k.hB3 = 1.0;
  if (k.mode == 3) {   // the map on its own grid runs in the map kernels
    k.mode = 2;
    k.own_grid = 1;
    k.nB1 = bf->nB[0]; k.nB2 = bf->nB[1]; k.nB3 = bf->nB[2];
    k.sBy = (int64_t)k.nB1 + 3;
    k.sBz = ((int64_t)k.nB1 + 3) * ((int64_t)k.nB2 + 3);
    k.hB1 = bf->hB[0]; k.hB2 = bf->hB[1]; k.hB3 = bf->hB[2];
  }
  k.qB1 = qdiv_make(k.hB1);
  k.qB2 = qdiv_make(k.hB2);
  k.qB3 = qdiv_make(k.hB3);
  k.magnetized = bf ? bf->magnetized : 1;
  k.bx = bf ? bf->B[0] : 0.0; k.by = bf ? bf->B[1] : 0.0; k.bz = bf ? bf->B[2] : 0.0;
  k.B4 = bf ? reinterpret_cast<const double4 *>(bf->B4) : nullptr;
  double Bt = std::sqrt(k.bx * k.bx + k.by * k.by + k.bz * k.bz);
  k.k2u = k1 * (2.0 / (1.0 + (k1 * Bt) * (k1 * Bt)));
  return k;
}

static inline unsigned grid_blocks(int64_t n, int block) {
  int64_t b = (n + block - 1) / block;
  return (unsigned)(b > 0 ? b : 1);
}
