// lepic_mg.hip -- V-cycle multigrid with red-black SOR smoothing (a8):
// pdesolver (modules/legacy/pdesolver.f90:1-135), mg (mg.f90:1-246),
// restriction (mg.f90:249-806), getres (mg.f90:809-848), prolongation
// (mg.f90:850-940) and sor_rb (modules/legacy/sors.f90:1-535), one rank.
//
// A sweep of a global level is one launch over tiles held in LDS (k_sweep):
// red, black and the L1 residual, with sor_rb's exit rule (res/res_s <= 0.6,
// at most 4 sweeps) taken by every block of the next launch.  Levels with
// periodic walls take two launches per sweep (k_per_half); narrow and flat levels
// (sweeps_tiled) and a coarsest level too large for one workgroup take one per
// colour, a deterministic block-tree residual and a one-block decision.  Sweeps queued after the exit return at
// once, so a V-cycle needs no host round trip; the host reads the fine
// residual once per V-cycle for pdesolver's convergence test.  Levels below a
// few thousand nodes run inside one workgroup (k_mg_coarse).
#include <algorithm>
#include <cmath>
#include <cstring>

#include "lepic_internal.h"
#include "lepic_walk.h"

namespace {

constexpr int BLOCK = 256;
constexpr int MAX_LEVELS = 12;

struct MGCtl {
  int64_t active;
  int64_t ksor;
  double res;
  double res_s;
  int64_t total;
  int64_t pad[11];
};
static_assert(sizeof(MGCtl) == 16 * sizeof(int64_t), "MGCtl layout");

// a + the value CTRL (a DPP row operation) brings, 0 where it brings none.
template <int CTRL, int ROWS>
__device__ inline double dpp_add(double a) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(a), CTRL, ROWS, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(a), CTRL, ROWS, 0xf, true);
  return a + __hiloint2double(hi, lo);
}

__device__ inline double read_lane(double a, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(a), lane),
                          __builtin_amdgcn_readlane(__double2loint(a), lane));
}

// Sum of each 16-lane row in its last lane.
__device__ inline double row_sum(double a) {
  a = dpp_add<0x111, 0xf>(a);   // row_shr:1, 2, 4, 8
  a = dpp_add<0x112, 0xf>(a);
  a = dpp_add<0x114, 0xf>(a);
  return dpp_add<0x118, 0xf>(a);
}

// Sum over a full wave in a fixed order, the same in every lane (register
// moves: six steps of shuffles through LDS take five times as long).
__device__ inline double wave_sum(double a) {
  a = row_sum(a);
  a = dpp_add<0x142, 0xa>(a);   // row_bcast:15 into rows 1 and 3
  a = dpp_add<0x143, 0xc>(a);   // row_bcast:31 into rows 2 and 3
  return read_lane(a, LEPIC_WAVE - 1);
}

// One multigrid level: geometry, stencil coefficients and the level's u, b
// and labels.  T is the storage and arithmetic type of u and b (double for
// the reference's solver, float for the smoother of the mixed-precision one).
// floor(x / d) for x < 2^32 by a 64-bit multiply-high: m = ceil(2^64 / d),
// and x m / 2^64 exceeds x / d by less than x / 2^64 < 2^-32 <= 1/d, so the
// floor is exact.  Decodes thread numbers into (i, j, k) without a division.
struct MDiv {
  uint64_t m;
  uint32_t d;
};

inline MDiv mdiv(uint32_t d) {
  MDiv v;
  v.d = d;
  v.m = d <= 1 ? 0 : (~0ull) / d + 1;
  return v;
}

__device__ inline uint32_t mdiv_q(uint32_t x, const MDiv &v) {
  return v.d <= 1 ? x : (uint32_t)__umul64hi((uint64_t)x, v.m);
}

// B: the label type (int32_t in global memory; int16_t in the coarse
// workgroup's LDS, labels saturated to that range, which keeps every test
// the solver makes of them: sign, 0, -1, -2).
template <class T, class B = int32_t>
struct KLevelT {
  KGrid g;
  T aw, ae, an, as, at, ab, ac;
  T *u;
  T *b;
  B *bc;
  // thread-number decoders: n1/2+1, n2+1, n1+1, n1+3, n1+2, n2/2+1
  MDiv d_h1, d_n2p1, d_n1p1, d_n1p3, d_n1p2, d_h2;
  double acy;   // RN(1 / ac) for the FP64 levels' division (0: plain division)
};

// x / ac of the SOR update: for FP64 levels by the reciprocal and two FMA
// corrections (lepic_qdiv.h: the correctly rounded quotient, identical to
// the division), the plain division otherwise.
template <class T, class B>
__device__ inline T div_ac(T x, const KLevelT<T, B> &L) {
  return x / L.ac;
}
template <class B>
__device__ inline double div_ac(double x, const KLevelT<double, B> &L) {
  if (L.acy == 0.0) return x / L.ac;
  QDiv d;
  d.h = L.ac;
  d.y = L.acy;
  return qdiv(x, d);
}

template <class T>
inline void set_level_divs(KLevelT<T> &L) {
  const KGrid &g = L.g;
  L.d_h1 = mdiv((uint32_t)(g.n1 / 2 + 1));
  L.d_n2p1 = mdiv((uint32_t)(g.n2 + 1));
  L.d_n1p1 = mdiv((uint32_t)(g.n1 + 1));
  L.d_n1p3 = mdiv((uint32_t)(g.n1 + 3));
  L.d_n1p2 = mdiv((uint32_t)(g.n1 + 2));
  L.d_h2 = mdiv((uint32_t)(g.n2 / 2 + 1));
}
using KLevel = KLevelT<double>;

template <class T, class B>
__device__ inline T getres(const KLevelT<T, B> &L, int ir, int jr, int kr, int flag_nmn) {
  const KGrid &g = L.g;
  if (ir < 0 || ir > g.n1 + 1 || jr < 0 || jr > g.n2 + 1 || kr < 0 || kr > g.n3 + 1) return T(0);
  const T *u = L.u;
  T aw = L.aw, ae = L.ae;
  const int64_t c = gidx(g, ir, jr, kr);
  T uij = u[c];
  T un = u[c + g.sy];
  T us = u[c - g.sy];
  T ue = u[c + 1];
  T ut = u[c + g.sz];
  T ub = kr >= 1 ? u[c - g.sz] : T(0);
  T uw;
  if (ir == 1 && flag_nmn == 1) {
    uw = T(0); aw = T(0); ae = T(2) * ae;
  } else {
    uw = u[c - 1];
  }
  T urhs = L.b[c];
  return urhs - (aw * uw + ae * ue + L.an * un + L.as * us + L.ac * uij + L.at * ut + L.ab * ub);
}

// sor_rb's start (the level active, no sweep counted yet).
__device__ inline void ctl_begin(MGCtl *ctl) {
  ctl->active = 1;
  ctl->ksor = 0;
  ctl->res = 0.0;
  ctl->res_s = 0.0;
}

__global__ void k_reset_totals(MGCtl *ctl, int n) {
  int t = threadIdx.x;
  if (t < n) ctl[t].total = 0;
}

// One colour of sor_rb (sors.f90:87-140 red, 249-302 black).
// colour 0 = red = (i+j+k) odd, 1 = black.  Threads over (i2, j, k).
template <class T, class B>
__device__ inline void sor_node(const KLevelT<T, B> &L, int colour, T omega, int64_t t) {
  const KGrid &g = L.g;
  const int ni2 = g.n1 / 2 + 1;
  int64_t total = (int64_t)ni2 * (g.n2 + 1) * (g.n3 + 1);
  if (t >= total) return;
  const uint32_t tt = (uint32_t)t, r = mdiv_q(tt, L.d_h1), rk = mdiv_q(r, L.d_n2p1);
  int i2 = (int)(tt - r * (uint32_t)ni2);
  int j = 1 + (int)(r - rk * (uint32_t)(g.n2 + 1));
  int k = 1 + (int)rk;
  int ks = (k % 2 == 0) ? 0 : 1;
  int is;
  if (colour == 0) is = (j % 2 == 0) ? 1 : 2;
  else is = (j % 2 == 0) ? 2 : 1;
  is += ks;
  if (is > 2) is = 1;
  int i = is + 2 * i2;
  if (i > g.n1 + 1) return;
  const int64_t c = gidx(g, i, j, k);
  const int bcv = L.bc[c];
  if (bcv > 0) return;
  if (bcv == 0 && (k == g.n3 + 1 || j == g.n2 + 1)) return;
  T *u = L.u;
  // every operand read before any arithmetic, so the reads overlap (the
  // ghost layer keeps u[c - 1] in bounds where the -2 rows do not use it)
  const T uc = u[c], uw = u[c - 1], ue = u[c + 1], un = u[c + g.sy], us = u[c - g.sy],
          ut = u[c + g.sz], ub = u[c - g.sz], bb = L.b[c];
  if (bcv == -2) {
    u[c] = (T(1) - omega) * uc +
           div_ac(omega * (bb - L.an * un - L.as * us - T(2) * L.ae * ue - L.at * ut - L.ab * ub),
                  L);
    return;
  }
  u[c] = (T(1) - omega) * uc +
         div_ac(omega * (bb - L.aw * uw - L.an * un - L.as * us - L.ae * ue - L.at * ut -
                         L.ab * ub),
                L);
}

// ctl == nullptr: a fixed sweep count (the level is always active).
// begin != nullptr: the first red sweep of an sor_rb, which always runs and
// arms the level's control block for the kernels after it.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_sor(KLevelT<T> L, int colour, T omega,
                                               const MGCtl *ctl, MGCtl *begin) {
  if (begin) {
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl_begin(begin);
  } else if (ctl && ctl->active == 0) {
    return;
  }
  sor_node(L, colour, omega, blockIdx.x * (int64_t)BLOCK + threadIdx.x);
}

// Periodic ghost copies (sors.f90:184-239, single rank): y planes for every
// (i, k), then z planes for every (i, j).
template <class T, class B>
__device__ inline void per_y_node(const KLevelT<T, B> &L, int64_t t) {
  const KGrid &g = L.g;
  int64_t ni = g.n1 + 3, nk = g.n3 + 3;
  if (t >= ni * nk) return;
  const uint32_t tt = (uint32_t)t, kk = mdiv_q(tt, L.d_n1p3);
  int i = (int)(tt - kk * (uint32_t)ni), k = (int)kk;
  int b1 = L.bc[gidx(g, i, 1, k)], b2 = L.bc[gidx(g, i, g.n2 + 1, k)];
  if (b1 == 0 || b1 == -2) L.u[gidx(g, i, 0, k)] = L.u[gidx(g, i, g.n2, k)];
  if (b2 == 0 || b2 == -2) L.u[gidx(g, i, g.n2 + 1, k)] = L.u[gidx(g, i, 1, k)];
}

template <class T, class B>
__device__ inline void per_z_node(const KLevelT<T, B> &L, int64_t t) {
  const KGrid &g = L.g;
  int64_t ni = g.n1 + 3, nj = g.n2 + 3;
  if (t >= ni * nj) return;
  const uint32_t tt = (uint32_t)t, jj = mdiv_q(tt, L.d_n1p3);
  int i = (int)(tt - jj * (uint32_t)ni), j = (int)jj;
  const int m = g.n3;
  int b1 = L.bc[gidx(g, i, j, 1)], b2 = L.bc[gidx(g, i, j, m + 1)];
  if (b1 == 0 || b1 == -2) L.u[gidx(g, i, j, 0)] = L.u[gidx(g, i, j, m)];
  if (b2 == 0 || b2 == -2) L.u[gidx(g, i, j, m + 1)] = L.u[gidx(g, i, j, 1)];
}

template <class T>
__global__ void k_per_y(KLevelT<T> L, const MGCtl *ctl) {
  if (ctl && ctl->active == 0) return;
  per_y_node(L, blockIdx.x * (int64_t)blockDim.x + threadIdx.x);
}

template <class T>
__global__ void k_per_z(KLevelT<T> L, const MGCtl *ctl) {
  if (ctl && ctl->active == 0) return;
  per_z_node(L, blockIdx.x * (int64_t)blockDim.x + threadIdx.x);
}

// L1 residual over bcnd == -1 nodes (sors.f90:409-431), block partials.
// |b - A u| at interior node t of the residual range (0 outside plasma).
template <class T, class B>
__device__ inline double resid_node(const KLevelT<T, B> &L, int64_t t) {
  const KGrid &g = L.g;
  int64_t nx = g.n1 + 1, ny = g.n2 + 1, nz = g.n3 + 1;
  double a = 0.0;
  if (t < nx * ny * nz) {
    const uint32_t tt = (uint32_t)t, r = mdiv_q(tt, L.d_n1p1), rk = mdiv_q(r, L.d_n2p1);
    int i = 1 + (int)(tt - r * (uint32_t)nx);
    int j = 1 + (int)(r - rk * (uint32_t)ny);
    int k = 1 + (int)rk;
    const int64_t c = gidx(g, i, j, k);
    if (L.bc[c] == -1) {
      const T *u = L.u;
      const T uc = u[c], uw = u[c - 1], ue = u[c + 1], un = u[c + g.sy], us = u[c - g.sy],
              ut = u[c + g.sz], ub = u[c - g.sz], bb = L.b[c];
      T rij = bb - (L.aw * uw + L.an * un + L.as * us + L.ae * ue + L.ac * uc + L.at * ut +
                    L.ab * ub);
      a = fabs((double)rij);
    }
  }
  return a;
}

// At most RESID_BLOCKS blocks, each thread striding over the nodes, so that
// the one-block decision sums few partials.  The order of the sum is fixed
// for a level (deterministic from run to run).
constexpr int RESID_BLOCKS = 1024;

template <class T>
__global__ __launch_bounds__(BLOCK) void k_resid(KLevelT<T> L, double *partials, const MGCtl *ctl,
                                                 int64_t nres) {
  if (ctl->active == 0) return;
  __shared__ double red[BLOCK / LEPIC_WAVE];
  double a = 0.0;
  const int64_t stride = (int64_t)gridDim.x * BLOCK;
  for (int64_t t = blockIdx.x * (int64_t)BLOCK + threadIdx.x; t < nres; t += stride)
    a = a + resid_node(L, t);
  for (int d = LEPIC_WAVE / 2; d > 0; d >>= 1) a = a + __shfl_down(a, d);
  if (__lane_id() == 0) red[threadIdx.x / LEPIC_WAVE] = a;
  __syncthreads();
  if (threadIdx.x == 0) {
    double b = 0.0;
    for (int w = 0; w < BLOCK / LEPIC_WAVE; ++w) b = b + red[w];
    partials[blockIdx.x] = b;
  }
}

// Sum the partials in a fixed order and apply sor_rb's exit rules
// (sors.f90:446-454).  A separate one-block launch: the kernel boundary
// makes every block's partial visible without a fence per block (a
// last-block-done reduction inside k_resid, with an agent-scope
// acquire-release count per block, measured slower than this launch).
__global__ __launch_bounds__(BLOCK) void k_decide(const double *partials, int64_t nparts,
                                                  MGCtl *ctl, double eps, int dig, int64_t nr) {
  if (ctl->active == 0) return;
  __shared__ double red[BLOCK];
  double a = 0.0;
  for (int64_t p = threadIdx.x; p < nparts; p += BLOCK) a = a + partials[p];
  red[threadIdx.x] = a;
  __syncthreads();
  for (int s = BLOCK / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] = red[threadIdx.x] + red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    double res = red[0];
    ctl->res = res;
    ctl->ksor += 1;
    ctl->total += 1;
    bool stop;
    if (dig == 0) stop = (res <= eps);
    else stop = (ctl->res_s > 0.0 && (res / ctl->res_s) <= 0.6);
    ctl->res_s = res;
    if (stop || ctl->ksor >= nr) ctl->active = 0;
  }
}


// --------------------------------------------------------------------------
// Whole sweeps of a global level in one launch.  A block takes a TX x TY x TZ
// tile, reads it with a halo of H nodes into LDS, runs the colour phases on
// rings of the halo that shrink by one per phase (the halo's nodes relaxed
// again by each tile that needs them: the same operands and expression, so
// the same bits as the owner's) and writes its own nodes to the other of two
// u arrays, which the next launch reads.  One launch per colour, residual and
// decision spends 60 us per sweep at 128^3 (19.6 + 19.6 + 15.2 + 5) and 12 at
// 16^3, all of it launches and L2 round trips; the fused sweep takes 28 us and
// 9 (an idle one 4.5), FP64, split about evenly between the reads (390 KB per
// block through one CU's L1), the three LDS phases and launch + decision.
//
// The two colours are held apart in LDS, so that the lanes of a phase read
// consecutive words.  Row (j, k) of node colours: red nodes have i + j + k
// odd; pair p of a row holds the nodes xb + 2 p and xb + 2 p + 1, xb even.
// --------------------------------------------------------------------------

// One sor_rb of at most 4 sweeps is 4 launches ("slots").  Every block of
// slot s sums slot s - 1's block residuals in the same fixed order and so
// takes the same exit decision; block 0 records it for slot s + 1.
struct SlotState {
  int64_t active;   // the slot swept
  int64_t pad;
  double res_s;     // the residual its decision compared against next
};

constexpr int SLOTS = 4;

struct SlotCtl {
  SlotState *state;     // SLOTS entries
  double *partials;     // 2 x nparts: slot s writes half s & 1
  int64_t nparts;       // blocks of the level's sweep launches
};

// Sum of slot s's block residuals, the same in every thread and block: this
// thread's first one (read early), then the rest and the block's sum.
__device__ inline double slot_first(const SlotCtl &sc, int s) {
  const double *p = sc.partials + (int64_t)(s & 1) * sc.nparts;
  return threadIdx.x < sc.nparts ? p[threadIdx.x] : 0.0;
}

template <int NT>
__device__ inline double slot_sum(const SlotCtl &sc, int s, double a, double *red) {
  const double *p = sc.partials + (int64_t)(s & 1) * sc.nparts;
  for (int64_t t = (int64_t)threadIdx.x + NT; t < sc.nparts; t += NT) a = a + p[t];
  for (int d = LEPIC_WAVE / 2; d > 0; d >>= 1) a = a + __shfl_down(a, d);
  if (__lane_id() == 0) red[threadIdx.x / LEPIC_WAVE] = a;
  __syncthreads();
  double r = 0.0;
  for (int w = 0; w < NT / LEPIC_WAVE; ++w) r = r + red[w];
  __syncthreads();
  return r;
}

// The exit rule of sor_rb above the coarsest level (sors.f90:446-454).
__device__ inline bool sor_stops(double res, double res_s) {
  return res_s > 0.0 && (res / res_s) <= 0.6;
}

// After the last slot: the counters of a sor_rb that ran all its sweeps (an
// earlier exit has already left its own).  Called by one block of NT threads.
template <int NT>
__device__ inline void slots_finish(const SlotCtl &sc, MGCtl *ctl, double *red) {
  if (sc.state[SLOTS - 1].active == 0) return;
  const double res = slot_sum<NT>(sc, SLOTS - 1, slot_first(sc, SLOTS - 1), red);
  if (threadIdx.x == 0) {
    ctl->res = res;
    ctl->total += SLOTS;
  }
}

__global__ __launch_bounds__(BLOCK) void k_slots_finish(SlotCtl sc, MGCtl *ctl) {
  __shared__ double red[BLOCK / LEPIC_WAVE];
  slots_finish<BLOCK>(sc, ctl, red);
}

template <class T>
struct Vec2 {
  typedef T type __attribute__((ext_vector_type(2), aligned(sizeof(T))));
};

// SWEEPS sweeps from src to dst.  RES: one sweep, the L1 residual after it
// to this slot's partials, the exit decided from the slot before.  !RES: a
// fixed count, zero != 0 when src is known to be 0 everywhere (not read).
//
// A thread owns one pair position (p, jj) of every HZ-th plane: with HZ even
// the parity of its nodes, and with it every LDS offset, is the same in all
// its planes, so a phase has no index arithmetic.
template <class T, int TX, int TY, int TZ, int NT, int HZ, int SWEEPS, bool RES>
__global__ __launch_bounds__(NT) void k_sweep(KLevelT<T> L, const T *src, T *dst, T omega, int ntx,
                                              int nty, int zero, int slot, SlotCtl sc,
                                              MGCtl *ctl) {
  constexpr int H = 2 * SWEEPS + (RES ? 1 : 0);
  constexpr int NP = (TX + 2 * H + 2) / 2;              // pairs per row
  constexpr int BY = TY + 2 * H, BZ = TZ + 2 * H;       // rows of the black array
  constexpr int RY = BY - 2, RZ = BZ - 2;               // rows of the red array
  constexpr int BSY = NP, BSZ = BY * NP, RSY = NP, RSZ = RY * NP;
  constexpr int R = (BZ + HZ - 1) / HZ;                 // planes per thread
  static_assert(HZ % 2 == 0 && NP * BY * HZ <= NT, "a thread per pair of HZ planes");
  __shared__ T sb[BZ * BSZ];
  __shared__ T sr[RZ * RSZ];
  __shared__ double red[NT / LEPIC_WAVE];
  const KGrid &g = L.g;
  const int n1 = g.n1, n2 = g.n2, n3 = g.n3;
  const int64_t nodes = ((int64_t)n1 + 3) * (n2 + 3) * (n3 + 3);
  // consecutive tiles on one XCD (blocks go to the XCDs in turn), so that they
  // find each other's halos in its L2
  const int per = (int)gridDim.x / LEPIC_XCDS;
  const int tile = (int)blockIdx.x < per * LEPIC_XCDS
                       ? ((int)blockIdx.x % LEPIC_XCDS) * per + (int)blockIdx.x / LEPIC_XCDS
                       : (int)blockIdx.x;
  const int bx = tile % ntx, by = (tile / ntx) % nty, bz = tile / (ntx * nty);
  const int xs = 1 + bx * TX, ys = 1 + by * TY, zs = 1 + bz * TZ;
  const int xb = (xs - H) & ~1, yb = ys - H, zb = zs - H;
  const int p = (int)threadIdx.x % NP, jj = ((int)threadIdx.x / NP) % BY,
            h = (int)threadIdx.x / BSZ;
  const bool mine = h < HZ;
  const int j = yb + jj, q = (j + zb + h) & 1;
  const int ir = xb + 2 * p + 1 - q, ib = xb + 2 * p + q;   // the pair's red and black node
  // how far outside the tile, in the plane (H: not a relaxed position)
  auto ring_xy = [&](int i, bool in) {
    const int d = max(max(xs - i, i - (xs + TX - 1)), max(ys - j, j - (ys + TY - 1)));
    return in && i >= 1 && i <= n1 + 1 && j >= 1 && j <= n2 + 1 ? max(d, 0) : H;
  };
  const int ringr = ring_xy(ir, mine && jj >= 1 && jj <= RY);
  const int ringk = ring_xy(ib, mine && jj >= 2 && jj <= RY - 1);

  if (RES && slot > 0) {
    const SlotState st = sc.state[slot - 1];
    const double first = slot_first(sc, slot - 1);
    bool active = false;
    if (st.active) {
      const double res = slot_sum<NT>(sc, slot - 1, first, red);
      active = !sor_stops(res, st.res_s);
      if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc.state[slot].active = active ? 1 : 0;
        sc.state[slot].res_s = res;
        if (!active) {
          ctl->res = res;
          ctl->total += slot;
        }
      }
      // the first idle slot after an odd number of sweeps brings u home
      if (!active && (slot & 1)) {
        const int64_t stride = (int64_t)gridDim.x * NT;
        for (int64_t t = blockIdx.x * (int64_t)NT + threadIdx.x; t < nodes; t += stride)
          dst[t] = src[t];
      }
    } else if (blockIdx.x == 0 && threadIdx.x == 0) {
      sc.state[slot].active = 0;
    }
    if (!active) return;
  } else if (RES && blockIdx.x == 0 && threadIdx.x == 0) {
    sc.state[0].active = 1;
    sc.state[0].res_s = 0.0;
  }
  // Every read is issued before anything waits (a launch starts with a cold
  // L2, so each dependent read costs most of a microsecond), from addresses
  // that need no test of what was read: clamped into the arrays, and nothing
  // that nodes outside the relaxed range bring is used.
  typedef typename Vec2<T>::type V2;
  typedef typename Vec2<int32_t>::type I2;
  const int64_t off0 = (int64_t)(xb + 2 * p) + g.sy * (int64_t)j + g.sz * (int64_t)(zb + h);
  const int64_t step = HZ * g.sz;
  auto inside = [&](int64_t c) { return c < 0 ? 0 : (c > nodes - 2 ? nodes - 2 : c); };
  constexpr int RH = R / 3;   // planes whose b is read before the first wait (more spill)
  V2 uv[R], bv[R];
  int lr[R], lk[R];
  const bool relaxes = min(ringr, ringk) < H;
  if (!zero) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      uv[r] = *reinterpret_cast<const V2 *>(src + inside(off0 + r * step));
  } else {
#pragma unroll
    for (int r = 0; r < R; ++r) uv[r] = V2{T(0), T(0)};
  }
#pragma unroll
  for (int r = 0; r < R; ++r) lr[r] = lk[r] = 1;
  if (relaxes) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const I2 l2 = *reinterpret_cast<const I2 *>(L.bc + inside(off0 + r * step));
      lr[r] = q ? l2.x : l2.y;
      lk[r] = q ? l2.y : l2.x;
    }
  }
  auto read_b = [&](int r) {
    bv[r] = *reinterpret_cast<const V2 *>(L.b + inside(off0 + r * step));
  };
#pragma unroll
  for (int r = 0; r < RH; ++r) read_b(r);
  // class of a node: 0 not relaxed, 1 plasma, 2 Neumann, 3 other
  auto cls_of = [&](int lab, int k) {
    if (lab > 0 || k < 1 || k > n3 + 1) return 0;
    if (lab == 0 && (k == n3 + 1 || j == n2 + 1)) return 0;
    return lab == -1 ? 1 : (lab == -2 ? 2 : 3);
  };
  const int m0 = h * BSZ + jj * BSY + p, e0 = (h - 1) * RSZ + (jj - 1) * RSY + p;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int kk = h + r * HZ, m = m0 + r * HZ * BSZ, e = e0 + r * HZ * RSZ;
    lr[r] = cls_of(lr[r], zb + kk);
    lk[r] = cls_of(lk[r], zb + kk);
    if (off0 + r * step == nodes - 1) uv[r].x = uv[r].y;   // the last node has no pair
    if (mine && kk < BZ) {
      sb[m] = q ? uv[r].y : uv[r].x;
      if (jj >= 1 && jj <= RY && kk >= 1 && kk <= RZ) sr[e] = q ? uv[r].x : uv[r].y;
    }
  }
#pragma unroll
  for (int r = RH; r < R; ++r) read_b(r);   // in flight during the first planes' relaxation
  __syncthreads();
  double a = 0.0;
  auto relax = [&](int cls, T uc, T uw, T ue, T un, T us, T ut, T ub, T bb) {
    if (cls == 2)
      return (T(1) - omega) * uc +
             div_ac(omega * (bb - L.an * un - L.as * us - T(2) * L.ae * ue - L.at * ut - L.ab * ub),
                    L);
    return (T(1) - omega) * uc +
           div_ac(omega * (bb - L.aw * uw - L.an * un - L.as * us - L.ae * ue - L.at * ut -
                           L.ab * ub),
                  L);
  };
  auto resid = [&](T uc, T uw, T ue, T un, T us, T ut, T ub, T bb) {
    const T rij = bb - (L.aw * uw + L.an * un + L.as * us + L.ae * ue + L.ac * uc + L.at * ut +
                        L.ab * ub);
    return fabs((double)rij);
  };
#pragma unroll
  for (int s = 0; s < SWEEPS; ++s) {
    const int red_ring = H - 1 - 2 * s, black_ring = H - 2 - 2 * s;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int kk = h + r * HZ, m = m0 + r * HZ * BSZ, e = e0 + r * HZ * RSZ;
      if (ringr <= red_ring && kk >= H - red_ring && kk <= H + TZ - 1 + red_ring && lr[r])
        sr[e] = relax(lr[r], sr[e], sb[m - q], sb[m + 1 - q], sb[m + BSY], sb[m - BSY],
                      sb[m + BSZ], sb[m - BSZ], q ? bv[r].x : bv[r].y);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int kk = h + r * HZ, m = m0 + r * HZ * BSZ, e = e0 + r * HZ * RSZ;
      if (ringk <= black_ring && kk >= H - black_ring && kk <= H + TZ - 1 + black_ring && lk[r]) {
        const T uw = sr[e - 1 + q], ue = sr[e + q], un = sr[e + RSY], us = sr[e - RSY],
                ut = sr[e + RSZ], ub = sr[e - RSZ], bb = q ? bv[r].y : bv[r].x;
        const T u = relax(lk[r], sb[m], uw, ue, un, us, ut, ub, bb);
        sb[m] = u;
        if (RES && lk[r] == 1 && ringk == 0 && kk >= H && kk <= H + TZ - 1)
          a = a + resid(u, uw, ue, un, us, ut, ub, bb);
      }
    }
    __syncthreads();
  }
  if (RES) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int kk = h + r * HZ, m = m0 + r * HZ * BSZ, e = e0 + r * HZ * RSZ;
      if (ringr == 0 && kk >= H && kk <= H + TZ - 1 && lr[r] == 1)
        a = a + resid(sr[e], sb[m - q], sb[m + 1 - q], sb[m + BSY], sb[m - BSY], sb[m + BSZ],
                      sb[m - BSZ], q ? bv[r].x : bv[r].y);
    }
  }
  // the tile's nodes, with the ghost layer on the domain's faces
  const int x0 = bx == 0 ? 0 : xs, x1 = bx == ntx - 1 ? n1 + 2 : xs + TX - 1;
  const int y0 = by == 0 ? 0 : ys, y1 = by == nty - 1 ? n2 + 2 : ys + TY - 1;
  const int z0 = bz == 0 ? 0 : zs,
            z1 = tile + ntx * nty >= (int)gridDim.x ? n3 + 2 : zs + TZ - 1;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int kk = h + r * HZ, m = m0 + r * HZ * BSZ, e = e0 + r * HZ * RSZ;
    const int k = zb + kk, i = xb + 2 * p;
    if (!mine || j < y0 || j > y1 || k < z0 || k > z1) continue;
    const T ur = sr[e], uk = sb[m];
    const T lo = q ? ur : uk, hi = q ? uk : ur;
    T *d = dst + (off0 + r * step);
    if (i >= x0 && i < x1) {
      *reinterpret_cast<V2 *>(d) = V2{lo, hi};
    } else if (i == x1) {
      d[0] = lo;
    } else if (i == x0 - 1 && i < x1) {
      d[1] = hi;
    }
  }
  if (RES) {
    for (int d = LEPIC_WAVE / 2; d > 0; d >>= 1) a = a + __shfl_down(a, d);
    if (__lane_id() == 0) red[threadIdx.x / LEPIC_WAVE] = a;
    __syncthreads();
    if (threadIdx.x == 0) {
      double b = 0.0;
      for (int w = 0; w < NT / LEPIC_WAVE; ++w) b = b + red[w];
      sc.partials[(int64_t)(slot & 1) * sc.nparts + blockIdx.x] = b;
    }
  }
}

// --------------------------------------------------------------------------
// Levels with periodic walls: two launches per sweep and one at the end.
// sor_rb copies the ghost planes after every colour; here a colour reads
// through the copies (per_source: the node that a boundary node has its value
// from) and the copies are made once, at the end.  Only the first red half
// reads the ghosts as they stand.  The black residual is summed with the black
// half, the red one with the next sweep's red half, which goes to the other of
// two arrays of red values (X; black stays in u): if the decision, taken by
// every block of the black half as in k_sweep, ends the sor_rb, that half is
// not used.  9 launches of 6 to 7 us in place of 32 of 3 to 4 (two colours, four copies,
// residual, decision, four times): solve of 96 x 40 x 72 14.3 -> 10.3 ms.
// --------------------------------------------------------------------------
constexpr int PER_BLOCKS = 1024;   // block residuals that every block sums

__device__ inline bool per_ok(int lab) { return lab == 0 || lab == -2; }

// The node (i, j, k) has its value from after the copies of sors.f90:184-239
// (y planes, then z planes): j and k of that node.
template <class T>
__device__ inline void per_source(const KLevelT<T> &L, int i, int &j, int &k) {
  const KGrid &g = L.g;
  if (k == g.n3 + 1 && per_ok(L.bc[gidx(g, i, j, g.n3 + 1)])) k = 1;
  else if (k == 0 && per_ok(L.bc[gidx(g, i, j, 1)])) k = g.n3;
  if (j == g.n2 + 1 && per_ok(L.bc[gidx(g, i, g.n2 + 1, k)])) j = 1;
  else if (j == 0 && per_ok(L.bc[gidx(g, i, 1, k)])) j = g.n2;
}

// u where a node of one colour's array X (nodes 1..n+1) is read, through the
// copies with pull.
template <class T>
__device__ inline T per_read(const KLevelT<T> &L, const T *X, int i, int j, int k, bool pull) {
  const KGrid &g = L.g;
  if (pull) per_source(L, i, j, k);
  const bool in = i >= 1 && i <= g.n1 + 1 && j >= 1 && j <= g.n2 + 1 && k >= 1 && k <= g.n3 + 1;
  return (in ? X : (const T *)L.u)[gidx(g, i, j, k)];
}

template <class T>
struct Nbr6 {
  T uw, ue, un, us, ut, ub;
};

// The six neighbours of a node of [1, n+1].
template <class T>
__device__ inline Nbr6<T> per_neighbours(const KLevelT<T> &L, const T *X, int i, int j, int k,
                                         bool pull) {
  const KGrid &g = L.g;
  const int64_t c = gidx(g, i, j, k);
  Nbr6<T> v;
  if (j > 1 && j < g.n2 && k > 1 && k < g.n3) {
    v.uw = (i == 1 ? (const T *)L.u : X)[c - 1];
    v.ue = (i == g.n1 + 1 ? (const T *)L.u : X)[c + 1];
    v.un = X[c + g.sy]; v.us = X[c - g.sy];
    v.ut = X[c + g.sz]; v.ub = X[c - g.sz];
  } else {
    v.uw = per_read(L, X, i - 1, j, k, pull); v.ue = per_read(L, X, i + 1, j, k, pull);
    v.un = per_read(L, X, i, j + 1, k, pull); v.us = per_read(L, X, i, j - 1, k, pull);
    v.ut = per_read(L, X, i, j, k + 1, pull); v.ub = per_read(L, X, i, j, k - 1, pull);
  }
  return v;
}

// Node t of a colour: false when it is none.
template <class T>
__device__ inline bool per_node(const KLevelT<T> &L, int colour, int t, int &i, int &j, int &k) {
  const KGrid &g = L.g;
  const uint32_t r = mdiv_q((uint32_t)t, L.d_h1), rk = mdiv_q(r, L.d_n2p1);
  j = 1 + (int)(r - rk * (uint32_t)(g.n2 + 1));
  k = 1 + (int)rk;
  const int red = 1 + ((j + k) & 1);   // red: i + j + k odd
  i = (colour ? 3 - red : red) + 2 * (t - (int)r * (g.n1 / 2 + 1));
  return i <= g.n1 + 1;
}

template <class T>
__device__ inline double per_resid(const KLevelT<T> &L, T b, T uc, const Nbr6<T> &v) {
  const T rij = b - (L.aw * v.uw + L.an * v.un + L.as * v.us + L.ae * v.ue + L.ac * uc +
                     L.at * v.ut + L.ab * v.ub);
  return fabs((double)rij);
}

// A block's sum of a to out[blockIdx.x].
__device__ inline void per_partial(double a, double *out) {
  __shared__ double red[BLOCK / LEPIC_WAVE];
  a = wave_sum(a);
  if (__lane_id() == 0) red[threadIdx.x / LEPIC_WAVE] = a;
  __syncthreads();
  if (threadIdx.x == 0) {
    double b = 0.0;
    for (int w = 0; w < BLOCK / LEPIC_WAVE; ++w) b = b + red[w];
    out[blockIdx.x] = b;
  }
}

// The residual after sweep s from its partials (black of even sweeps, of odd
// ones, red): a thread's share, and the block's sum of them in every thread.
__device__ inline double per_share(const SlotCtl &sc, int s) {
  double v[2 * PER_BLOCKS / BLOCK];
#pragma unroll
  for (int q = 0; q < PER_BLOCKS / BLOCK; ++q) {
    const int64_t t = threadIdx.x + q * BLOCK;
    v[2 * q] = t < sc.nparts ? sc.partials[(s & 1) * sc.nparts + t] : 0.0;
    v[2 * q + 1] = t < sc.nparts ? sc.partials[2 * sc.nparts + t] : 0.0;
  }
  double a = 0.0;
#pragma unroll
  for (int q = 0; q < 2 * PER_BLOCKS / BLOCK; ++q) a = a + v[q];
  return a;
}

__device__ inline double per_sum(double a) {
  __shared__ double red[BLOCK / LEPIC_WAVE];
  a = wave_sum(a);
  if (__lane_id() == 0) red[threadIdx.x / LEPIC_WAVE] = a;
  __syncthreads();
  double r = 0.0;
  for (int w = 0; w < BLOCK / LEPIC_WAVE; ++w) r = r + red[w];
  __syncthreads();
  return r;
}

// An edge ghost that the y copy writes and the z copy does not (labels that
// differ between it and the node beside it) takes, from a ghost or copied node
// of its source plane, the value before the last black half: the owner of a
// black node leaves it there, k_per_end does the others.
template <class T>
__device__ inline void per_edge(const KLevelT<T> &L, int i, int j, int k, T old) {
  const KGrid &g = L.g;
  auto ok = [&](int b, int c) { return per_ok(L.bc[gidx(g, i, b, c)]); };
  if (j == g.n2 && k == 1 && ok(1, g.n3 + 1) && !ok(0, g.n3 + 1) && ok(g.n2, g.n3 + 1))
    L.u[gidx(g, i, 0, g.n3 + 1)] = old;
  if (j == g.n2 && k == g.n3 && ok(1, 0) && !ok(0, 1) && ok(g.n2, 1)) L.u[gidx(g, i, 0, 0)] = old;
  if (j == 1 && k == g.n3 && ok(g.n2 + 1, 0) && !ok(g.n2 + 1, 1) && ok(1, 1))
    L.u[gidx(g, i, g.n2 + 1, 0)] = old;
}

// One half of sweep s.  colour 0: red, from X (s even: u, else u2) to Xn;
// colour 1: black in u, the red values in X.  ctl null: a fixed sweep count.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_per_half(KLevelT<T> L, const T *X, T *Xn, int colour,
                                                    T omega, int s, SlotCtl sc, MGCtl *ctl) {
  const bool judged = ctl != nullptr;
  const KGrid &g = L.g;
  const uint32_t n = (uint32_t)(g.n1 / 2 + 1) * (uint32_t)(g.n2 + 1) * (uint32_t)(g.n3 + 1);
  const T *own = colour ? (const T *)L.u : X, *other = colour ? X : (const T *)L.u;
  T *out = colour ? L.u : Xn;
  const bool pull = colour == 1 || s > 0;
  int i = 0, j = 0, k = 0, lab = 1;
  T b = T(0), uc = T(0);
  Nbr6<T> v = {};
  bool node = false;
  auto load = [&](uint32_t t) {
    node = t < n && per_node(L, colour, (int)t, i, j, k);
    if (!node) return;
    const int64_t c = gidx(g, i, j, k);
    lab = L.bc[c];
    b = L.b[c];
    uc = own[c];
    v = per_neighbours(L, other, i, j, k, pull);
  };
  // everything the launch reads is under way before the decision
  auto nw = walk_strided<uint32_t>(n, (int)blockIdx.x, (int)gridDim.x, (int)threadIdx.x, BLOCK);
  load(nw.t);
  if (judged && s > 0) {
    const double share = colour ? per_share(sc, s - 1) : 0.0;
    const SlotState st = sc.state[s - 1];
    if (colour == 0) {
      if (st.active == 0) return;
    } else {
      bool active = st.active != 0;
      double res = 0.0;
      if (active) {
        res = per_sum(share);
        active = !sor_stops(res, st.res_s);
        if (!active && blockIdx.x == 0 && threadIdx.x == 0) {
          ctl->res = res;
          ctl->total += s;
        }
      }
      if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc.state[s].active = active ? 1 : 0;
        sc.state[s].res_s = res;
      }
      if (!active) return;
    }
  } else if (judged && colour == 1 && blockIdx.x == 0 && threadIdx.x == 0) {
    sc.state[0].active = 1;
    sc.state[0].res_s = 0.0;
  }
  double a = 0.0;
  for (;;) {
    if (node) {
      const int64_t c = gidx(g, i, j, k);
      if (colour == 1 && (j == 1 || j == g.n2) && (k == 1 || k == g.n3)) per_edge(L, i, j, k, uc);
      if (judged && colour == 0 && s > 0 && lab == -1) a = a + per_resid(L, b, uc, v);
      if (!(lab > 0 || (lab == 0 && (k == g.n3 + 1 || j == g.n2 + 1)))) {
        if (lab == -2)
          uc = (T(1) - omega) * uc +
               div_ac(omega * (b - L.an * v.un - L.as * v.us - T(2) * L.ae * v.ue - L.at * v.ut -
                               L.ab * v.ub),
                      L);
        else
          uc = (T(1) - omega) * uc +
               div_ac(omega * (b - L.aw * v.uw - L.an * v.un - L.as * v.us - L.ae * v.ue -
                               L.at * v.ut - L.ab * v.ub),
                      L);
        out[c] = uc;
      } else if (colour == 0) {
        out[c] = uc;   // the other array's copy of a node that is not relaxed
      }
      if (judged && colour == 1 && lab == -1) a = a + per_resid(L, b, uc, v);
    }
    nw.t += nw.step;
    if (nw.t >= nw.end) break;
    load(nw.t);
  }
  if (judged && (colour == 1 || s > 0))
    per_partial(a, sc.partials + (colour ? (int64_t)(s & 1) : 2) * sc.nparts);
}

// The end of a sor_rb: the red values back in u, the periodic copies, and with
// resid the last red residual (when all sweeps ran).  count: the sweeps, of a
// fixed count (ctl null).
template <class T>
__global__ __launch_bounds__(BLOCK) void k_per_end(KLevelT<T> L, MDiv d_n2p3, const T *u2, int count,
                                                   int resid, SlotCtl sc, MGCtl *ctl) {
  bool all = false;
  if (ctl) {
    count = 0;
    for (int s = 0; s < SLOTS; ++s) count += sc.state[s].active != 0 ? 1 : 0;
    all = count == SLOTS;
    if (all && blockIdx.x == 0 && threadIdx.x == 0) ctl->total += SLOTS;
  }
  const KGrid &g = L.g;
  const T *X = (count & 1) ? u2 : (const T *)L.u;
  const int nx = g.n1 + 3;
  double a = 0.0;
  const auto nw = walk_strided<uint32_t>((int64_t)nx * (g.n2 + 3) * (g.n3 + 3), (int)blockIdx.x,
                                         (int)gridDim.x, (int)threadIdx.x, BLOCK);
  for (uint32_t t = nw.t; t < nw.end; t += nw.step) {
    const uint32_t r = mdiv_q(t, L.d_n1p3), rk = mdiv_q(r, d_n2p3);
    const int i = (int)(t - r * (uint32_t)nx), j = (int)(r - rk * (uint32_t)(g.n2 + 3)),
              k = (int)rk;
    const bool is_red = (i + j + k) & 1;
    int sj = j, sk = k;
    per_source(L, i, sj, sk);
    const bool in = i >= 1 && i <= g.n1 + 1 && j >= 1 && j <= g.n2 + 1 && k >= 1 && k <= g.n3 + 1;
    if (resid && all && in && is_red && L.bc[t] == -1)
      a = a + per_resid(L, L.b[t], X[t], per_neighbours(L, (const T *)L.u, i, j, k, true));
    if (sj != j && (sk == 0 || sk == g.n3 + 1)) {   // an edge ghost (per_edge)
      const bool copied = per_ok(L.bc[gidx(g, i, sj, sk == 0 ? 1 : g.n3 + 1)]);
      if (copied && !is_red) continue;
      if (copied) sk = sk == 0 ? g.n3 : 1;
    }
    if (sj != j || sk != k) L.u[t] = per_read(L, is_red ? X : (const T *)L.u, i, sj, sk, false);
    else if (is_red && in && (count & 1)) L.u[t] = u2[t];
  }
  if (resid && all) per_partial(a, sc.partials + 2 * sc.nparts);
}

__global__ __launch_bounds__(BLOCK) void k_per_res(SlotCtl sc, MGCtl *ctl) {
  if (sc.state[SLOTS - 1].active == 0) return;
  const double res = per_sum(per_share(sc, SLOTS - 1));
  if (threadIdx.x == 0) ctl->res = res;
}

// r_pbc: residual of plane k = m, the periodic image of k = 0
// (mg.f90:322-392).  The reference loops over coarse (j, i) and each
// iteration writes up to nine overlapping entries, the later iteration
// winning; here one thread per entry finds that last writer (largest jr,
// then largest ir) and applies its branch: getres when bcnd(ir,jr,m+1) <= 0,
// else 0.  The two branches guard the (ir, jr-1) entry differently.
template <class T, class B>
__device__ inline void rpbc_entry(const KLevelT<T, B> &F, T *rp, int flag_nmn, int64_t t) {
  const KGrid &g = F.g;
  const int64_t rs = g.n1 + 2;
  const int64_t total = rs * (g.n2 + 2);
  if (t >= total) return;
  const uint32_t tt = (uint32_t)t, bb = mdiv_q(tt, F.d_n1p2);
  const int a = (int)(tt - bb * (uint32_t)rs), b = (int)bb;
  const int m = g.n3, N1 = g.n1 + 1, N2 = g.n2 + 1;
  T val = T(0);
  bool found = false;
  for (int jr = b + 1; jr >= b - 1 && !found; --jr) {
    if (jr < 1 || jr > N2 || (jr % 2) == 0) continue;
    const int db = b - jr;
    for (int ir = a + 1; ir >= a - 1 && !found; --ir) {
      if (ir < 1 || ir > N1 || (ir % 2) == 0) continue;
      const int da = a - ir;
      const bool live = F.bc[gidx(g, ir, jr, m + 1)] <= 0;
      bool writes = true;
      if (da == -1 && ir == 1) writes = false;
      if (da == 1 && ir == N1) writes = false;
      if (db == 1 && jr == N2) writes = false;
      if (db == -1) {
        if (jr == 1) writes = false;
        if (live && da == 0 && ir == 1) writes = false;  // getres branch also needs ir /= 1
      }
      if (!writes) continue;
      found = true;
      val = live ? getres(F, a, b, m, flag_nmn) : T(0);
    }
  }
  rp[t] = val;
}

template <class T>
__global__ void k_rpbc(KLevelT<T> F, T *rp, int flag_nmn) {
  rpbc_entry(F, rp, flag_nmn, blockIdx.x * (int64_t)blockDim.x + threadIdx.x);
}

// Restriction (mg.f90:413-718): coarse labels injected from the fine grid and
// the 27-point full-weighting residual with the reference's neighbour rules.

// The labels of coarse node (i, j, k) and of the ghost nodes next to it; the
// node's own.
template <class T, class LB>
__device__ inline LB restrict_labels(const KLevelT<T, LB> &F, const KLevelT<T, LB> &C, int i, int j,
                                     int k) {
  const KGrid &g = F.g, &gc = C.g;
  const int ir = 2 * i - 1, jr = 2 * j - 1, kr = 2 * k - 1;
  const LB *bc = F.bc;
  LB *bc2 = C.bc;
  const LB lab = bc[gidx(g, ir, jr, kr)];
  bc2[gidx(gc, i, j, k)] = lab;
  if (ir == 1) bc2[gidx(gc, 0, j, k)] = bc[gidx(g, 0, jr, kr)];
  if (ir == g.n1 + 1) bc2[gidx(gc, g.n1 / 2 + 2, j, k)] = bc[gidx(g, g.n1 + 2, jr, kr)];
  if (jr == 1) bc2[gidx(gc, i, 0, k)] = bc[gidx(g, ir, 0, kr)];
  if (jr == g.n2 + 1) bc2[gidx(gc, i, g.n2 / 2 + 2, k)] = bc[gidx(g, ir, g.n2 + 2, kr)];
  if (kr == 1) bc2[gidx(gc, i, j, 0)] = bc[gidx(g, ir, jr, 0)];
  if (kr == g.n3 + 1) bc2[gidx(gc, i, j, g.n3 / 2 + 2)] = bc[gidx(g, ir, jr, g.n3 + 2)];
  return lab;
}

// The weighted sum; r(a, b, c): the residual at that offset, 0 where the
// reference takes none.
template <class T, class RD>
__device__ inline T restrict_sum(RD r) {
  return (T(8) * r(0, 0, 0) +
          T(4) * (r(1, 0, 0) + r(-1, 0, 0) + r(0, 1, 0) + r(0, -1, 0) + r(0, 0, 1) + r(0, 0, -1)) +
          T(2) * (r(1, 1, 0) + r(-1, 1, 0) + r(1, -1, 0) + r(-1, -1, 0) + r(1, 0, 1) + r(-1, 0, 1) +
                  r(0, 1, 1) + r(0, -1, 1) + r(1, 0, -1) + r(-1, 0, -1) + r(0, 1, -1) +
                  r(0, -1, -1)) +
          r(1, 1, 1) + r(-1, 1, 1) + r(1, -1, 1) + r(-1, -1, 1) + r(1, 1, -1) + r(-1, 1, -1) +
          r(1, -1, -1) + r(-1, -1, -1)) /
         T(64);
}

// R != nullptr: getres of every node of the fine residual range, formed
// beforehand (the same expression, so the same bits).  masked: R is 0 on the
// ghost nodes and on electrodes outside the plane j = n2 (which the wrap of
// j = 1 reads whatever its label), so that the 27 values need no label.
template <class T, class LB>
__device__ inline void restrict_node(const KLevelT<T, LB> &F, const KLevelT<T, LB> &C, const T *rp,
                                     int flag_nmn, int64_t t, const T *R = nullptr,
                                     bool masked = false) {
  const KGrid &g = F.g;
  const KGrid &gc = C.g;
  const int m = g.n3;
  const int kp = m / 2 + 1;
  int64_t ni = g.n1 / 2 + 1, nj = g.n2 / 2 + 1;
  if (t >= ni * nj * kp) return;
  const uint32_t tt = (uint32_t)t, r = mdiv_q(tt, F.d_h1), rk = mdiv_q(r, F.d_h2);
  int i = 1 + (int)(tt - r * (uint32_t)ni);
  int j = 1 + (int)(r - rk * (uint32_t)nj);
  int k = 1 + (int)rk;
  const int ir = 2 * i - 1, jr = 2 * j - 1, kr = 2 * k - 1;
  const int N1 = g.n1 + 1, N2 = g.n2 + 1, M1 = m + 1;
  const LB *bc = F.bc;
  const LB lab = restrict_labels(F, C, i, j, k);
  T re = T(0);
  if (lab <= 0 && masked && jr != 1 && (kr != 1 || !rp)) {
    const int64_t c = gidx(g, ir, jr, kr);
    T v[3][3][3];
#pragma unroll
    for (int b_ = 0; b_ < 3; ++b_) {
      const bool edge = jr + b_ - 1 == g.n2;
#pragma unroll
      for (int c_ = 0; c_ < 3; ++c_)
#pragma unroll
        for (int a_ = 0; a_ < 3; ++a_) {
          const int64_t q = c + (a_ - 1) + g.sy * (b_ - 1) + g.sz * (c_ - 1);
          v[a_][b_][c_] = R[q];
          if (edge && bc[q] > 0) v[a_][b_][c_] = T(0);
        }
    }
    re = restrict_sum<T>([&](int a, int b_, int c_) { return v[a + 1][b_ + 1][c_ + 1]; });
  } else if (lab <= 0) {
    const int n2 = g.n2;
    const int64_t rs = g.n1 + 2;
    auto B = [&](int a, int b_, int c) { return bc[gidx(g, a, b_, c)]; };
    auto GR = [&](int a, int b_, int c) {
      const bool in = a >= 1 && a <= N1 && b_ >= 1 && b_ <= N2 && c >= 1 && c <= M1;
      return (R && in) ? R[gidx(g, a, b_, c)] : getres(F, a, b_, c, flag_nmn);
    };
    auto RP = [&](int a, int b_) { return rp ? rp[(int64_t)a + rs * b_] : T(0); };
    const bool kb = (kr == 1);
    T r000 = 0, rpp0 = 0, rp00 = 0, rpm0 = 0, r0m0 = 0, rmm0 = 0, rm00 = 0, rmp0 = 0,
      r0p0 = 0, r00p = 0, rppp = 0, rp0p = 0, rpmp = 0, r0mp = 0, rmmp = 0, rm0p = 0,
      rmpp = 0, r0pp = 0, r00m = 0, rppm = 0, rp0m = 0, rpmm = 0, r0mm = 0, rmmm = 0,
      rm0m = 0, rmpm = 0, r0pm = 0;
    r000 = GR(ir, jr, kr);
    if (ir != N1 && jr != N2) { if (B(ir + 1, jr + 1, kr) <= 0) rpp0 = GR(ir + 1, jr + 1, kr); }
    if (ir != N1) { if (B(ir + 1, jr, kr) <= 0) rp00 = GR(ir + 1, jr, kr); }
    if (B(ir + 1, jr - 1, kr) <= 0) {
      if (ir != N1 && jr != 1) rpm0 = GR(ir + 1, jr - 1, kr);
      else if (jr == 1) rpm0 = GR(ir + 1, n2, kr);
    }
    if (B(ir, jr - 1, kr) <= 0) {
      if (jr == 1) r0m0 = GR(ir, n2, kr);
      else r0m0 = GR(ir, jr - 1, kr);
    }
    if (B(ir - 1, jr - 1, kr) <= 0 && ir != 1) {
      if (jr != 1) rmm0 = GR(ir - 1, jr - 1, kr);
      else rmm0 = GR(ir - 1, n2, kr);
    }
    if (ir != 1) { if (B(ir - 1, jr, kr) <= 0) rm00 = GR(ir - 1, jr, kr); }
    if (ir != 1 && jr != N2) { if (B(ir - 1, jr + 1, kr) <= 0) rmp0 = GR(ir - 1, jr + 1, kr); }
    if (jr != N2) { if (B(ir, jr + 1, kr) <= 0) r0p0 = GR(ir, jr + 1, kr); }
    if (kr != M1) { if (B(ir, jr, kr + 1) <= 0) r00p = GR(ir, jr, kr + 1); }
    if (ir != N1 && jr != N2 && kr != M1) {
      if (B(ir + 1, jr + 1, kr + 1) <= 0) rppp = GR(ir + 1, jr + 1, kr + 1);
    }
    if (ir != N1 && kr != M1) { if (B(ir + 1, jr, kr + 1) <= 0) rp0p = GR(ir + 1, jr, kr + 1); }
    if (B(ir + 1, jr - 1, kr + 1) <= 0) {
      if (ir != N1 && jr != 1 && kr != M1) rpmp = GR(ir + 1, jr - 1, kr + 1);
      else if (jr == 1 && kr != M1) rpmp = GR(ir + 1, n2, kr + 1);
    }
    if (B(ir, jr - 1, kr + 1) <= 0) {
      if (jr != 1 && kr != M1) r0mp = GR(ir, jr - 1, kr + 1);
      else if (jr == 1 && kr != M1) r0mp = GR(ir, n2, kr + 1);
    }
    if (B(ir - 1, jr - 1, kr + 1) <= 0 && ir != 1) {
      if (jr != 1 && kr != M1) rmmp = GR(ir - 1, jr - 1, kr + 1);
      else if (jr == 1 && kr != M1) rmmp = GR(ir - 1, n2, kr + 1);
    }
    if (ir != 1 && kr != M1) { if (B(ir - 1, jr, kr + 1) <= 0) rm0p = GR(ir - 1, jr, kr + 1); }
    if (ir != 1 && jr != N2 && kr != M1) {
      if (B(ir - 1, jr + 1, kr + 1) <= 0) rmpp = GR(ir - 1, jr + 1, kr + 1);
    }
    if (jr != N2 && kr != M1) { if (B(ir, jr + 1, kr + 1) <= 0) r0pp = GR(ir, jr + 1, kr + 1); }
    if (B(ir, jr, kr - 1) <= 0) {
      if (kb) r00m = RP(ir, jr);
      else r00m = GR(ir, jr, kr - 1);
    }
    if (B(ir + 1, jr + 1, kr - 1) <= 0) {
      if (kb) { if (ir != N1 && jr != N2) rppm = RP(ir + 1, jr + 1); }
      else { if (ir != N1 && jr != N2) rppm = GR(ir + 1, jr + 1, kr - 1); }
    }
    if (B(ir + 1, jr, kr - 1) <= 0) {
      if (kb) { if (ir != N1) rp0m = RP(ir + 1, jr); }
      else { if (ir != N1) rp0m = GR(ir + 1, jr, kr - 1); }
    }
    if (B(ir + 1, jr - 1, kr - 1) <= 0) {
      if (kb) { if (ir != N1 && jr != 1) rpmm = RP(ir + 1, jr - 1); }
      else {
        if (ir != N1 && jr != 1) rpmm = GR(ir + 1, jr - 1, kr - 1);
        if (jr == 1) rpmm = GR(ir + 1, n2, kr - 1);
      }
    }
    if (B(ir, jr - 1, kr - 1) <= 0) {
      if (kb) { if (jr != 1) r0mm = RP(ir, jr - 1); }
      else {
        if (jr != 1) r0mm = GR(ir, jr - 1, kr - 1);
        if (jr == 1) r0mm = GR(ir, n2, kr - 1);
      }
    }
    if (B(ir - 1, jr - 1, kr - 1) <= 0 && ir != 1) {
      if (kb) { if (jr != 1) rmmm = RP(ir - 1, jr - 1); }
      else {
        if (jr != 1) rmmm = GR(ir - 1, jr - 1, kr - 1);
        if (jr == 1) rmmm = GR(ir - 1, n2, kr - 1);
      }
    }
    if (B(ir - 1, jr, kr - 1) <= 0 && ir != 1) {
      if (kb) rm0m = RP(ir - 1, jr);
      else rm0m = GR(ir - 1, jr, kr - 1);
    }
    if (B(ir - 1, jr + 1, kr - 1) <= 0 && ir != 1) {
      if (kb) { if (jr != N2) rmpm = RP(ir - 1, jr + 1); }
      else { if (jr != N2) rmpm = GR(ir - 1, jr + 1, kr - 1); }
    }
    if (B(ir, jr + 1, kr - 1) <= 0) {
      if (kb) { if (jr != N2) r0pm = RP(ir, jr + 1); }
      else { if (jr != N2) r0pm = GR(ir, jr + 1, kr - 1); }
    }
    re = (T(8) * r000 + T(4) * (rp00 + rm00 + r0p0 + r0m0 + r00p + r00m) +
          T(2) * (rpp0 + rmp0 + rpm0 + rmm0 + rp0p + rm0p + r0pp + r0mp + rp0m + rm0m + r0pm + r0mm) +
          rppp + rmpp + rpmp + rmmp + rppm + rmpm + rpmm + rmmm) /
         T(64);
  }
  C.b[gidx(gc, i, j, k)] = re;
}

template <class T>
__global__ __launch_bounds__(BLOCK) void k_restrict(KLevelT<T> F, KLevelT<T> C, const T *rp,
                                                    int flag_nmn, const T *R) {
  restrict_node(F, C, rp, flag_nmn, blockIdx.x * (int64_t)BLOCK + threadIdx.x, R);
}

// The restriction without periodic walls: a block takes RCX x RCY x RCZ coarse
// nodes (one per thread; 16 x 4 x 4, on narrow grids 4 x 8 x 8), forms getres (mg.f90:809-848) of the fine nodes they
// read in LDS, 0 where the reference takes none, and sums the 27 values there.
// The residual goes to memory and back otherwise, and 27 labels are waited for
// before the values they admit: 16 + 15 us at 128^3, 11 + 5 at 32^3 (FP64), 87
// + 78 at 256^3 (FP32); this launch 20, 6.5 and 90.  The wrap of j = 1 (labels
// <= 0 there) takes the general routine.  fin != nullptr: one more block, the
// last, closes the sor_rb before it (slots_finish).
template <class T, int RCX, int RCY, int RCZ>
__global__ __launch_bounds__(BLOCK) void k_restrict_tile(KLevelT<T> F, KLevelT<T> C, int flag_nmn,
                                                         int ntx, int nty, SlotCtl sc, MGCtl *fin) {
  static_assert(RCX * RCY * RCZ == BLOCK, "a thread per coarse node");
  constexpr int FX = 2 * RCX + 1, FY = 2 * RCY + 1, FZ = 2 * RCZ + 1;
  constexpr int UN = sizeof(T) == 8 ? 11 : 4;   // nodes of a thread read before the first wait
  __shared__ T R[FX * FY * FZ];
  if (fin && blockIdx.x == gridDim.x - 1) {
    __shared__ double red[BLOCK / LEPIC_WAVE];
    slots_finish<BLOCK>(sc, fin, red);
    return;
  }
  const KGrid &g = F.g;
  const int per = (int)(gridDim.x - (fin ? 1 : 0)) / LEPIC_XCDS;   // consecutive tiles on one XCD
  const int tile = (int)blockIdx.x < per * LEPIC_XCDS
                       ? ((int)blockIdx.x % LEPIC_XCDS) * per + (int)blockIdx.x / LEPIC_XCDS
                       : (int)blockIdx.x;
  const int bx = tile % ntx, by = (tile / ntx) % nty, bz = tile / (ntx * nty);
  const int x0 = 2 * bx * RCX, y0 = 2 * by * RCY, z0 = 2 * bz * RCZ;   // R's first fine node
#pragma unroll 1
  for (int t0 = threadIdx.x; t0 < FX * FY * FZ; t0 += UN * BLOCK) {
    // read within the residual range whatever the node, so that no read waits for a test
    int lab[UN];
    bool first[UN];
    T v[UN][8];
#pragma unroll
    for (int e = 0; e < UN; ++e) {
      const int t = imin(t0 + e * BLOCK, FX * FY * FZ - 1);
      const int z = t / (FX * FY), r = t - z * (FX * FY), y = r / FX, x = r - y * FX;
      const int i = imax(1, imin(g.n1 + 1, x0 + x)), j = imax(1, imin(g.n2 + 1, y0 + y)),
                k = imax(1, imin(g.n3 + 1, z0 + z));
      const int64_t c = gidx(g, i, j, k);
      const T *u = F.u;
      lab[e] = F.bc[c];
      v[e][0] = F.b[c];
      v[e][1] = u[c - 1]; v[e][2] = u[c + 1];
      v[e][3] = u[c + g.sy]; v[e][4] = u[c - g.sy];
      v[e][5] = u[c]; v[e][6] = u[c + g.sz]; v[e][7] = u[c - g.sz];
      if (i != x0 + x || j != y0 + y || k != z0 + z) lab[e] = 1;
      first[e] = i == 1 && flag_nmn == 1;
    }
#pragma unroll
    for (int e = 0; e < UN; ++e) {
      const int t = t0 + e * BLOCK;
      const T aw = first[e] ? T(0) : F.aw, ae = first[e] ? T(2) * F.ae : F.ae,
              uw = first[e] ? T(0) : v[e][1];
      const T res = v[e][0] - (aw * uw + ae * v[e][2] + F.an * v[e][3] + F.as * v[e][4] +
                               F.ac * v[e][5] + F.at * v[e][6] + F.ab * v[e][7]);
      if (t < FX * FY * FZ) R[t] = lab[e] <= 0 ? res : T(0);
    }
  }
  __syncthreads();
  const int lx = (int)threadIdx.x % RCX, ly = (int)threadIdx.x / RCX % RCY,
            lz = (int)threadIdx.x / (RCX * RCY);
  const int i = 1 + bx * RCX + lx, j = 1 + by * RCY + ly, k = 1 + bz * RCZ + lz;
  const int ni = g.n1 / 2 + 1, nj = g.n2 / 2 + 1, nk = g.n3 / 2 + 1;
  if (i > ni || j > nj || k > nk) return;
  const int lab = F.bc[gidx(g, 2 * i - 1, 2 * j - 1, 2 * k - 1)];
  if (lab <= 0 && j == 1) {
    restrict_node(F, C, (const T *)nullptr, flag_nmn, (i - 1) + (int64_t)ni * (nj * (int64_t)(k - 1)));
    return;
  }
  restrict_labels(F, C, i, j, k);
  T re = T(0);
  if (lab <= 0) {
    const T *c = R + (2 * lx + 1) + FX * (2 * ly + 1) + FX * FY * (2 * lz + 1);
    re = restrict_sum<T>([&](int a, int b, int c_) { return c[a + FX * b + FX * FY * c_]; });
  }
  C.b[gidx(C.g, i, j, k)] = re;
}

// The periodic restriction's first half: getres (mg.f90:809-848) at every node of
// the fine level's residual range (1..n+1 in each direction) into R, once
// per node instead of once per coarse neighbour that reads it, and the
// coarse correction u zeroed (nc nodes).  The restriction's few getres
// calls outside that range (the n2 wrap at i = n1 + 2) still go to getres.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_getres(KLevelT<T> F, T *R, T *cu, int64_t nc,
                                                  int flag_nmn) {
  const int64_t t = blockIdx.x * (int64_t)BLOCK + threadIdx.x;
  if (t < nc) cu[t] = T(0);
  const KGrid &g = F.g;
  const int64_t nx = g.n1 + 1, ny = g.n2 + 1, nz = g.n3 + 1;
  if (t >= nx * ny * nz) return;
  const uint32_t tt = (uint32_t)t, r = mdiv_q(tt, F.d_n1p1), rk = mdiv_q(r, F.d_n2p1);
  const int i = 1 + (int)(tt - r * (uint32_t)nx);
  const int j = 1 + (int)(r - rk * (uint32_t)ny);
  const int k = 1 + (int)rk;
  R[gidx(g, i, j, k)] = getres(F, i, j, k, flag_nmn);
}

// Prolongation (mg.f90:886-935): one thread per coarse node updates its 8
// fine nodes (disjoint between threads).
template <class T, class B>
__device__ inline void prolong_node(const KLevelT<T, B> &F, const KLevelT<T, B> &C, int64_t t) {
  const KGrid &g = F.g;
  const KGrid &gc = C.g;
  const int kp = g.n3 / 2 + 1;
  int64_t ni = g.n1 / 2 + 1, nj = g.n2 / 2 + 1;
  if (t >= ni * nj * kp) return;
  const uint32_t tt = (uint32_t)t, r = mdiv_q(tt, F.d_h1), rk = mdiv_q(r, F.d_h2);
  int i = 1 + (int)(tt - r * (uint32_t)ni);
  int j = 1 + (int)(r - rk * (uint32_t)nj);
  int k = 1 + (int)rk;
  const T *e = C.u;
  T r000 = e[gidx(gc, i, j, k)], r0m0 = e[gidx(gc, i, j - 1, k)],
         rmm0 = e[gidx(gc, i - 1, j - 1, k)], rm00 = e[gidx(gc, i - 1, j, k)],
         r00m = e[gidx(gc, i, j, k - 1)], r0mm = e[gidx(gc, i, j - 1, k - 1)],
         rmmm = e[gidx(gc, i - 1, j - 1, k - 1)], rm0m = e[gidx(gc, i - 1, j, k - 1)];
  const int ir = 2 * i - 1, jr = 2 * j - 1, kr = 2 * k - 1;
  T *u = F.u;
  const B *bc = F.bc;
  const T add[8] = {r000,
                    (r000 + r0m0) / T(2),
                    (r000 + r0m0 + rmm0 + rm00) / T(4),
                    (r000 + rm00) / T(2),
                    (r000 + r00m) / T(2),
                    (r000 + r00m + r0mm + r0m0) / T(4),
                    (r000 + r00m + rm0m + rm00) / T(4),
                    (r000 + r00m + rm0m + rm00 + r0m0 + r0mm + rmmm + rmm0) / T(8)};
  const int64_t c0 = gidx(g, ir, jr, kr);
  const int64_t c[8] = {c0, c0 - g.sy, c0 - g.sy - 1, c0 - 1,
                        c0 - g.sz, c0 - g.sz - g.sy, c0 - g.sz - 1, c0 - g.sz - g.sy - 1};
  T old[8];
  int lab[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {   // no read waits for a label
    old[q] = u[c[q]];
    lab[q] = bc[c[q]];
  }
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (lab[q] <= 0) u[c[q]] = old[q] + add[q];
}

template <class T>
__global__ __launch_bounds__(BLOCK) void k_prolong(KLevelT<T> F, KLevelT<T> C, SlotCtl sc,
                                                   MGCtl *fin) {
  if (fin && blockIdx.x == gridDim.x - 1) {   // one more block closes the coarse level's sor_rb
    __shared__ double red[BLOCK / LEPIC_WAVE];
    slots_finish<BLOCK>(sc, fin, red);
    return;
  }
  prolong_node(F, C, blockIdx.x * (int64_t)BLOCK + threadIdx.x);
}

// --------------------------------------------------------------------------
// Coarse levels in one workgroup.  Below a few thousand nodes a level's
// sweep is far shorter than a kernel dispatch, so the part of a V-cycle that
// only touches levels lc..ng-1 (sor_rb down from lc, the coarsest solve and
// sor_rb back up to lc, with the restrictions and prolongations between
// them) runs as one launch: the same per-node routines as the multi-block
// kernels, phases separated by workgroup barriers, the exit rules of sor_rb
// evaluated in the workgroup.
// --------------------------------------------------------------------------
constexpr int CBLOCK = 1024;
// u, b and the labels of every level the workgroup handles live in its LDS
// during the launch (2 x 9056 doubles and 9056 int16 labels, 159 KB): each
// barrier-separated phase then waits on LDS instead of L2.  lc is the first level from which the remaining
// levels fit.
constexpr int64_t COARSE_LDS_NODES = 9056;
constexpr int COARSE_SLOTS = (int)((COARSE_LDS_NODES / 2 + CBLOCK - 1) / CBLOCK);

template <class T>
struct CoarseArgs {
  KLevelT<T> L[MAX_LEVELS];   // u and b point to global memory; the kernel works on LDS copies
  int lc, ng;
  T omega;
  double eps;
  int flag_pbc, flag_nmn;
  int first_cycle;
  int fixed;                  // 1: every sor_rb runs its sweep count, no residual exit
  int nr_fixed, nr_coarsest;  // those counts (fixed = 1)
  T *rp;
  MGCtl *ctl;
  int lds_off[MAX_LEVELS];    // level l's u at lds + lds_off[l], b lds_nn[l] after it
  int lds_nn[MAX_LEVELS];
  int lab_off[MAX_LEVELS];    // level l's labels at labs + lab_off[l]
  // whole solves: pdesolver's normalisation, tolerance and cycle bound, and the
  // cycle and first residual to go on from
  double alpha, tol, res_s;
  int k, ncycl;
};

// V-cycles of a whole solve per launch (the host launches again for more).
constexpr int WHOLE_CYCLES = 64;
// ctl[0].pad after it: the cycle reached, WHOLE_*, the first residual's bits
enum : int { WHOLE_DONE = 0, WHOLE_MORE = 1, WHOLE_DIVERGED = 2 };

// A label as the coarse workgroup keeps it: saturated to int16, which keeps
// its sign and the values 0, -1 and -2, all the solver tests.
__device__ inline int16_t label16(int32_t v) {
  return (int16_t)(v > 32767 ? 32767 : (v < -32768 ? -32768 : v));
}

// Level l as the workgroup sees it: u and b in LDS.  The pointers are formed
// from the workgroup's LDS array itself, never stored and reloaded, so the
// compiler keeps them in the LDS address space (ds_read/ds_write rather than
// flat accesses, which wait on the vector memory counter too).
template <class T>
__device__ inline KLevelT<T, int16_t> lds_level(const CoarseArgs<T> &A, T *lds, int16_t *labs,
                                                int l) {
  const KLevelT<T> &G = A.L[l];
  KLevelT<T, int16_t> v;
  v.g = G.g;
  v.aw = G.aw; v.ae = G.ae; v.an = G.an; v.as = G.as; v.at = G.at; v.ab = G.ab; v.ac = G.ac;
  v.u = lds + A.lds_off[l];
  v.b = lds + A.lds_off[l] + A.lds_nn[l];
  v.bc = labs + A.lab_off[l];
  v.d_h1 = G.d_h1; v.d_n2p1 = G.d_n2p1; v.d_n1p1 = G.d_n1p1;
  v.d_n1p3 = G.d_n1p3; v.d_n1p2 = G.d_n1p2; v.d_h2 = G.d_h2;
  v.acy = G.acy;
  return v;
}

// Workgroup sum in a fixed order, every thread gets it: the waves' sums to
// red[0..15], one barrier, and a row sum of those.  The next call needs a
// barrier in between.
__device__ inline double wg_sum(double a, double *red) {
  static_assert(CBLOCK / LEPIC_WAVE == 16, "a row of wave sums");
  a = wave_sum(a);
  if (__lane_id() == 0) red[threadIdx.x / LEPIC_WAVE] = a;
  __syncthreads();
  return read_lane(row_sum(red[__lane_id() & 15]), 15);
}

// sor_rb (sors.f90:1-535) on level l with periodic walls: at most nr sweeps,
// exit rules as k_decide (with A.fixed, exactly nr sweeps and no residual).
template <class T>
__device__ __forceinline__ void wg_sor_rb(const CoarseArgs<T> &A, T *S, int16_t *Lb, int l, int dig, int64_t nr,
                          double *red) {
  const KLevelT<T, int16_t> Lv = lds_level(A, S, Lb, l);
  const KGrid &g = Lv.g;
  const int64_t nsor = (int64_t)(g.n1 / 2 + 1) * (g.n2 + 1) * (g.n3 + 1);
  const int64_t nres = (int64_t)(g.n1 + 1) * (g.n2 + 1) * (g.n3 + 1);
  const int64_t npy = (int64_t)(g.n1 + 3) * (g.n3 + 3), npz = (int64_t)(g.n1 + 3) * (g.n2 + 3);
  int64_t ksor = 0;
  double res = 0.0, res_s = 0.0;
  for (;;) {
    for (int colour = 0; colour < 2; ++colour) {
      for (int64_t t = threadIdx.x; t < nsor; t += CBLOCK) sor_node(Lv, colour, A.omega, t);
      __syncthreads();
      for (int64_t t = threadIdx.x; t < npy; t += CBLOCK) per_y_node(Lv, t);
      __syncthreads();
      for (int64_t t = threadIdx.x; t < npz; t += CBLOCK) per_z_node(Lv, t);
      __syncthreads();
    }
    ++ksor;
    if (A.fixed) {
      if (ksor >= nr) break;
      continue;
    }
    double a = 0.0;
    for (int64_t t = threadIdx.x; t < nres; t += CBLOCK) a = a + resid_node(Lv, t);
    res = wg_sum(a, red);   // two barriers and more before red is written again
    bool stop;
    if (dig == 0) stop = (res <= A.eps);
    else stop = (res_s > 0.0 && (res / res_s) <= 0.6);
    res_s = res;
    if (stop || ksor >= nr) break;
  }
  if (threadIdx.x == 0 && !A.fixed) {
    MGCtl *c = &A.ctl[l];
    c->active = 0;
    c->ksor = ksor;
    c->res = res;
    c->res_s = res_s;
    c->total += ksor;
  }
}

// One level without periodic walls: sor_rb by the workgroup's first NT
// threads, and on the way down (restricts) the restriction to level l + 1 by
// all of them.  Every sweep of the loops that index, read labels and b and
// sum anew costs 2 us at any size (a chain of LDS reads, 64-bit index
// products, shuffles and five barriers), so here
//  - a thread keeps its nodes' offsets, classes, b and u in registers for the
//    whole sor_rb (SL pairs of a red and a black node; with them b's place in
//    LDS is free to hold the residual that the restriction reads),
//  - the residual of the red nodes shares its reads with the next sweep's
//    relaxation of them, which is taken back if that sweep is not to run: two
//    barriers per sweep, and no residual where the sweep count ends the sor_rb,
//  - a level of at most 64 SL nodes per colour is left to one wave, whose LDS
//    accesses are in order without a barrier.
// want_res: the residual after the last sweep is returned, to every thread.
// Up to 3 pairs per thread have their own copy of the routine: five spill in FP64
// (16^3: 240 us a solve instead of 281).  With its spills the copy of five is
// still the faster form past 3072 pairs (coarsest levels of 3213 and 3519: 24
// V-cycles of 32 x 32 x 40 4.6 -> 3.5 ms, 26 of 32 x 32 x 44 7.5 -> 3.8).
// Launch of 16^3 and below, FP64: 98 -> 62 us; 8^3 and below 47 -> 32.
template <class T, int NT, int SL>
__device__ __forceinline__ double wg_level(const CoarseArgs<T> &A, T *S, int16_t *Lb, int l,
                                           int dig, int64_t nr, bool restricts, bool want_res,
                                           double *red) {
  const KLevelT<T, int16_t> Lv = lds_level(A, S, Lb, l);
  const KGrid &g = Lv.g;
  const int tid = (int)threadIdx.x;
  const bool works = NT == CBLOCK || tid < NT;
  const int sy = (int)g.sy, sz = (int)g.sz;
  const int ni2 = g.n1 / 2 + 1;
  const int nsor = ni2 * (g.n2 + 1) * (g.n3 + 1);
  T *u = Lv.u, *bl = Lv.b;
  const T omega = A.omega;
  // per node: LDS offset << 5 | a node (not a filled-up slot) << 4 | first plane
  // of a Neumann level << 3 | residual wanted by the restriction << 2 | class
  // (0 not relaxed, 1 plasma, 2 Neumann, 3 other)
  int pk[2][SL];
  T bb[2][SL], uc[2][SL];
  double res = 0.0;
  auto sync = [&]() {
    if (NT == CBLOCK) {
      __syncthreads();
    } else {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  };
  if (works) {
#pragma unroll
    for (int s = 0; s < SL; ++s) {
      pk[0][s] = pk[1][s] = 0;
      const int t = tid + s * NT;
      if (t < nsor) {
        const uint32_t r = mdiv_q((uint32_t)t, Lv.d_h1), rk = mdiv_q(r, Lv.d_n2p1);
        const int i2 = t - (int)r * ni2, j = 1 + (int)(r - rk * (uint32_t)(g.n2 + 1)),
                  k = 1 + (int)rk;
        const int is = 1 + ((j + k) & 1);   // red: i + j + k odd
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const int i = (c ? 3 - is : is) + 2 * i2;
          if (i <= g.n1 + 1) {
            const int at = i + sy * j + sz * k, lab = Lv.bc[at];
            const int cls = lab > 0 || (lab == 0 && (k == g.n3 + 1 || j == g.n2 + 1)) ? 0
                      : (lab == -1 ? 1 : (lab == -2 ? 2 : 3));
            pk[c][s] = at << 5 | 16 | (i == 1 && A.flag_nmn == 1 ? 8 : 0) |
                       (lab <= 0 || j == g.n2 ? 4 : 0) | cls;
          }
        }
      }
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        bb[c][s] = bl[pk[c][s] >> 5];
        uc[c][s] = u[pk[c][s] >> 5];
      }
    }
    auto relax = [&](int cls, T c, T uw, T ue, T un, T us, T ut, T ub, T b) {
      if (cls == 2)
        return (T(1) - omega) * c +
               div_ac(omega * (b - Lv.an * un - Lv.as * us - T(2) * Lv.ae * ue - Lv.at * ut -
                               Lv.ab * ub),
                      Lv);
      return (T(1) - omega) * c +
             div_ac(omega * (b - Lv.aw * uw - Lv.an * un - Lv.as * us - Lv.ae * ue - Lv.at * ut -
                             Lv.ab * ub),
                    Lv);
    };
    double a = 0.0;
    // one colour: its L1 residual before (pre) or after (post) the relaxation
    auto phase = [&](auto colour, bool relaxes, bool pre, bool post, T *old) {
      constexpr int c = decltype(colour)::value;
#pragma unroll
      for (int s = 0; s < SL; ++s) {
        const int cls = pk[c][s] & 3;
        if (s * NT < nsor && cls) {
          int at = pk[c][s] >> 5;
          asm("" : "+v"(at));   // the neighbours' addresses formed here, not kept over the sweeps
          const T uw = u[at - 1], ue = u[at + 1], un = u[at + sy], us = u[at - sy],
                  ut = u[at + sz], ub = u[at - sz];
          auto resid = [&]() {
            const T rij = bb[c][s] - (Lv.aw * uw + Lv.an * un + Lv.as * us + Lv.ae * ue +
                                      Lv.ac * uc[c][s] + Lv.at * ut + Lv.ab * ub);
            a = a + fabs((double)rij);
          };
          if (pre && cls == 1) resid();
          if (relaxes) {
            if (old) old[s] = uc[c][s];
            uc[c][s] = relax(cls, uc[c][s], uw, ue, un, us, ut, ub, bb[c][s]);
            u[at] = uc[c][s];
          }
          if (post && cls == 1) resid();
        }
      }
    };
    const std::integral_constant<int, 0> RED{};
    const std::integral_constant<int, 1> BLACK{};
    int64_t ksor = 0;
    double res_s = 0.0;
    phase(RED, true, false, false, nullptr);
    sync();
    for (;;) {
      ++ksor;
      const bool last = ksor >= nr, judged = !A.fixed && (!last || want_res);
      a = 0.0;
      phase(BLACK, true, false, judged, nullptr);
      sync();
      if (last && !judged) break;
      T old[SL];
      phase(RED, !last, judged, false, old);
      if (judged) {
        if (NT == CBLOCK) {
          res = wg_sum(a, red);
        } else {
          res = wave_sum(a);
          sync();
        }
        if (last) break;
        const bool stop = dig == 0 ? res <= A.eps : res_s > 0.0 && (res / res_s) <= 0.6;
        res_s = res;
        if (stop) {   // the next sweep's red half is not to be
#pragma unroll
          for (int s = 0; s < SL; ++s)
            if (s * NT < nsor && (pk[0][s] & 3)) {
              uc[0][s] = old[s];
              u[pk[0][s] >> 5] = old[s];
            }
          sync();
          break;
        }
      } else {
        sync();
      }
    }
    if (tid == 0 && !A.fixed) A.ctl[l].total += ksor;
    if (restricts) {
      // getres (mg.f90:809-848) of every node, 0 on electrodes, in b's place
      // (the plane j = n2 keeps its electrodes' too: see restrict_node)
#pragma unroll
      for (int s = 0; s < SL; ++s)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const int at = pk[c][s] >> 5;
          if (pk[c][s] & 4) {
            const bool first = pk[c][s] & 8;
            const T aw = first ? T(0) : Lv.aw, ae = first ? T(2) * Lv.ae : Lv.ae,
                    uw = first ? T(0) : u[at - 1];
            bl[at] = bb[c][s] - (aw * uw + ae * u[at + 1] + Lv.an * u[at + sy] + Lv.as * u[at - sy] +
                                 Lv.ac * uc[c][s] + Lv.at * u[at + sz] + Lv.ab * u[at - sz]);
          } else if (pk[c][s] & 16) {
            bl[at] = T(0);
          }
        }
    }
  }
  __syncthreads();
  if (want_res && NT != CBLOCK) {
    if (tid == 0) red[0] = res;
    __syncthreads();
    res = red[0];
    __syncthreads();
  }
  if (!restricts) return res;
  const KLevelT<T, int16_t> Cv = lds_level(A, S, Lb, l + 1);
  const int nt = ni2 * (g.n2 / 2 + 1) * (g.n3 / 2 + 1);
  for (int t = tid; t < nt; t += CBLOCK)
    restrict_node(Lv, Cv, (const T *)nullptr, A.flag_nmn, t, (const T *)bl, true);
  __syncthreads();
  if (works) {
#pragma unroll
    for (int s = 0; s < SL; ++s)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        if (pk[c][s] & 16) bl[pk[c][s] >> 5] = bb[c][s];
  }
  // the up leg's reads of b lie behind further barriers
  return res;
}

template <class T>
__device__ __forceinline__ void wg_restriction(const CoarseArgs<T> &A, T *S, int16_t *Lb, int l) {
  const KLevelT<T, int16_t> F = lds_level(A, S, Lb, l);
  const KLevelT<T, int16_t> C = lds_level(A, S, Lb, l + 1);
  const KGrid &g = F.g;
  const int64_t nent = ((int64_t)g.n1 + 2) * ((int64_t)g.n2 + 2);
  for (int64_t t = threadIdx.x; t < nent; t += CBLOCK) rpbc_entry(F, A.rp, A.flag_nmn, t);
  __syncthreads();
  const int64_t nt = (int64_t)(g.n1 / 2 + 1) * (g.n2 / 2 + 1) * (g.n3 / 2 + 1);
  for (int64_t t = threadIdx.x; t < nt; t += CBLOCK) restrict_node(F, C, (const T *)A.rp, A.flag_nmn, t);
  __syncthreads();
}

template <class T>
__device__ __forceinline__ void wg_prolongation(const CoarseArgs<T> &A, T *S, int16_t *Lb, int l) {  // L[l] += P(L[l+1])
  const KLevelT<T, int16_t> F = lds_level(A, S, Lb, l);
  const KLevelT<T, int16_t> C = lds_level(A, S, Lb, l + 1);
  const KGrid &g = F.g;
  const int64_t nt = (int64_t)(g.n1 / 2 + 1) * (g.n2 / 2 + 1) * (g.n3 / 2 + 1);
  for (int64_t t = threadIdx.x; t < nt; t += CBLOCK) prolong_node(F, C, t);
  __syncthreads();
}

// The V-cycle of mg (mg.f90:1-246) restricted to levels lc..ng-1; the
// prolongation into level lc-1 is left to the caller.
// The host sizes lc so that levels lc..ng-1 hold at most COARSE_LDS_NODES
// nodes together.  Level lc's b and labels are copied in at the start; u is 0
// on every level then, and b 0 at the ghost nodes, which no restriction
// writes.  u of level lc, the only array read after the launch, is copied back
// at the end.
// WHOLE: lc = 0, and the launch is pdesolver's loop (pdesolver.f90:97-115) of
// up to WHOLE_CYCLES V-cycles.  A V-cycle of 16^3 takes 16 launches and a host
// round trip else, 108 us; here 55 (solve 434 -> 240 us).
template <class T, bool PBC, bool WHOLE>
__global__ __launch_bounds__(CBLOCK) void k_mg_coarse(CoarseArgs<T> A) {
  __shared__ double red[CBLOCK / LEPIC_WAVE];
  __shared__ T lds[2 * COARSE_LDS_NODES];
  __shared__ int16_t labs[COARSE_LDS_NODES];
  T *const S = lds;
  int16_t *const Lb = labs;
  const int ng = A.ng;
  {
    constexpr int RL = (int)((COARSE_LDS_NODES + CBLOCK - 1) / CBLOCK);
    const KLevelT<T> &G = A.L[A.lc];
    const KGrid &g = G.g;
    const int nn = A.lds_nn[A.lc], nx = g.n1 + 1, nb = nx * (g.n2 + 1) * (g.n3 + 1);
    int at[RL];
    T bv[RL], uv[RL];
    int32_t lv[RL];
#pragma unroll
    for (int r = 0; r < RL; ++r) {   // every read before the first wait
      const int t = (int)threadIdx.x + r * CBLOCK;
      lv[r] = t < nn ? G.bc[t] : 0;
      uv[r] = WHOLE && t < nn ? G.u[t] : T(0);
      const uint32_t row = mdiv_q((uint32_t)t, G.d_n1p1), rk = mdiv_q(row, G.d_n2p1);
      at[r] = t < nb ? (int)gidx(g, 1 + t - (int)row * nx, 1 + (int)(row - rk * (g.n2 + 1)),
                                 1 + (int)rk)
                     : -1;
      bv[r] = at[r] >= 0 ? G.b[at[r]] : T(0);
    }
    const int all = A.lds_off[ng - 1] + 2 * A.lds_nn[ng - 1];
    for (int t = threadIdx.x; t < all; t += CBLOCK) lds[t] = T(0);
    for (int t = threadIdx.x; t < all / 2; t += CBLOCK) labs[t] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RL; ++r) {
      const int t = (int)threadIdx.x + r * CBLOCK;
      if (t < nn) labs[t] = label16(lv[r]);
      if (WHOLE && t < nn) lds[t] = uv[r];
      if (at[r] >= 0) lds[nn + at[r]] = bv[r];
    }
  }
  __syncthreads();
  const int64_t nr = A.fixed ? A.nr_fixed : 4;
  const int m = ng - 1 - A.lc;
  int cycle = WHOLE ? A.k : (A.first_cycle ? 1 : 2), state = WHOLE_DONE;
  double fine = 0.0, first = A.res_s;
  for (int done = 0;;) {
    // down from lc, the coarsest level, back up (one place that calls each
    // routine: inlined, the arguments stay in scalar memory)
    for (int v = 0; v <= 2 * m; ++v) {
      const int l = v <= m ? A.lc + v : A.lc + 2 * m - v;
      const int dig = v == m ? 0 : (v < m ? l + 1 - ng : ng - 1 - l);
      const int64_t count =
          v == m ? (A.fixed ? A.nr_coarsest : (cycle == 1 ? 1000000 : 4)) : nr;
      if (v > m) wg_prolongation(A, S, Lb, l);
      if (PBC) {
        wg_sor_rb(A, S, Lb, l, dig, count, red);
        __syncthreads();
        if (v < m) wg_restriction(A, S, Lb, l);
      } else {
        const KGrid &g = A.L[l].g;
        const bool last = WHOLE && v == 2 * m;
        const int nsor = (g.n1 / 2 + 1) * (g.n2 + 1) * (g.n3 + 1);
        if (nsor <= 2 * LEPIC_WAVE)
          fine = wg_level<T, LEPIC_WAVE, 2>(A, S, Lb, l, dig, count, v < m, last, red);
        else if (nsor <= 3 * CBLOCK)
          fine = wg_level<T, CBLOCK, 3>(A, S, Lb, l, dig, count, v < m, last, red);
        else
          fine = wg_level<T, CBLOCK, COARSE_SLOTS>(A, S, Lb, l, dig, count, v < m, last, red);
      }
    }
    if (!WHOLE) break;
    const double res = fine / A.alpha;
    if (cycle == 1) {
      first = res;
    } else if (fabs(res / first) > 10.0) {
      state = WHOLE_DIVERGED;
      break;
    }
    if (res < A.tol || cycle == A.ncycl) break;
    ++cycle;
    if (++done == WHOLE_CYCLES) {
      state = WHOLE_MORE;
      break;
    }
    for (int c = 1; c < ng; ++c)   // the corrections start from 0 again
      for (int t = threadIdx.x; t < A.lds_nn[c]; t += CBLOCK) lds[A.lds_off[c] + t] = T(0);
    __syncthreads();
  }
  if (WHOLE && threadIdx.x == 0) {
    A.ctl[0].res = fine;
    A.ctl[0].pad[0] = cycle;
    A.ctl[0].pad[1] = state;
    A.ctl[0].pad[2] = __double_as_longlong(first);
  }
  __syncthreads();
  {
    const KGrid &g = A.L[A.lc].g;
    const int64_t nn = ((int64_t)g.n1 + 3) * ((int64_t)g.n2 + 3) * ((int64_t)g.n3 + 3);
    for (int64_t t = threadIdx.x; t < nn; t += CBLOCK) A.L[A.lc].u[t] = lds[A.lds_off[A.lc] + t];
  }
}

template <class T>
__global__ void k_fill_d(T *a, int64_t n, T v) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) a[i] = v;
}

// Tiles of the whole-sweep launches (k_sweep): the large one fills a CU's LDS
// (155 KB in FP64) and relaxes the fewest halo nodes, the small one spreads a
// level that would leave CUs idle.  Per sweep: 22 us against 10 at 64^3 (32
// and 256 blocks), 28 against 42 at 128^3 (256 and 1800), 239 against 263 at
// 256^3; a launch of one large block per CU takes 28 us whatever its count, so
// the line is where the small tiles need as long, near 112^3 (196 blocks).
constexpr int BIG_X = 33, BIG_Y = 17, BIG_Z = 17, BIG_NT = 1024;
constexpr int SML_X = 17, SML_Y = 9, SML_Z = 9, SML_NT = 768;

struct SweepGrid {
  int nx, ny, nz;
  bool big;
  unsigned blocks() const { return (unsigned)nx * (unsigned)ny * (unsigned)nz; }
};

inline SweepGrid sweep_grid(const KGrid &g) {
  auto tiles = [](int n, int t) { return (n + 1 + t - 1) / t; };
  SweepGrid w{tiles(g.n1, BIG_X), tiles(g.n2, BIG_Y), tiles(g.n3, BIG_Z), true};
  if ((int64_t)w.nx * w.ny * w.nz < 192)
    w = SweepGrid{tiles(g.n1, SML_X), tiles(g.n2, SML_Y), tiles(g.n3, SML_Z), false};
  return w;
}

// Blocks of a restriction whose tiles are x x y x z coarse nodes.
struct RestrictGrid {
  int nx, ny, nz;
  RestrictGrid(const KGrid &g, int x, int y, int z)
      : nx((g.n1 / 2 + x) / x), ny((g.n2 / 2 + y) / y), nz((g.n3 / 2 + z) / z) {}
  unsigned blocks() const { return (unsigned)nx * (unsigned)ny * (unsigned)nz; }
};

// Whether a level sweeps in whole-sweep launches.  A flat or narrow grid leaves
// most of a large tile empty, which costs as much as a full one: unless the grid
// fills 0.42 of them (0.27 up to two tiles per CU), one launch per colour is as
// fast or faster.  Solves with tiles / per colour (FP64, and CG with the FP64
// preconditioner, ms): 8 x 1024 x 1024 (0.26 filled) 17.8 / 11.7 and 10.0 / 7.9, 12 x
// 1024 x 1024 (0.39) 18.8 / 15.3 and 11.5 / 10.3, 12 x 512 x 512 (0.37) 5.2 / 5.6 and
// 3.5 / 3.4, 16 x 512 x 512 (0.49) 5.7 / 6.8 and 3.6 / 4.0, 512 x 512 x 4 (0.28, 496
// tiles) 1.6 / 2.0 and 1.2 / 1.3.  The small tiles' levels are launch-bound: always.
inline bool sweeps_tiled(const KGrid &g) {
  const SweepGrid w = sweep_grid(g);
  const double filled = (double)(g.n1 + 1) * (g.n2 + 1) * (g.n3 + 1) /
                        ((double)w.blocks() * (BIG_X * BIG_Y * BIG_Z));
  return !w.big || filled >= (w.blocks() <= 512 ? 0.27 : 0.42);
}

template <class T>
struct Solver {
  lepic_ctx *ctx;
  KLevelT<T> L[MAX_LEVELS];
  int ng;
  T omega;
  int flag_pbc, flag_nmn;
  double *partials;
  T *rp;
  MGCtl *ctl;  // device, MAX_LEVELS entries
  int lc;      // first level handled by k_mg_coarse (ng: none)
  // fixed sweep counts (the inner smoother of the mixed-precision solve):
  // nr_fixed per sor_rb, nr_coarsest on the coarsest level, no residuals
  int fixed = 0, nr_fixed = 2, nr_coarsest = 64;
  // the fine residual of a periodic restriction (the finest level's ghosted size)
  T *resbuf = nullptr;
  // the second u array of the levels that sweep in one or two launches
  // (nullptr: one launch per colour), and the sweeps' exit bookkeeping
  T *u2[MAX_LEVELS] = {};
  SlotState *slot_state = nullptr;
  double *slot_partials = nullptr;   // 3 x the most blocks of a sweep launch
  MGCtl *fin = nullptr;              // the level whose last sor_rb is still to be closed
  SlotCtl fin_sc = {};

  CoarseArgs<T> coarse_args(double eps, int kmg) {
    CoarseArgs<T> A = {};
    for (int l = 0; l < MAX_LEVELS; ++l) A.L[l] = L[l];
    A.lc = lc;
    A.ng = ng;
    A.omega = omega;
    A.eps = eps;
    A.flag_pbc = flag_pbc;
    A.flag_nmn = flag_nmn;
    A.first_cycle = kmg == 1 ? 1 : 0;
    A.fixed = fixed;
    A.nr_fixed = nr_fixed;
    A.nr_coarsest = nr_coarsest;
    A.rp = rp;
    A.ctl = ctl;
    int off = 0;
    for (int l = 0; l < MAX_LEVELS; ++l) {
      A.lds_off[l] = 0;
      A.lds_nn[l] = 0;
      A.lab_off[l] = 0;
      if (l < lc || l >= ng) continue;
      A.lds_off[l] = off;
      A.lds_nn[l] = (int)grid_nodes_k(L[l].g);
      A.lab_off[l] = off / 2;
      off += 2 * A.lds_nn[l];
    }
    return A;
  }

  void coarse(double eps, int kmg) {
    const CoarseArgs<T> A = coarse_args(eps, kmg);
    if (flag_pbc)
      hipLaunchKernelGGL((k_mg_coarse<T, true, false>), dim3(1), dim3(CBLOCK), 0, ctx->stream, A);
    else
      hipLaunchKernelGGL((k_mg_coarse<T, false, false>), dim3(1), dim3(CBLOCK), 0, ctx->stream, A);
  }

  // The launch of a whole solve from V-cycle k on (all levels in the workgroup).
  void whole(double eps, int k, int ncycl, double alpha, double tol, double res_s) {
    CoarseArgs<T> A = coarse_args(eps, k);
    A.alpha = alpha;
    A.tol = tol;
    A.res_s = res_s;
    A.k = k;
    A.ncycl = ncycl;
    hipLaunchKernelGGL((k_mg_coarse<T, false, true>), dim3(1), dim3(CBLOCK), 0, ctx->stream, A);
  }

  // One sweep; first: the sor_rb's first, whose red half arms ctl[l].
  void sor_sweep(int l, double eps, int dig, int64_t nr, bool first) {
    KLevelT<T> &Lv = L[l];
    const KGrid &g = Lv.g;
    int64_t nsor = (int64_t)(g.n1 / 2 + 1) * (g.n2 + 1) * (g.n3 + 1);
    int64_t nres = (int64_t)(g.n1 + 1) * (g.n2 + 1) * (g.n3 + 1);
    unsigned bs = grid_blocks(nsor, BLOCK);
    const unsigned br = std::min<unsigned>(grid_blocks(nres, BLOCK), RESID_BLOCKS);
    hipStream_t s = ctx->stream;
    const MGCtl *c = fixed ? nullptr : &ctl[l];   // fixed counts: no exit, no control block
    for (int colour = 0; colour < 2; ++colour) {
      MGCtl *begin = (first && colour == 0 && !fixed) ? &ctl[l] : nullptr;
      hipLaunchKernelGGL(k_sor<T>, dim3(bs), dim3(BLOCK), 0, s, Lv, colour, omega, c, begin);
      if (flag_pbc) {
        hipLaunchKernelGGL(k_per_y<T>, dim3(grid_blocks((int64_t)(g.n1 + 3) * (g.n3 + 3), BLOCK)),
                           dim3(BLOCK), 0, s, Lv, c);
        hipLaunchKernelGGL(k_per_z<T>, dim3(grid_blocks((int64_t)(g.n1 + 3) * (g.n2 + 3), BLOCK)),
                           dim3(BLOCK), 0, s, Lv, c);
      }
    }
    if (fixed) return;   // a fixed sweep count: no residual, the level stays active
    hipLaunchKernelGGL(k_resid<T>, dim3(br), dim3(BLOCK), 0, s, Lv, partials, &ctl[l], nres);
    hipLaunchKernelGGL(k_decide, dim3(1), dim3(BLOCK), 0, s, partials, (int64_t)br, &ctl[l], eps,
                       dig, nr);
  }

  // A level with a second u array sweeps in whole-sweep launches, with periodic
  // walls in two per sweep; the others and the coarsest level's sor_rb (another
  // exit rule, up to 10^6 sweeps) in one launch per colour.
  bool tiled(int l, int dig) const { return !flag_pbc && dig != 0 && u2[l]; }
  bool periodic(int l, int dig) const { return flag_pbc && dig != 0 && u2[l]; }

  void sor_periodic(int l) {
    const KLevelT<T> &Lv = L[l];
    const KGrid &g = Lv.g;
    const int64_t n = (int64_t)(g.n1 / 2 + 1) * (g.n2 + 1) * (g.n3 + 1);
    const unsigned nb = std::min<unsigned>(grid_blocks(n, BLOCK), PER_BLOCKS);
    const SlotCtl sc{slot_state, slot_partials, (int64_t)nb};
    MGCtl *c = fixed ? nullptr : &ctl[l];
    const int sweeps = fixed ? nr_fixed : SLOTS;
    T *X[2] = {Lv.u, u2[l]};
    for (int s = 0; s < sweeps; ++s) {
      hipLaunchKernelGGL(k_per_half<T>, dim3(nb), dim3(BLOCK), 0, ctx->stream, Lv,
                         (const T *)X[s & 1], X[1 - (s & 1)], 0, omega, s, sc, c);
      hipLaunchKernelGGL(k_per_half<T>, dim3(nb), dim3(BLOCK), 0, ctx->stream, Lv,
                         (const T *)X[1 - (s & 1)], (T *)nullptr, 1, omega, s, sc, c);
    }
    const int resid = l == 0 && !fixed ? 1 : 0;   // the level whose residual is read
    hipLaunchKernelGGL(k_per_end<T>, dim3(nb), dim3(BLOCK), 0, ctx->stream, Lv,
                       mdiv((uint32_t)(g.n2 + 3)), (const T *)u2[l], sweeps, resid, sc, c);
    if (resid) hipLaunchKernelGGL(k_per_res, dim3(1), dim3(BLOCK), 0, ctx->stream, sc, c);
  }

  void sor_slots(int l, bool zero) {
    const KLevelT<T> &Lv = L[l];
    const SweepGrid w = sweep_grid(Lv.g);
    SlotCtl sc{slot_state, slot_partials, (int64_t)w.blocks()};
    for (int s = 0; s < SLOTS; ++s) {
      const T *src = (s & 1) ? u2[l] : Lv.u;
      T *dst = (s & 1) ? Lv.u : u2[l];
      if (w.big)
        hipLaunchKernelGGL((k_sweep<T, BIG_X, BIG_Y, BIG_Z, BIG_NT, 2, 1, true>), dim3(w.blocks()),
                           dim3(BIG_NT), 0, ctx->stream, Lv, src, dst, omega, w.nx, w.ny,
                           zero && s == 0 ? 1 : 0, s, sc, &ctl[l]);
      else
        hipLaunchKernelGGL((k_sweep<T, SML_X, SML_Y, SML_Z, SML_NT, 4, 1, true>), dim3(w.blocks()),
                           dim3(SML_NT), 0, ctx->stream, Lv, src, dst, omega, w.nx, w.ny,
                           zero && s == 0 ? 1 : 0, s, sc, &ctl[l]);
    }
    fin = &ctl[l];
    fin_sc = sc;
  }

  // nr_fixed sweeps of a level whose u is L[l].u on entry and on return: each
  // launch writes the other array, which then takes its place (both legs of a
  // V-cycle issue the same launches, so u is at home again after the second).
  // zero: u is 0 everywhere and is not read.
  void sor_fixed(int l, bool zero) {
    const SweepGrid w = sweep_grid(L[l].g);
    const SlotCtl none = {};
    auto launch = [&](auto kernel, int tx, int ty, int tz, int nt) {
      const KGrid &g = L[l].g;
      const int nx = (g.n1 + tx) / tx, ny = (g.n2 + ty) / ty, nz = (g.n3 + tz) / tz;
      hipLaunchKernelGGL(kernel, dim3((unsigned)nx * ny * nz), dim3(nt), 0, ctx->stream, L[l],
                         (const T *)L[l].u, u2[l], omega, nx, ny, zero ? 1 : 0, 0, none,
                         (MGCtl *)nullptr);
      std::swap(L[l].u, u2[l]);
      zero = false;
    };
    // Two sweeps a launch on the small tile (launch-bound levels: 7 us against
    // 2 x 5 at 64^3); large levels are read-bound and take one, on the tile
    // whose blocks leave room for others on the CU.  FP32 256^3 conjugate
    // gradients: 33 x 9 x 9 8.9 ms, 33 x 15 x 17 with two sweeps 9.7, 33 x 9 x 9
    // with two 9.3, 17 x 9 x 9 10.4, one launch per colour 10.9.  FP64 128^3
    // preconditioner: 33 x 17 x 17 1.27 ms, 33 x 9 x 9 1.31, per colour 1.49.
    constexpr int LY = sizeof(T) == 4 ? 9 : BIG_Y, LZ = sizeof(T) == 4 ? 9 : BIG_Z,
                  LNT = sizeof(T) == 4 ? 512 : BIG_NT;
    for (int c = 0; c < nr_fixed;) {
      if (w.big) {
        launch(k_sweep<T, BIG_X, LY, LZ, LNT, 2, 1, false>, BIG_X, LY, LZ, LNT);
        c += 1;
      } else if (c + 2 <= nr_fixed) {
        launch(k_sweep<T, SML_X, SML_Y, SML_Z, 896, 4, 2, false>, SML_X, SML_Y, SML_Z, 896);
        c += 2;
      } else {
        launch(k_sweep<T, SML_X, SML_Y, SML_Z, SML_NT, 4, 1, false>, SML_X, SML_Y, SML_Z, SML_NT);
        c += 1;
      }
    }
  }

  // sor_rb: returns LEPIC_OK; sweeps are counted on the device.  zero: the
  // level's u is 0 everywhere.
  int sor_rb(int l, double eps, int kmg, int dig, bool zero = false) {
    if (periodic(l, dig)) {
      sor_periodic(l);
      return LEPIC_OK;
    }
    if (tiled(l, dig)) {
      if (fixed) sor_fixed(l, zero);
      else sor_slots(l, zero);
      return LEPIC_OK;
    }
    if (fixed) {
      for (int c = 0; c < (dig == 0 ? nr_coarsest : nr_fixed); ++c) sor_sweep(l, eps, dig, 4, false);
      return LEPIC_OK;
    }
    if (kmg == 1 && dig == 0) {
      // first V-cycle's coarsest level: up to 1e6 sweeps to res <= eps.
      const int64_t nr = 1000000;
      int64_t done = 0;
      while (done < nr) {
        int chunk = 32;
        for (int c = 0; c < chunk; ++c) sor_sweep(l, eps, dig, nr, done == 0 && c == 0);
        done += chunk;
        LEPIC_HIP(ctx, hipMemcpyAsync(ctx->h_pinned, &ctl[l], sizeof(MGCtl), hipMemcpyDeviceToHost,
                                      ctx->stream));
        LEPIC_HIP(ctx, hipStreamSynchronize(ctx->stream));
        if (ctx->h_pinned[0] == 0) break;
      }
    } else {
      for (int c = 0; c < 4; ++c) sor_sweep(l, eps, dig, 4, c == 0);
    }
    return LEPIC_OK;
  }

  void restriction(int l) {
    KLevelT<T> &F = L[l];
    KLevelT<T> &C = L[l + 1];
    const KGrid &g = F.g;
    const int64_t nc = grid_nodes_k(C.g);
    if (!flag_pbc) {
      // whole sweeps and the one-workgroup levels start from 0 without reading u
      if (l + 1 < lc && !(l + 1 < ng - 1 && u2[l + 1]))
        hipLaunchKernelGGL(k_fill_d<T>, dim3(grid_blocks(nc, BLOCK)), dim3(BLOCK), 0, ctx->stream,
                           C.u, nc, T(0));
      // 42 us against 22 at 8 x 32768 x 8 (FP64), where the first fills a fifth of its tiles
      auto launch = [&](auto kernel, const RestrictGrid &r) {
        hipLaunchKernelGGL(kernel, dim3(r.blocks() + (fin ? 1 : 0)), dim3(BLOCK), 0, ctx->stream, F,
                           C, flag_nmn, r.nx, r.ny, fin_sc, fin);
      };
      const RestrictGrid wide(g, 16, 4, 4), narrow(g, 4, 8, 8);
      if (2 * (int64_t)wide.blocks() < 3 * (int64_t)narrow.blocks())
        launch(k_restrict_tile<T, 16, 4, 4>, wide);
      else
        launch(k_restrict_tile<T, 4, 8, 8>, narrow);
      fin = nullptr;
      return;
    }
    const int64_t nres = (int64_t)(g.n1 + 1) * (g.n2 + 1) * (g.n3 + 1);
    hipLaunchKernelGGL(k_getres<T>, dim3(grid_blocks(std::max(nc, nres), BLOCK)), dim3(BLOCK), 0,
                       ctx->stream, F, resbuf, C.u, nc, flag_nmn);
    const int64_t nent = (int64_t)(g.n1 + 2) * (g.n2 + 2);
    hipLaunchKernelGGL(k_rpbc<T>, dim3(grid_blocks(nent, BLOCK)), dim3(BLOCK), 0, ctx->stream, F,
                       rp, flag_nmn);
    const int64_t nt = (int64_t)(g.n1 / 2 + 1) * (g.n2 / 2 + 1) * (g.n3 / 2 + 1);
    hipLaunchKernelGGL(k_restrict<T>, dim3(grid_blocks(nt, BLOCK)), dim3(BLOCK), 0, ctx->stream, F,
                       C, (const T *)rp, flag_nmn, (const T *)resbuf);
  }

  void prolongation(int l) {  // L[l] += P(L[l+1])
    const KGrid &g = L[l].g;
    int64_t nt = (int64_t)(g.n1 / 2 + 1) * (g.n2 / 2 + 1) * (g.n3 / 2 + 1);
    hipLaunchKernelGGL(k_prolong<T>, dim3(grid_blocks(nt, BLOCK) + (fin ? 1 : 0)), dim3(BLOCK), 0, ctx->stream,
                       L[l], L[l + 1], fin_sc, fin);
    fin = nullptr;
  }

  // The levels with a second u array, its nodes in all, and its places from at on.
  bool has_u2(int l) const { return ng > 1 && (flag_pbc || sweeps_tiled(L[l].g)); }
  int64_t u2_nodes() const {
    int64_t n = 0;
    for (int l = 0; l < ng; ++l) n += has_u2(l) ? grid_nodes_k(L[l].g) : 0;
    return n;
  }
  void place_u2(T *at) {
    for (int l = 0; l < ng; ++l) {
      u2[l] = has_u2(l) ? at : nullptr;
      at += has_u2(l) ? grid_nodes_k(L[l].g) : 0;
    }
  }

  static int64_t grid_nodes_k(const KGrid &g) {
    return ((int64_t)g.n1 + 3) * ((int64_t)g.n2 + 3) * ((int64_t)g.n3 + 3);
  }

  // One V-cycle of mg (mg.f90:99-239).  Levels lc..ng-1 run inside
  // k_mg_coarse: the stretch from the down-leg sor_rb on lc to the up-leg
  // sor_rb on lc touches no level above lc and is issued as one launch.
  int vcycle(int kmg, double epsa, bool zero = false) {
    for (int ig = 1; ig <= 2 * ng - 1; ++ig) {
      for (int il = 1; il <= ng - 1 && il <= 11; ++il) {
        const int l = il - 1;
        if (ig < ng && ig == il) {
          if (l < lc) {
            int st = sor_rb(l, epsa, kmg, ig - ng, l > 0 || zero);
            if (st) return st;
            restriction(l);
          } else if (l == lc) {
            coarse(epsa, kmg);
          }
        }
        if (ig > ng && ig == 2 * ng - il) {
          if (l < lc) {
            int st = sor_rb(l, epsa, kmg, ig - ng);
            if (st) return st;
          }
          if (l <= lc && il >= 2) prolongation(il - 2);
        }
      }
      if (ig == ng) {
        if (lc >= ng) {
          int st = sor_rb(ng - 1, epsa, kmg, 0);
          if (st) return st;
        } else if (lc == ng - 1) {
          coarse(epsa, kmg);
        }
        if (ng >= 2 && ng - 2 < lc) prolongation(ng - 2);
      }
    }
    if (fin) {
      hipLaunchKernelGGL(k_slots_finish, dim3(1), dim3(BLOCK), 0, ctx->stream, fin_sc, fin);
      fin = nullptr;
    }
    return LEPIC_OK;
  }

  // lc: the first level from which the remaining levels fit the coarse
  // workgroup's LDS (ng: none do), from the given one on.
  void choose_lc(int from = 1) {
    lc = ng;
    for (int l = from; l < ng; ++l) {
      int64_t tot = 0;
      for (int m = l; m < ng; ++m) tot += grid_nodes_k(L[m].g);
      if (tot <= COARSE_LDS_NODES) {
        lc = l;
        break;
      }
    }
  }
};

// mg.h:9-15, formed in FP64 (and rounded once for an FP32 level).
template <class T>
void set_coeffs(KLevelT<T> &L, double eps0) {
  const KGrid &g = L.g;
  const double aw = eps0 / (g.h1 * g.h1);
  const double ae = aw;
  const double an = eps0 / (g.h2 * g.h2);
  const double as = an;
  const double at = eps0 / (g.h3 * g.h3);
  const double ab = at;
  const double ac = -(an + as + aw + ae + at + ab);
  L.aw = (T)aw; L.ae = (T)ae; L.an = (T)an; L.as = (T)as; L.at = (T)at; L.ab = (T)ab;
  L.ac = (T)ac;
  L.acy = qdiv_divisor_ok(ac) ? 1.0 / ac : 0.0;
}

}  // namespace

extern "C" int lepic_poisson_solve(lepic_ctx *ctx, const lepic_grid *g, double *phi,
                                   const double *rho, const int32_t *bcnd,
                                   const lepic_mg_params *mp, lepic_mg_stats *stats) {
  if (!ctx) return LEPIC_ERR_ARG;
  if (!g || !phi || !rho || !bcnd || !mp) return lepic_fail(ctx, LEPIC_ERR_ARG, "poisson: null argument");
  const int ng = mp->ng;
  if (ng < 1 || ng > MAX_LEVELS) return lepic_fail(ctx, LEPIC_ERR_ARG, "poisson: ng outside [1,12]");
  if (grid_nodes(g) > INT32_MAX)   // thread numbers are decoded in 32 bits
    return lepic_fail(ctx, LEPIC_ERR_ARG, "poisson: more than 2^31 nodes");
  Solver<double> S;
  S.ctx = ctx;
  S.ng = ng;
  S.omega = mp->omega;
  S.flag_pbc = mp->flag_pbc;
  S.flag_nmn = mp->flag_nmn;
  // level geometry: n/2^(l-1), h*2^(l-1) (pdesolver.f90:42-51)
  int64_t coarse_nodes = 0, max_parts = 0;
  for (int l = 0; l < ng; ++l) {
    lepic_grid gl;
    for (int d = 0; d < 3; ++d) {
      gl.n[d] = g->n[d] >> l;
      gl.h[d] = g->h[d] * (double)(1 << l);
    }
    if (l < ng - 1)
      for (int d = 0; d < 3; ++d)
        if (gl.n[d] < 2 || (gl.n[d] % 2) != 0)
          return lepic_fail(ctx, LEPIC_ERR_ARG,
                            "poisson: every level above the coarsest needs even n >= 2");
    if (gl.n[0] < 1 || gl.n[1] < 1 || gl.n[2] < 1)
      return lepic_fail(ctx, LEPIC_ERR_ARG, "poisson: too many levels for this grid");
    S.L[l].g = make_kgrid(&gl);
    set_level_divs(S.L[l]);
    set_coeffs(S.L[l], mp->eps0);
    if (l > 0) coarse_nodes += grid_nodes(&gl);
    int64_t nres = (int64_t)(gl.n[0] + 1) * (gl.n[1] + 1) * (gl.n[2] + 1);
    max_parts = std::max(max_parts, (nres + BLOCK - 1) / BLOCK);
  }
  // coarse-level storage (kept across calls; labels zeroed once)
  const int64_t rp_len = ((int64_t)g->n[0] + 2) * ((int64_t)g->n[1] + 2);
  const int64_t fine_nodes = ng > 1 && mp->flag_pbc ? grid_nodes(g) : 0;   // the restriction's residual
  // the sweeps' second u arrays, block residuals and slot states
  const int64_t u2_nodes = S.u2_nodes();
  int64_t sweep_parts = 0;
  for (int l = 0; l < ng; ++l)
    sweep_parts = std::max<int64_t>(sweep_parts, sweep_grid(S.L[l].g).blocks());
  sweep_parts = std::max<int64_t>(sweep_parts, PER_BLOCKS);
  const int64_t slot_len = 3 * sweep_parts + (int64_t)(SLOTS * sizeof(SlotState) / sizeof(double));
  size_t need = sizeof(double) * (size_t)(2 * coarse_nodes + max_parts + rp_len + fine_nodes +
                                          u2_nodes + slot_len) +
                sizeof(int32_t) * (size_t)coarse_nodes + 4096;
  const int layout = ng + (mp->flag_pbc ? 256 : 0);   // the arrays' places depend on both
  bool same = ctx->mg_mem && ctx->mg_ng == layout && ctx->mg_n[0] == g->n[0] &&
              ctx->mg_n[1] == g->n[1] && ctx->mg_n[2] == g->n[2] && ctx->mg_bytes >= need;
  if (!same) {
    if (ctx->mg_mem) {
      LEPIC_HIP(ctx, hipStreamSynchronize(ctx->stream));
      LEPIC_HIP(ctx, hipFree(ctx->mg_mem));
      ctx->mg_mem = nullptr;
    }
    LEPIC_HIP(ctx, hipMalloc(&ctx->mg_mem, need));
    LEPIC_HIP(ctx, hipMemsetAsync(ctx->mg_mem, 0, need, ctx->stream));
    ctx->mg_bytes = need;
    ctx->mg_ng = layout;
    for (int d = 0; d < 3; ++d) ctx->mg_n[d] = g->n[d];
  }
  char *mem = reinterpret_cast<char *>(ctx->mg_mem);
  double *dmem = reinterpret_cast<double *>(mem);
  S.partials = dmem;
  S.rp = dmem + max_parts;
  double *lv = S.rp + rp_len;
  S.resbuf = fine_nodes ? lv + 2 * coarse_nodes : nullptr;
  double *u2 = lv + 2 * coarse_nodes + fine_nodes;
  S.slot_state = reinterpret_cast<SlotState *>(u2 + u2_nodes);
  S.slot_partials = u2 + u2_nodes + (int64_t)(SLOTS * sizeof(SlotState) / sizeof(double));
  int32_t *lb = reinterpret_cast<int32_t *>(u2 + u2_nodes + slot_len);
  S.L[0].u = phi;
  S.L[0].b = const_cast<double *>(rho);
  S.L[0].bc = const_cast<int32_t *>(bcnd);
  for (int l = 1; l < ng; ++l) {
    int64_t nn = Solver<double>::grid_nodes_k(S.L[l].g);
    S.L[l].u = lv;
    S.L[l].b = lv + nn;
    lv += 2 * nn;
    S.L[l].bc = lb;
    lb += nn;
  }
  S.place_u2(u2);
  S.ctl = reinterpret_cast<MGCtl *>(ctx->d_ctrl + CTRL_MG);
  hipLaunchKernelGGL(k_reset_totals, dim3(1), dim3(64), 0, ctx->stream, S.ctl, MAX_LEVELS);

  // pdesolver: alpha with the fine-grid ac (pdesolver.f90:33-34)
  const double alpha =
      std::fabs((double)((g->n[0] + 1) * (g->n[1] + 1) * (g->n[2] + 1)) * S.L[0].ac) * 1.0;
  const double epsa = alpha * mp->eps;
  double res = 0.0, res_s = 0.0;
  int k = 1;
  int status = LEPIC_OK;
  // a solve that fits one workgroup altogether is one launch
  S.choose_lc(ng > 1 && !S.flag_pbc ? 0 : 1);
  const bool whole = S.lc == 0;
  auto vcycle = [&](int kmg) -> int { return S.vcycle(kmg, epsa); };
  // With the coarsest level inside k_mg_coarse a V-cycle's launches are fixed
  // (every decision is taken on the device), so they are captured once per
  // solve configuration -- the first V-cycle and the later ones differ in one
  // argument -- and replayed: one submission per V-cycle instead of ~100.
  const bool replay = mp->graph && !whole && S.lc < ng;
  if (replay) {
    const int32_t ints[9] = {ng, g->n[0], g->n[1], g->n[2], S.flag_pbc, S.flag_nmn, S.lc, 0, 0};
    const void *ptrs[5] = {phi, rho, bcnd, ctx->mg_mem, ctx->d_ctrl};
    // eps0: the levels' coefficients are in the captured launches
    const double dbl[6] = {g->h[0], g->h[1], g->h[2], S.omega, epsa, mp->eps0};
    std::vector<unsigned char> key(sizeof(ints) + sizeof(ptrs) + sizeof(dbl));
    std::memcpy(key.data(), ints, sizeof(ints));
    std::memcpy(key.data() + sizeof(ints), ptrs, sizeof(ptrs));
    std::memcpy(key.data() + sizeof(ints) + sizeof(ptrs), dbl, sizeof(dbl));
    if (key != ctx->mg_key || !ctx->mg_exec[0] || !ctx->mg_exec[1]) {
      for (hipGraphExec_t &e : ctx->mg_exec)
        if (e) {
          LEPIC_HIP(ctx, hipGraphExecDestroy(e));
          e = nullptr;
        }
      ctx->mg_key.clear();
      if (!ctx->capture_stream)
        LEPIC_HIP(ctx, hipStreamCreateWithFlags(&ctx->capture_stream, hipStreamNonBlocking));
      const hipStream_t eager = ctx->stream;
      ctx->stream = ctx->capture_stream;   // the Solver launches on ctx->stream
      int st = LEPIC_OK;
      for (int which = 0; which < 2 && st == LEPIC_OK; ++which) {
        hipGraph_t graph = nullptr;
        hipError_t e = hipStreamBeginCapture(ctx->capture_stream, hipStreamCaptureModeThreadLocal);
        if (e == hipSuccess) {
          st = vcycle(which == 0 ? 1 : 2);
          e = hipStreamEndCapture(ctx->capture_stream, &graph);
        }
        if (e == hipSuccess && st == LEPIC_OK)
          e = hipGraphInstantiate(&ctx->mg_exec[which], graph, nullptr, nullptr, 0);
        if (graph) (void)hipGraphDestroy(graph);
        if (e != hipSuccess && st == LEPIC_OK) st = lepic_fail(ctx, LEPIC_ERR_HIP, hipGetErrorString(e));
      }
      ctx->stream = eager;
      if (st) return st;
      ctx->mg_key = key;
    }
  }
  for (;;) {
    if (whole) {
      S.whole(epsa, k, mp->ncycl, alpha, mp->eps, res_s);
    } else if (replay) {
      LEPIC_HIP(ctx, hipGraphLaunch(ctx->mg_exec[k == 1 ? 0 : 1], ctx->stream));
    } else {
      int st = vcycle(k);
      if (st) return st;
    }
    LEPIC_LAUNCH_CHECK(ctx, "multigrid launch");
    // the V-cycle's residual is the last sor_rb's: level 1 (or the only level)
    // every level's counters come back with the fine residual (no extra
    // round trip for the statistics)
    LEPIC_HIP(ctx, hipMemcpyAsync(ctx->h_pinned, S.ctl, sizeof(MGCtl) * MAX_LEVELS,
                                  hipMemcpyDeviceToHost, ctx->stream));
    LEPIC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    double r;
    std::memcpy(&r, &ctx->h_pinned[2], sizeof(double));
    res = r / alpha;
    if (whole) {   // the device has judged its cycles by the rules below
      k = (int)ctx->h_pinned[5];
      std::memcpy(&res_s, &ctx->h_pinned[7], sizeof(double));
      if (ctx->h_pinned[6] == WHOLE_MORE) continue;
      if (ctx->h_pinned[6] == WHOLE_DIVERGED)
        status = lepic_fail(ctx, LEPIC_ERR_DIVERGED, "poisson: res/res_s > 10 (diverging)");
      break;
    }
    if (k == 1) res_s = res;
    else if (std::fabs(res / res_s) > 10.0) {
      status = lepic_fail(ctx, LEPIC_ERR_DIVERGED, "poisson: res/res_s > 10 (diverging)");
      break;
    }
    if (res < mp->eps || k == mp->ncycl) break;
    k = k + 1;
  }
  if (stats) {
    std::memset(stats, 0, sizeof(*stats));
    double ktot = 0.0;
    for (int l = 0; l < ng; ++l) {
      int64_t tot = ctx->h_pinned[16 * l + 4];
      stats->sweeps[l] = tot;
      ktot = ktot + (double)tot / std::pow(2.0, 2.0 * l);
    }
    stats->cycles = k;
    stats->ktot = ktot;
    stats->res = res;
  }
  return status;
}

// ---------------------------------------------------------------------------
// Mixed precision: FP32 red-black smoothing V-cycles inside an FP64 iterative
// refinement.  Each refinement step forms the FP64 residual r = b - A phi at
// every node the smoother updates (the smoother's own row rules: Neumann rows
// with 2 ae and no west term, periodic copies left to the ghost update),
// rounds it to FP32, runs a few fixed-sweep FP32 V-cycles of the same
// multigrid on A e = r with e = 0 on electrodes, and adds e to phi in FP64.
// Convergence is the reference's: L1 residual over plasma nodes / alpha
// below eps (pdesolver.f90:97-115), measured on the FP64 residual.
// ---------------------------------------------------------------------------
namespace {

constexpr int MIX_BLOCKS = 1024;

// A thread's nodes in k_mix_resid and k_pcg_dir: each XCD (blocks go to them in
// turn) walks its own eighth of the nodes in order, so that the planes above and
// below are still in its L2: CG direction at 256^3 221 -> 181 us.  (k_pcg_resid
// writes more than it reads and is 4 % faster striding over all blocks.)  On fewer
// than 16 planes an XCD has one or two, and the outermost little plasma in its:
// striding, 33 us against 42 at 8 x 32768 x 8.
__device__ inline NodeWalk node_walk(const KGrid &g, int64_t nodes) {
  if (g.n3 + 3 < 16)
    return walk_strided(nodes, (int)blockIdx.x, (int)gridDim.x, (int)threadIdx.x, BLOCK);
  return walk_grouped(nodes, (int)blockIdx.x, (int)gridDim.x, (int)threadIdx.x, BLOCK, LEPIC_XCDS);
}

// FP64 residual of the refinement step at ghosted node t; r32, e32 (the
// FP32 right-hand side and correction) written for every node, the L1 sum
// over plasma nodes (in the order of sors.f90:409-431's residual) to
// partials.
__global__ __launch_bounds__(BLOCK) void k_mix_resid(KLevel L, float *r32, float *e32,
                                                     double *partials, int64_t nodes) {
  __shared__ double red[BLOCK / LEPIC_WAVE];
  const KGrid &g = L.g;
  double a = 0.0;
  const NodeWalk nw = node_walk(g, nodes);
  for (int64_t t = nw.t; t < nw.end; t += nw.step) {
    const int i = (int)(t % g.sy);
    const int64_t q = t / g.sy;
    const int j = (int)(q % (g.n2 + 3)), k = (int)(q / (g.n2 + 3));
    double r = 0.0;
    if (i >= 1 && i <= g.n1 + 1 && j >= 1 && j <= g.n2 + 1 && k >= 1 && k <= g.n3 + 1) {
      const int bcv = L.bc[t];
      const double *u = L.u;
      if (bcv == -2) {
        r = L.b[t] - (L.an * u[t + g.sy] + L.as * u[t - g.sy] + 2.0 * L.ae * u[t + 1] +
                      L.at * u[t + g.sz] + L.ab * u[t - g.sz] + L.ac * u[t]);
      } else if (bcv == -1 || (bcv == 0 && j != g.n2 + 1 && k != g.n3 + 1)) {
        r = L.b[t] - (L.aw * u[t - 1] + L.an * u[t + g.sy] + L.as * u[t - g.sy] +
                      L.ae * u[t + 1] + L.ac * u[t] + L.at * u[t + g.sz] + L.ab * u[t - g.sz]);
      }
      if (bcv == -1) a = a + fabs(r);
    }
    r32[t] = (float)r;
    e32[t] = 0.0f;
  }
  for (int d = LEPIC_WAVE / 2; d > 0; d >>= 1) a = a + __shfl_down(a, d);
  if (__lane_id() == 0) red[threadIdx.x / LEPIC_WAVE] = a;
  __syncthreads();
  if (threadIdx.x == 0) {
    double b = 0.0;
    for (int w = 0; w < BLOCK / LEPIC_WAVE; ++w) b = b + red[w];
    partials[blockIdx.x] = b;
  }
}

__global__ __launch_bounds__(BLOCK) void k_mix_sum(const double *partials, int64_t nparts,
                                                   double *out) {
  __shared__ double red[BLOCK];
  double a = 0.0;
  for (int64_t p = threadIdx.x; p < nparts; p += BLOCK) a = a + partials[p];
  red[threadIdx.x] = a;
  __syncthreads();
  for (int s = BLOCK / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] = red[threadIdx.x] + red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
}

// phi += e where the smoother may change phi (bcnd <= 0).
__global__ void k_mix_correct(double *phi, const float *e32, const int32_t *bc, int64_t nodes) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t < nodes && bc[t] <= 0) phi[t] = phi[t] + (double)e32[t];
}

}  // namespace

// ---------------------------------------------------------------------------
// Set-up shared by the two solves that smooth in FP32: the FP32 correction
// hierarchy and the FP64 work arrays on ctx->mgx_mem, laid out as
// [MIX_COLS x MIX_BLOCKS partial sums][8 scalars][nf64 FP64 node arrays]
// [e32, r32][periodic residual plane][coarse u, b][fine residual][second u
// arrays][coarse labels].
// ---------------------------------------------------------------------------
namespace {

constexpr int MIX_COLS = 4;

template <class T>
struct MixSetup {
  Solver<T> S;         // the correction hierarchy (T: FP32, or FP64 for the CG preconditioner)
  KLevel F64;          // the FP64 fine level: phi, rho, labels
  double *partials = nullptr, *scal = nullptr, *f64 = nullptr;
  T *e32 = nullptr, *r32 = nullptr;
  int64_t nodes = 0;
  double alpha = 0.0;  // pdesolver's residual normalisation
  unsigned rb = 0;     // blocks of the FP64 residual kernels
};

template <class T>
int mix_setup(lepic_ctx *ctx, const lepic_grid *g, double *phi, const double *rho,
              const int32_t *bcnd, const lepic_mg_params *mp, const lepic_mgmix_params *xp,
              int nf64, const char *who, MixSetup<T> &M) {
  const std::string w(who);
  if (!g || !phi || !rho || !bcnd || !mp || !xp)
    return lepic_fail(ctx, LEPIC_ERR_ARG, w + ": null argument");
  const int ng = mp->ng;
  if (ng < 1 || ng > MAX_LEVELS) return lepic_fail(ctx, LEPIC_ERR_ARG, w + ": ng outside [1,12]");
  if (xp->inner_cycles < 1 || xp->inner_cycles > 64 || xp->nu < 1 || xp->nu > 16 ||
      xp->nu_coarsest < 1 || xp->nu_coarsest > 100000 || !(xp->omega > 0.0 && xp->omega < 2.0))
    return lepic_fail(ctx, LEPIC_ERR_ARG, w + ": inner V-cycle parameters out of range");
  if (grid_nodes(g) > INT32_MAX)   // thread numbers are decoded in 32 bits
    return lepic_fail(ctx, LEPIC_ERR_ARG, w + ": more than 2^31 nodes");
  Solver<T> &S = M.S;
  S.ctx = ctx;
  S.ng = ng;
  S.omega = (T)xp->omega;
  S.flag_pbc = mp->flag_pbc;
  S.flag_nmn = mp->flag_nmn;
  S.fixed = 1;
  S.nr_fixed = xp->nu;
  S.nr_coarsest = xp->nu_coarsest;
  int64_t coarse_nodes = 0;
  for (int l = 0; l < ng; ++l) {
    lepic_grid gl;
    for (int d = 0; d < 3; ++d) {
      gl.n[d] = g->n[d] >> l;
      gl.h[d] = g->h[d] * (double)(1 << l);
    }
    if (l < ng - 1)
      for (int d = 0; d < 3; ++d)
        if (gl.n[d] < 2 || (gl.n[d] % 2) != 0)
          return lepic_fail(ctx, LEPIC_ERR_ARG,
                            w + ": every level above the coarsest needs even n >= 2");
    if (gl.n[0] < 1 || gl.n[1] < 1 || gl.n[2] < 1)
      return lepic_fail(ctx, LEPIC_ERR_ARG, w + ": too many levels for this grid");
    S.L[l].g = make_kgrid(&gl);
    set_level_divs(S.L[l]);
    set_coeffs(S.L[l], mp->eps0);
    if (l == 0) {
      M.F64.g = S.L[0].g;
      set_level_divs(M.F64);
      set_coeffs(M.F64, mp->eps0);
    } else {
      coarse_nodes += grid_nodes(&gl);
    }
  }
  const int64_t nodes = grid_nodes(g);
  const int64_t rp_len = ((int64_t)g->n[0] + 2) * ((int64_t)g->n[1] + 2);
  // the sweeps' second u arrays
  const int64_t u2_nodes = S.u2_nodes();
  const int64_t res_nodes = ng > 1 && mp->flag_pbc ? nodes : 0;   // the restriction's residual
  const size_t need = sizeof(double) * (size_t)(MIX_COLS * MIX_BLOCKS + 8) +
                      sizeof(double) * (size_t)nf64 * (size_t)nodes +
                      sizeof(T) * (size_t)(2 * nodes + 2 * coarse_nodes + rp_len) +
                      sizeof(T) * (size_t)res_nodes +
                      sizeof(T) * (size_t)u2_nodes +
                      sizeof(int32_t) * (size_t)coarse_nodes + 4096;
  if (!ctx->mgx_mem || ctx->mgx_bytes < need) {
    if (ctx->mgx_mem) {
      LEPIC_HIP(ctx, hipStreamSynchronize(ctx->stream));
      LEPIC_HIP(ctx, hipFree(ctx->mgx_mem));
      ctx->mgx_mem = nullptr;
      ctx->mgx_bytes = 0;
      ctx->mgx_key.clear();
      ctx->pcg_key.clear();
    }
    LEPIC_HIP(ctx, hipMalloc(&ctx->mgx_mem, need));
    LEPIC_HIP(ctx, hipMemsetAsync(ctx->mgx_mem, 0, need, ctx->stream));
    ctx->mgx_bytes = need;
  }
  M.partials = reinterpret_cast<double *>(ctx->mgx_mem);
  M.scal = M.partials + MIX_COLS * MIX_BLOCKS;
  M.f64 = M.scal + 8;
  T *fmem = reinterpret_cast<T *>(M.f64 + (size_t)nf64 * (size_t)nodes);
  M.e32 = fmem;
  M.r32 = fmem + nodes;
  T *lv = M.r32 + nodes;
  S.rp = lv;
  lv += rp_len;
  S.resbuf = res_nodes ? lv + 2 * coarse_nodes : nullptr;
  T *u2 = lv + 2 * coarse_nodes + res_nodes;
  int32_t *lb = reinterpret_cast<int32_t *>(u2 + u2_nodes);
  S.place_u2(u2);
  S.L[0].u = M.e32;
  S.L[0].b = M.r32;
  S.L[0].bc = const_cast<int32_t *>(bcnd);
  for (int l = 1; l < ng; ++l) {
    const int64_t nn = Solver<T>::grid_nodes_k(S.L[l].g);
    S.L[l].u = lv;
    S.L[l].b = lv + nn;
    lv += 2 * nn;
    S.L[l].bc = lb;
    lb += nn;
  }
  S.partials = M.partials;   // unused with fixed sweeps
  S.ctl = reinterpret_cast<MGCtl *>(ctx->d_ctrl + CTRL_MG);
  S.choose_lc();
  M.F64.u = phi;
  M.F64.b = const_cast<double *>(rho);
  M.F64.bc = const_cast<int32_t *>(bcnd);
  M.nodes = nodes;
  M.alpha =
      std::fabs((double)((g->n[0] + 1) * (g->n[1] + 1) * (g->n[2] + 1)) * M.F64.ac) * 1.0;
  M.rb = (unsigned)std::min<int64_t>(grid_blocks(nodes, BLOCK), MIX_BLOCKS);
  return LEPIC_OK;
}

}  // namespace

extern "C" int lepic_poisson_solve_mixed(lepic_ctx *ctx, const lepic_grid *g, double *phi,
                                         const double *rho, const int32_t *bcnd,
                                         const lepic_mg_params *mp, const lepic_mgmix_params *xp,
                                         lepic_mg_stats *stats) {
  if (!ctx) return LEPIC_ERR_ARG;
  MixSetup<float> M;
  int st0 = mix_setup(ctx, g, phi, rho, bcnd, mp, xp, 0, "poisson_mixed", M);
  if (st0) return st0;
  Solver<float> &S = M.S;
  KLevel &F64 = M.F64;
  const int ng = mp->ng;
  const int64_t nodes = M.nodes;
  double *partials = M.partials;
  double *res_dev = M.scal;
  float *e32 = M.e32, *r32 = M.r32;
  const double alpha = M.alpha;
  const unsigned rb = M.rb;
  // phi's periodic ghosts from their images (sors.f90:184-239): before the first
  // residual, which reads them as a caller left them, and after a correction
  auto ghosts = [&]() {
    if (!mp->flag_pbc) return;
    const KGrid &gg = F64.g;
    const MGCtl *always = nullptr;
    hipLaunchKernelGGL(k_per_y<double>, dim3(grid_blocks((int64_t)(gg.n1 + 3) * (gg.n3 + 3), BLOCK)),
                       dim3(BLOCK), 0, ctx->stream, F64, always);
    hipLaunchKernelGGL(k_per_z<double>, dim3(grid_blocks((int64_t)(gg.n1 + 3) * (gg.n2 + 3), BLOCK)),
                       dim3(BLOCK), 0, ctx->stream, F64, always);
  };
  // the inner V-cycles and the correction of one refinement step: one
  // captured graph per solve configuration
  auto inner = [&]() -> int {
    for (int c = 0; c < xp->inner_cycles; ++c) {
      int st = S.vcycle(2, 0.0, c == 0);
      if (st) return st;
    }
    hipLaunchKernelGGL(k_mix_correct, dim3(grid_blocks(nodes, 256)), dim3(256), 0, ctx->stream,
                       phi, e32, bcnd, nodes);
    ghosts();
    return LEPIC_OK;
  };
  const bool replay = mp->graph != 0;
  if (replay) {
    const int32_t ints[10] = {ng, g->n[0], g->n[1], g->n[2], mp->flag_pbc, mp->flag_nmn,
                              xp->inner_cycles, xp->nu, xp->nu_coarsest, S.lc};
    const void *ptrs[4] = {phi, bcnd, ctx->mgx_mem, ctx->d_ctrl};
    const double dbl[5] = {g->h[0], g->h[1], g->h[2], xp->omega, mp->eps0};
    std::vector<unsigned char> key(sizeof(ints) + sizeof(ptrs) + sizeof(dbl));
    std::memcpy(key.data(), ints, sizeof(ints));
    std::memcpy(key.data() + sizeof(ints), ptrs, sizeof(ptrs));
    std::memcpy(key.data() + sizeof(ints) + sizeof(ptrs), dbl, sizeof(dbl));
    if (key != ctx->mgx_key || !ctx->mgx_exec) {
      if (ctx->mgx_exec) {
        LEPIC_HIP(ctx, hipGraphExecDestroy(ctx->mgx_exec));
        ctx->mgx_exec = nullptr;
      }
      ctx->mgx_key.clear();
      if (!ctx->capture_stream)
        LEPIC_HIP(ctx, hipStreamCreateWithFlags(&ctx->capture_stream, hipStreamNonBlocking));
      const hipStream_t eager = ctx->stream;
      ctx->stream = ctx->capture_stream;   // the Solver launches on ctx->stream
      int st = LEPIC_OK;
      hipGraph_t graph = nullptr;
      hipError_t e = hipStreamBeginCapture(ctx->capture_stream, hipStreamCaptureModeThreadLocal);
      if (e == hipSuccess) {
        st = inner();
        e = hipStreamEndCapture(ctx->capture_stream, &graph);
      }
      if (e == hipSuccess && st == LEPIC_OK)
        e = hipGraphInstantiate(&ctx->mgx_exec, graph, nullptr, nullptr, 0);
      if (graph) (void)hipGraphDestroy(graph);
      ctx->stream = eager;
      if (st) return st;
      if (e != hipSuccess) return lepic_fail(ctx, LEPIC_ERR_HIP, hipGetErrorString(e));
      ctx->mgx_key = key;
    }
  }
  hipLaunchKernelGGL(k_reset_totals, dim3(1), dim3(64), 0, ctx->stream, S.ctl, MAX_LEVELS);
  ghosts();
  double res = 0.0, res_s = 0.0;
  int k = 0;
  int status = LEPIC_OK;
  for (;;) {
    hipLaunchKernelGGL(k_mix_resid, dim3(rb), dim3(BLOCK), 0, ctx->stream, F64, r32, e32,
                       partials, nodes);
    hipLaunchKernelGGL(k_mix_sum, dim3(1), dim3(BLOCK), 0, ctx->stream, partials, (int64_t)rb,
                       res_dev);
    LEPIC_LAUNCH_CHECK(ctx, "mixed residual");
    LEPIC_HIP(ctx, hipMemcpyAsync(ctx->h_pinned, res_dev, sizeof(double), hipMemcpyDeviceToHost,
                                  ctx->stream));
    LEPIC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    double r;
    std::memcpy(&r, &ctx->h_pinned[0], sizeof(double));
    res = r / alpha;
    if (k == 0) res_s = res;
    else if (std::fabs(res / res_s) > 10.0) {
      status = lepic_fail(ctx, LEPIC_ERR_DIVERGED, "poisson_mixed: res/res_s > 10 (diverging)");
      break;
    }
    if (res < mp->eps || k == mp->ncycl) break;
    ++k;
    if (replay) {
      LEPIC_HIP(ctx, hipGraphLaunch(ctx->mgx_exec, ctx->stream));
    } else {
      int st = inner();
      if (st) return st;
    }
    LEPIC_LAUNCH_CHECK(ctx, "mixed refinement step");
  }
  if (stats) {
    std::memset(stats, 0, sizeof(*stats));
    double ktot = 0.0;
    for (int l = 0; l < ng; ++l) {
      // fixed sweep counts: nu per leg on every level above the coarsest
      const int64_t per = (l == ng - 1) ? xp->nu_coarsest : 2 * xp->nu;
      const int64_t tot = per * (int64_t)xp->inner_cycles * k;
      stats->sweeps[l] = tot;
      ktot = ktot + (double)tot / std::pow(2.0, 2.0 * l);
    }
    stats->cycles = k;
    stats->ktot = ktot;
    stats->res = res;
  }
  return status;
}

// ---------------------------------------------------------------------------
// Preconditioned conjugate gradients: the FP32 V-cycles of the mixed solve
// used as the preconditioner of an FP64 flexible CG (Notay's FCG with one
// previous direction kept) on the plasma nodes.  With plasma (-1) and
// electrode (> 0) labels and no periodic or Neumann walls the operator is
// the symmetric 7-point Dirichlet operator of sors.f90 restricted to plasma
// nodes; the V-cycle is applied to A z = r from z = 0 with fixed sweeps.  An
// iteration: z = M(r); p = z - (<z, A p_old> / <p_old, A p_old>) p_old;
// q = A p; phi += a p, r -= a q with a = <p, r> / <p, q>.  It stops on the
// reference's criterion (L1 residual over plasma nodes / alpha < eps),
// confirmed on the residual recomputed from phi.
// ---------------------------------------------------------------------------
namespace {

__device__ inline double block_sum_d(double a, double *red) {
  for (int d = LEPIC_WAVE / 2; d > 0; d >>= 1) a = a + __shfl_down(a, d);
  if (__lane_id() == 0) red[threadIdx.x / LEPIC_WAVE] = a;
  __syncthreads();
  double b = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < BLOCK / LEPIC_WAVE; ++w) b = b + red[w];
  __syncthreads();
  return b;
}

// The residual from phi (start and restarts): r = b - A phi on plasma nodes,
// 0 elsewhere; the directions p, q cleared; r32 = r, e32 = 0; the L1 sum to
// partials column 0; a physical node labelled 0 or -2, or a ghost node
// labelled -1, raises *bad.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_pcg_resid(KLevel L, MDiv dy, double *r, double *p,
                                                     double *q, T *r32, T *e32,
                                                     double *partials, int *bad, int64_t nodes) {
  __shared__ double red[BLOCK / LEPIC_WAVE];
  const KGrid &g = L.g;
  double a = 0.0;
  int flag = 0;
  const int64_t stride = (int64_t)gridDim.x * BLOCK;
  for (int64_t t = blockIdx.x * (int64_t)BLOCK + threadIdx.x; t < nodes; t += stride) {
    const uint32_t tt = (uint32_t)t, row = mdiv_q(tt, L.d_n1p3), kk = mdiv_q(row, dy);
    const int i = (int)(tt - row * (uint32_t)(g.n1 + 3));
    const int j = (int)(row - kk * (uint32_t)(g.n2 + 3)), k = (int)kk;
    double rv = 0.0;
    if (i >= 1 && i <= g.n1 + 1 && j >= 1 && j <= g.n2 + 1 && k >= 1 && k <= g.n3 + 1) {
      const int bcv = L.bc[t];
      const double *u = L.u;
      if (bcv == -1) {
        rv = L.b[t] - (L.aw * u[t - 1] + L.an * u[t + g.sy] + L.as * u[t - g.sy] +
                       L.ae * u[t + 1] + L.ac * u[t] + L.at * u[t + g.sz] + L.ab * u[t - g.sz]);
        a = a + fabs(rv);
      } else if (bcv == 0 || bcv == -2) {
        flag = 1;
      }
    } else if (L.bc[t] == -1) {
      flag = 1;   // a plasma label on a ghost node: its stencil would leave the array
    }
    r[t] = rv;
    p[t] = 0.0;
    q[t] = 0.0;
    r32[t] = (T)rv;
    e32[t] = T(0);
  }
  const double s = block_sum_d(a, red);
  if (threadIdx.x == 0) partials[blockIdx.x] = s;
  if (__syncthreads_or(flag) && threadIdx.x == 0) atomicOr(bad, 1);
}

// <z, q_old> (z = e32, zero off the plasma nodes) to partials column 1.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_pcg_zq(const T *e32, const double *q,
                                                  double *partials, int64_t nodes) {
  __shared__ double red[BLOCK / LEPIC_WAVE];
  double a = 0.0;
  const int64_t stride = (int64_t)gridDim.x * BLOCK;
  for (int64_t t = blockIdx.x * (int64_t)BLOCK + threadIdx.x; t < nodes; t += stride)
    a = a + (double)e32[t] * q[t];
  const double s = block_sum_d(a, red);
  if (threadIdx.x == 0) partials[MIX_BLOCKS + blockIdx.x] = s;
}

// The new direction p_new = z - beta p (beta = scal[1] / scal[2], the
// previous <p, q>) on plasma nodes, 0 elsewhere, and q = A p_new from the
// neighbours' p_new formed on the fly (z and p are 0 off the plasma nodes);
// <p_new, q> and <p_new, r> to partials columns 2 and 3.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_pcg_dir(KLevel L, const T *e32, const double *p,
                                                   double *pn_out, double *q, const double *r,
                                                   const double *scal, double *partials,
                                                   int64_t nodes) {
  __shared__ double red[BLOCK / LEPIC_WAVE];
  const KGrid &g = L.g;
  const double beta = scal[2] != 0.0 ? scal[1] / scal[2] : 0.0;
  double apq = 0.0, apr = 0.0;
  const NodeWalk nw = node_walk(g, nodes);
  for (int64_t t = nw.t; t < nw.end; t += nw.step) {
    double pn = 0.0, qv = 0.0;
    if (L.bc[t] == -1) {
      auto P = [&](int64_t u) { return (double)e32[u] - beta * p[u]; };
      pn = P(t);
      qv = L.aw * P(t - 1) + L.an * P(t + g.sy) + L.as * P(t - g.sy) + L.ae * P(t + 1) +
           L.ac * pn + L.at * P(t + g.sz) + L.ab * P(t - g.sz);
      apq = apq + pn * qv;
      apr = apr + pn * r[t];
    }
    pn_out[t] = pn;
    q[t] = qv;
  }
  const double s1 = block_sum_d(apq, red);
  const double s2 = block_sum_d(apr, red);
  if (threadIdx.x == 0) {
    partials[2 * MIX_BLOCKS + blockIdx.x] = s1;
    partials[3 * MIX_BLOCKS + blockIdx.x] = s2;
  }
}

// phi += a p_new, r -= a q (a = scal[3] / scal[2]) on plasma nodes; r32 = r,
// e32 = 0 (unless null), p = p_new; the L1 sum of r to partials column 0.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_pcg_update(double *phi, const int32_t *bc,
                                                      const double *pn, const double *q,
                                                      double *p, double *r, T *r32,
                                                      T *e32, const double *scal,
                                                      double *partials, int64_t nodes) {
  __shared__ double red[BLOCK / LEPIC_WAVE];
  const double a = scal[2] != 0.0 ? scal[3] / scal[2] : 0.0;
  double l1 = 0.0;
  const int64_t stride = (int64_t)gridDim.x * BLOCK;
  for (int64_t t = blockIdx.x * (int64_t)BLOCK + threadIdx.x; t < nodes; t += stride) {
    const double pv = pn[t];
    if (bc[t] == -1) {
      phi[t] = phi[t] + a * pv;
      const double rv = r[t] - a * q[t];
      r[t] = rv;
      r32[t] = (T)rv;
      l1 = l1 + fabs(rv);
    }
    p[t] = pv;
    if (e32) e32[t] = T(0);
  }
  const double s = block_sum_d(l1, red);
  if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// scal[first + c] = the sum of partials column first + c (one block each).
__global__ __launch_bounds__(BLOCK) void k_pcg_sum(const double *partials, int64_t nparts,
                                                   int first, double *scal) {
  __shared__ double red[BLOCK];
  const int col = first + (int)blockIdx.x;
  const double *pc = partials + (int64_t)col * MIX_BLOCKS;
  double a = 0.0;
  for (int64_t i = threadIdx.x; i < nparts; i += BLOCK) a = a + pc[i];
  red[threadIdx.x] = a;
  __syncthreads();
  for (int s = BLOCK / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] = red[threadIdx.x] + red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) scal[col] = red[0];
}

__global__ void k_pcg_clear_flag(int *bad) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *bad = 0;
}

}  // namespace

namespace {

template <class T>
int pcg_solve(lepic_ctx *ctx, const lepic_grid *g, double *phi, const double *rho,
              const int32_t *bcnd, const lepic_mg_params *mp, const lepic_mgmix_params *xp,
              lepic_mg_stats *stats) {
  MixSetup<T> M;
  // FP64 arrays: r, p, p_new, q
  int st0 = mix_setup(ctx, g, phi, rho, bcnd, mp, xp, 4, "poisson_pcg", M);
  if (st0) return st0;
  Solver<T> &S = M.S;
  KLevel &F64 = M.F64;
  const int ng = mp->ng;
  const int64_t nodes = M.nodes;
  double *r = M.f64, *p = r + nodes, *pn = p + nodes, *q = pn + nodes;
  double *scal = M.scal;
  int *bad = reinterpret_cast<int *>(scal + 4);
  const unsigned rb = M.rb;
  const MDiv dy = mdiv((uint32_t)(g->n[1] + 3));
  hipStream_t &s = ctx->stream;
  auto iteration = [&]() -> int {
    for (int c = 0; c < xp->inner_cycles; ++c) {
      int st = S.vcycle(2, 0.0, c == 0);
      if (st) return st;
    }
    hipLaunchKernelGGL(k_pcg_zq<T>, dim3(rb), dim3(BLOCK), 0, s, M.e32, q, M.partials, nodes);
    hipLaunchKernelGGL(k_pcg_sum, dim3(1), dim3(BLOCK), 0, s, M.partials, (int64_t)rb, 1, scal);
    hipLaunchKernelGGL(k_pcg_dir<T>, dim3(rb), dim3(BLOCK), 0, s, F64, M.e32, p, pn, q, r, scal,
                       M.partials, nodes);
    hipLaunchKernelGGL(k_pcg_sum, dim3(2), dim3(BLOCK), 0, s, M.partials, (int64_t)rb, 2, scal);
    hipLaunchKernelGGL(k_pcg_update<T>, dim3(rb), dim3(BLOCK), 0, s, phi, bcnd, pn, q, p, r, M.r32,
                       S.tiled(0, -1) ? (T *)nullptr : M.e32, scal, M.partials, nodes);
    hipLaunchKernelGGL(k_pcg_sum, dim3(1), dim3(BLOCK), 0, s, M.partials, (int64_t)rb, 0, scal);
    return LEPIC_OK;
  };
  const bool replay = mp->graph != 0;
  if (replay) {
    const int32_t ints[10] = {ng, g->n[0], g->n[1], g->n[2], 0, (int32_t)sizeof(T),
                              xp->inner_cycles, xp->nu, xp->nu_coarsest, S.lc};
    const void *ptrs[4] = {phi, bcnd, ctx->mgx_mem, ctx->d_ctrl};
    const double dbl[5] = {g->h[0], g->h[1], g->h[2], xp->omega, mp->eps0};
    std::vector<unsigned char> key(sizeof(ints) + sizeof(ptrs) + sizeof(dbl));
    std::memcpy(key.data(), ints, sizeof(ints));
    std::memcpy(key.data() + sizeof(ints), ptrs, sizeof(ptrs));
    std::memcpy(key.data() + sizeof(ints) + sizeof(ptrs), dbl, sizeof(dbl));
    if (key != ctx->pcg_key || !ctx->pcg_exec) {
      if (ctx->pcg_exec) {
        LEPIC_HIP(ctx, hipGraphExecDestroy(ctx->pcg_exec));
        ctx->pcg_exec = nullptr;
      }
      ctx->pcg_key.clear();
      if (!ctx->capture_stream)
        LEPIC_HIP(ctx, hipStreamCreateWithFlags(&ctx->capture_stream, hipStreamNonBlocking));
      const hipStream_t eager = ctx->stream;
      ctx->stream = ctx->capture_stream;   // the Solver and the lambda launch on ctx->stream
      int st = LEPIC_OK;
      hipGraph_t graph = nullptr;
      hipError_t e = hipStreamBeginCapture(ctx->capture_stream, hipStreamCaptureModeThreadLocal);
      if (e == hipSuccess) {
        st = iteration();
        e = hipStreamEndCapture(ctx->capture_stream, &graph);
      }
      if (e == hipSuccess && st == LEPIC_OK)
        e = hipGraphInstantiate(&ctx->pcg_exec, graph, nullptr, nullptr, 0);
      if (graph) (void)hipGraphDestroy(graph);
      ctx->stream = eager;
      if (st) return st;
      if (e != hipSuccess) return lepic_fail(ctx, LEPIC_ERR_HIP, hipGetErrorString(e));
      ctx->pcg_key = key;
    }
  }
  // r from phi (and the directions cleared), read back with the label flag
  auto restart = [&]() -> int {
    hipLaunchKernelGGL(k_pcg_clear_flag, dim3(1), dim3(64), 0, s, bad);
    hipLaunchKernelGGL(k_pcg_resid<T>, dim3(rb), dim3(BLOCK), 0, s, F64, dy, r, p, q, M.r32, M.e32,
                       M.partials, bad, nodes);
    hipLaunchKernelGGL(k_pcg_sum, dim3(1), dim3(BLOCK), 0, s, M.partials, (int64_t)rb, 0, scal);
    LEPIC_LAUNCH_CHECK(ctx, "pcg residual");
    return LEPIC_OK;
  };
  auto read_back = [&](double &res, int &flag) -> int {
    LEPIC_HIP(ctx, hipMemcpyAsync(ctx->h_pinned, scal, 5 * sizeof(double), hipMemcpyDeviceToHost,
                                  s));
    LEPIC_HIP(ctx, hipStreamSynchronize(s));
    double v;
    std::memcpy(&v, &ctx->h_pinned[0], sizeof(double));
    std::memcpy(&flag, &ctx->h_pinned[4], sizeof(int));
    res = v / M.alpha;
    return LEPIC_OK;
  };
  hipLaunchKernelGGL(k_reset_totals, dim3(1), dim3(64), 0, s, S.ctl, MAX_LEVELS);
  int st = restart();
  if (st) return st;
  double res = 0.0;
  int flag = 0;
  if ((st = read_back(res, flag))) return st;
  if (flag)
    return lepic_fail(ctx, LEPIC_ERR_ARG,
                      "poisson_pcg: labels 0 or -2 (the operator is not symmetric), or plasma "
                      "on a ghost node");
  const double res_s = res;
  int k = 0;
  bool fresh = true;   // r was just formed from phi
  int status = LEPIC_OK;
  for (;;) {
    if (res < mp->eps) {
      if (fresh) break;
      if ((st = restart())) return st;   // confirm on the residual from phi
      if ((st = read_back(res, flag))) return st;
      fresh = true;
      if (res < mp->eps) break;
    }
    if (k == mp->ncycl) break;
    ++k;
    if (replay) {
      LEPIC_HIP(ctx, hipGraphLaunch(ctx->pcg_exec, s));
    } else if ((st = iteration())) {
      return st;
    }
    LEPIC_LAUNCH_CHECK(ctx, "pcg iteration");
    if ((st = read_back(res, flag))) return st;
    fresh = false;
    // the residual of conjugate gradients need not fall at every iteration:
    // only a non-finite or exploding one stops the solve
    if (!(res <= 1.0e6 * res_s)) {
      status = lepic_fail(ctx, LEPIC_ERR_DIVERGED, "poisson_pcg: res/res_s > 1e6 (diverging)");
      break;
    }
  }
  if (stats) {
    std::memset(stats, 0, sizeof(*stats));
    double ktot = 0.0;
    for (int l = 0; l < ng; ++l) {
      const int64_t per = (l == ng - 1) ? xp->nu_coarsest : 2 * xp->nu;
      const int64_t tot = per * (int64_t)xp->inner_cycles * k;
      stats->sweeps[l] = tot;
      ktot = ktot + (double)tot / std::pow(2.0, 2.0 * l);
    }
    stats->cycles = k;
    stats->ktot = ktot;
    stats->res = res;
  }
  return status;
}

}  // namespace

extern "C" int lepic_poisson_solve_pcg(lepic_ctx *ctx, const lepic_grid *g, double *phi,
                                       const double *rho, const int32_t *bcnd,
                                       const lepic_mg_params *mp, const lepic_mgmix_params *xp,
                                       lepic_mg_stats *stats) {
  if (!ctx) return LEPIC_ERR_ARG;
  if (!mp || !xp) return lepic_fail(ctx, LEPIC_ERR_ARG, "poisson_pcg: null argument");
  if (mp->flag_pbc || mp->flag_nmn)
    return lepic_fail(ctx, LEPIC_ERR_ARG,
                      "poisson_pcg: periodic or Neumann walls (the operator is not symmetric)");
  if (xp->precond_fp64 != 0 && xp->precond_fp64 != 1)
    return lepic_fail(ctx, LEPIC_ERR_ARG, "poisson_pcg: precond_fp64 must be 0 or 1");
  return xp->precond_fp64 ? pcg_solve<double>(ctx, g, phi, rho, bcnd, mp, xp, stats)
                          : pcg_solve<float>(ctx, g, phi, rho, bcnd, mp, xp, stats);
}
