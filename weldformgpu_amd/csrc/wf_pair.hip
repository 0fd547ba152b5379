// wf_pair.hip — the pair loops of the step (gfx950), FP64 and mixed
// precision, on two kernel templates: k_pair_lds, with everything a pair reads
// of its neighbour staged in LDS (domains with one h), and k_pair_gather, which
// gathers it (the others, described first).
//
// One workgroup per tile of kTileP Morton-consecutive particles, two threads
// per particle.  The tile's staged set (the particles that are a neighbour of
// at least one of the tile's particles, in cell order) is written to LDS as
// {tile-frame position, particle index} slots; each thread walks half of its
// particle's neighbour list (16-bit staged positions in ascending order,
// four per 8-byte word, every other word), reads the neighbour's position and
// index from LDS and gathers the neighbour's packed record from global
// memory.  Two threads per particle give a CU twice the wavefronts for the
// same LDS; the loops' registers then allow 4-6 (FP32) or 3-4 (FP64)
// wavefronts per SIMD.  The per-pair physics is the reference's
// (InteractionAlt.cu, Thermal.cu, Geometry.cu), with per-particle factors
// (m/rho, sigma/rho^2, 1/h) formed once instead of once per pair; the
// policies (DensD/DensG, RatesD/RatesG, AccelD/AccelG, CondD/CondG, SurfD,
// CondDens) say what a neighbour record holds and what a pair adds.
#include <hip/hip_ext.h>

#include <climits>
#include <type_traits>

#include "wf_stress.hpp"
#include "wf_tiles.hpp"

// straight-line batches (drop(), below): not in the FP32 rates loop (0.072 vs
// 0.059 ms on a 759k-particle cylinder) and off in the gathering FP64
// acceleration loop (0.346 vs 0.321 ms)
#ifndef WF_DROP_ACCEL64
#define WF_DROP_ACCEL64 0
#endif
// cooperative record loads (coload_rec) in the FP64 acceleration, density
// and conduction loops (759k-particle cylinder, yielding: acceleration 0.333
// -> 0.291 ms, density 0.151 -> 0.143, conduction 0.137 -> 0.128); the FP64
// rates loop (0.145 -> 0.149) and the FP32 acceleration loop (0.118 ->
// 0.120) were slower with them and load per lane
#ifndef WF_COLOAD64
#define WF_COLOAD64 1
#endif

namespace wf {

// Neighbour-slot reader over the quad layout: four 16-bit slots per 8 bytes,
// the next quad prefetched one quad ahead.
struct SlotReader {
  const uint2* q;
  int64_t npad;
  int i, cnt, k;
  uint2 cur, nxt;
  __device__ __forceinline__ void init(const TileLists& tl, int i_, int cnt_) {
    q = tl.slotq;
    npad = tl.npad;
    i = i_;
    cnt = cnt_;
    k = 0;
    cur = cnt > 0 ? q[i] : make_uint2(0u, 0u);
    nxt = cnt > 4 ? q[npad + i] : make_uint2(0u, 0u);
  }
  __device__ __forceinline__ int slot() const {
    unsigned w = (k & 2) ? cur.y : cur.x;
    return (int)((w >> ((k & 1) * 16)) & 0xFFFFu);
  }
  __device__ __forceinline__ void advance() {
    k++;
    if ((k & 3) == 0) {
      cur = nxt;
      if (k + 4 < cnt) nxt = q[(int64_t)((k >> 2) + 1) * npad + i];
    }
  }
  // to the start of the next quad
  __device__ __forceinline__ void skip_quad() {
    k = (k | 3) + 1;
    cur = nxt;
    if (k + 4 < cnt) nxt = q[(int64_t)((k >> 2) + 1) * npad + i];
  }
};

// Workgroups are dispatched round-robin over the 8 XCDs (XCD = block % 8).
// Give each XCD one contiguous run of tiles so that tiles sharing staged
// cells share that XCD's L2.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_tile(int b, int nt) {
  const int q = nt / kXcds, r = nt % kXcds;
  const int x = b % kXcds, k = b / kXcds;
  return x * q + min(x, r) + k;
}

// Gather of particle j's record from an array of S-byte records (+ off
// bytes) through a 32-bit byte offset: the load then takes the array base
// from scalar registers and the offset costs one shift (a 64-bit index costs
// three instructions).  Domains hold at most kMaxParticles particles, so
// j * S stays below 2^32.
template <class T, unsigned S = sizeof(T)>
__device__ __forceinline__ T gat(const void* base, int j, unsigned off = 0) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + (unsigned)j * S + off);
}

// lanes 2p and 2p+1 swap a 32-bit word (DPP quad permutation [1, 0, 3, 2])
__device__ __forceinline__ unsigned swap_lane_pair(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false);
}

// Cooperative record loads for two lanes per particle: lanes 2p and 2p+1
// each hold one neighbour j, and both load both records, lane s reading the
// 16-byte chunks c with c % 2 == s ^ r of record r (r = 0: lane 2p's
// neighbour, r = 1: lane 2p+1's).  A load instruction then touches one record
// per lane pair instead of one per lane: the address unit's cost per gather
// grows with the distinct cache lines it touches, so this halves that cost
// for the same bytes.  Each lane keeps the half of its own record that it
// read and swaps the other half with its partner.  C: chunks per record of
// rec_bytes = 16 C at base.
template <int C>
__device__ __forceinline__ void coload_rec(const void* base, int j, int sub, uint4 (&out)[C]) {
  static_assert(C % 2 == 0, "whole chunk pairs");
  const int jo = (int)swap_lane_pair((unsigned)j);
  const int j0 = sub ? jo : j, j1 = sub ? j : jo;
  uint4 a[C / 2], b[C / 2];
#pragma unroll
  for (int c = 0; c < C / 2; c++) a[c] = gat<uint4, 16 * C>(base, j0, 16u * (2 * c + sub));
#pragma unroll
  for (int c = 0; c < C / 2; c++) b[c] = gat<uint4, 16 * C>(base, j1, 16u * (2 * c + (sub ^ 1)));
  // lane 2p read the even chunks of its record (a) and the odd ones of its
  // partner's (b); lane 2p+1 the odd chunks of lane 2p's record (a) and the
  // even ones of its own (b)
#pragma unroll
  for (int c = 0; c < C / 2; c++) {
    const uint4 send = sub ? a[c] : b[c];
    out[2 * c] = sub ? b[c] : a[c];
    out[2 * c + 1] = make_uint4(swap_lane_pair(send.x), swap_lane_pair(send.y),
                                swap_lane_pair(send.z), swap_lane_pair(send.w));
  }
}

// The acceleration pass may integrate each particle as soon as its sum
// is done (the step's BC + position/velocity update, integrate_apply):
// other tiles still read the old positions and records, so the new ones go to
// the spare planes in out, swapped in by the caller after the pass.
struct IntegratePrm {
  double dt;
  BcTable bc;
  Frame32 fr;
  IntegrateOut out;
  // a particle with contact candidates (contacts[i] > 0) is left to the contact
  // pass, which raises its acceleration first; null: none
  const int* contacts;
};

// FP64 policies need no per-tile context
struct NoCtx {};

// ---------------------------------------------------------------------------
// Per-pair cubic-spline gradient GK = (1/r) dW/dr (Functions.cu:76-88) from
// r^2: one refined reciprocal square root instead of sqrt + three IEEE
// divisions.  With hj == hi (the solver sets one h for all particles,
// Domain_d::Set_h) the thread's own 1/h and 3/(pi h^4) are reused, so the
// common case needs no division at all.
//
// The two branches of dW/dq (q < 1: -3q + 9/4 q^2; 1 <= q < 2: -3/4 (2-q)^2;
// else 0) are one branch-free expression: with u = clamp(1 - q, 0, 1) and
// t = clamp(1 - q/2, 0, 1),  dW/dq = 3 (u^2 - t^2) = 3 (u - t)(u + t)
// (for q < 1, 3[(1-q)^2 - (1-q/2)^2] = -3q + 9/4 q^2; for 1 <= q < 2, u = 0
// and -3 t^2 = -3/4 (2-q)^2; for q >= 2 both are 0).  Each clamp folds into
// the instruction that produces it, so the polynomial costs five operations
// and no divergent branch.  Differences from the reference's expression
// order are a few ulp.
struct HConst {
  double h, inv_h, C3;  // h, 1/h, 3/(pi h^4)
};
__device__ __forceinline__ HConst hconst(double h) {
  return HConst{h, 1.0 / h, 3.0 / (h * h * h * h * kPi)};
}
__device__ __forceinline__ double rsqrt_f64(double x) {
  double y = __builtin_amdgcn_rsq(x);
  const double hx = 0.5 * x;
  y = y * (1.5 - hx * y * y);
  y = y * (1.5 - hx * y * y);
  return y;
}
// 1/x to within an ulp: the hardware estimate and two Newton steps
__device__ __forceinline__ double rcp_f64(double x) {
  double y = __builtin_amdgcn_rcp(x);
  double e = __builtin_fma(-x, y, 1.0);
  y = __builtin_fma(y, e, y);
  e = __builtin_fma(-x, y, 1.0);
  return __builtin_fma(y, e, y);
}
__device__ __forceinline__ double clamp01(double x) { return fmin(fmax(x, 0.0), 1.0); }
__device__ __forceinline__ float clamp01f(float x) { return fminf(fmaxf(x, 0.f), 1.f); }
__device__ __forceinline__ double gk_pair(double r2, double hj, const HConst& hc, double& rinv,
                                          double& h_) {
  // coincident particles (never in a list built with d2 > 0, but possible
  // after motion) give q = 0, where dW/dq = 0, and contribute nothing
  rinv = rsqrt_f64(fmax(r2, 1e-300));
  const double rij = r2 * rinv;
  double inv_h = hc.inv_h, C3 = hc.C3;
  h_ = hc.h;
  if (hj != hc.h) {
    h_ = (hc.h + hj) / 2.0;
    inv_h = 1.0 / h_;
    C3 = 3.0 / (h_ * h_ * h_ * h_ * kPi);
  }
  const double q = rij * inv_h;
  const double u = clamp01(1.0 - q), t = clamp01(1.0 - 0.5 * q);
  return C3 * rinv * ((u - t) * (u + t));
}

// gather-kernel traits of a policy: the staged position type, positions per
// LDS pass, the per-tile context and a neighbour's staged position
// staged slots per LDS pass: 1024 x 32 B (FP64 position + index) = 32 KB;
// on a cubic lattice with h = 1.2 dx a tile's staged set holds ~740
// particles (at most ~910), so every tile takes the one-pass path
#ifndef WF_STAGE64
#define WF_STAGE64 1024
#endif
constexpr int kStage64 = WF_STAGE64;
// threads per particle in the pair loops (each takes every LANES-th slot
// quad); on a 759k-particle cylinder two threads take the FP32 step from
// 0.672 to 0.591 ms (four: 0.678 ms) and, with the 32 KB FP64 stage, the
// FP64 step from 1.00 to 0.90 ms
#ifndef WF_LANES64
#define WF_LANES64 2
#endif
#ifndef WF_LANES32
#define WF_LANES32 2
#endif
#define WF_GATHER64                                                                  \
  typedef double PT;                                                                 \
  static constexpr int STAGE = kStage64;                                             \
  static constexpr int LANES = WF_LANES64;                                           \
  typedef NoCtx Ctx;                                                                 \
  template <class P>                                                                 \
  __device__ static Ctx ctx(const Fields&, int, const P&) {                          \
    return Ctx{};                                                                    \
  }                                                                                  \
  __device__ static void pos(const Fields& f, int j, const Ctx&, double& x, double& y, \
                             double& z) {                                            \
    x = f.x[0][j];                                                                   \
    y = f.x[1][j];                                                                   \
    z = f.x[2][j];                                                                   \
  }

// LDS layout of a policy whose neighbours are staged whole (k_pair_lds): nv
// 16-byte and nw (0 or 1) 8- or 4-byte entries a neighbour, each entry its
// own array of SET.  On a cubic lattice with h = 1.2 dx a tile's staged set
// holds ~730 particles (at most ~930); under a list skin that reaches the
// next lattice shell ~760 (at most ~990, 1 % of the tiles above 960).  1,024
// leave the workgroups a CU that 960 leave, but for the loops with 56 bytes
// (FP64 density and rates: two instead of three) and 32 (FP32 density, rates
// and conduction: four instead of five; rates 0.061 against 0.057 ms): those
// take 960 where there are more tiles than two a CU (launch_pair).
#define WF_LDS64(nv, nw) \
  typedef double2 LV;    \
  typedef double LW;     \
  static constexpr int NV = nv, NW = nw, SET = 16 * nv + 8 * nw == 56 ? 960 : 1024;
#define WF_LDS32(nv, nw) \
  typedef float4 LV;     \
  typedef float LW;      \
  static constexpr int NV = nv, NW = nw, SET = 16 * nv + 4 * nw == 32 ? 960 : 1024;

// ---------------------------------------------------------------------------
// FP64 pair loops (WF_FP64) on the gather kernel below: FP64 positions of the
// staged set in LDS, the neighbour fields from packed FP64 records.  Each
// thread sums its pairs in ascending staged order and the two threads of a
// particle add their partial sums, a fixed order, so results are
// deterministic.

// A: density rate drho_i = rho_i sum_j (m_j/rho_j) v_ij . (GK x_ij)
// (InteractionAlt.cu:166-246) [+ update rho_i + dt drho_i into rho_alt and
// the next {v, m/rho} record]
template <bool UH>
struct DensD {
  WF_GATHER64
  static constexpr int NBATCH = 4;
  struct Prm {
    int limit, n;
    double dt;
    int fuse;
    int mdj_alt;  // write m/rho into the next conduction record (fused with conduction)
    int skip;     // drho is overwritten unread (StepParams::keep): don't store it
  };
  struct Own {
    double x, y, z, vx, vy, vz, rho, m;
    HConst hc;
  };
  struct Nb {
    double4 v;  // v, m/rho
    double h;
  };
  __device__ static void drop(Nb& nb) { nb.v.w = 0.0; }
  struct Acc {
    double s;
  };
  __device__ static void merge(Acc& a, const Acc& b) {
    a.s += b.s;
  }
  __device__ static void init(const Fields& f, int i, bool act, Own& o, Acc& a, const Ctx&) {
    a.s = 0.0;
    if (!act) return;
    o.x = f.x[0][i]; o.y = f.x[1][i]; o.z = f.x[2][i];
    o.vx = f.v[0][i]; o.vy = f.v[1][i]; o.vz = f.v[2][i];
    o.rho = f.rho[i];
    o.m = f.m[i];  // of the update after the loop
    o.hc = hconst(f.h[i]);
  }
  __device__ static void load(const Fields& f, int j, Nb& nb) {
    nb.v = gat<double4>(f.kv, j);
    nb.h = UH ? 0.0 : gat<double>(f.h, j);
  }
#if WF_COLOAD64
  static constexpr bool CO = true;
  __device__ static void coload(const Fields& f, int j, int sub, Nb& nb) {
    uint4 c[2];
    coload_rec<2>(f.kv, j, sub, c);
    __builtin_memcpy(&nb.v, c, 32);
    nb.h = UH ? 0.0 : gat<double>(f.h, j);
  }
#endif
  // staged whole: {x, y}, {z, m/rho}, {v_x, v_y}, v_z
  WF_LDS64(3, 1)
  __device__ static void lds_put(const Fields& f, int j, const Ctx&, double2 (&q)[3],
                                 double (&r)[1]) {
    const double4 v = gat<double4>(f.kv, j);
    q[0] = make_double2(f.x[0][j], f.x[1][j]);
    q[1] = make_double2(f.x[2][j], v.w);
    q[2] = make_double2(v.x, v.y);
    r[0] = v.z;
  }
  __device__ static void lds_get(const double2 (&q)[3], const double (&r)[1], double& x, double& y,
                                 double& z, Nb& nb) {
    x = q[0].x;
    y = q[0].y;
    z = q[1].x;
    nb.v = make_double4(q[2].x, q[2].y, r[0], q[1].y);
  }
  __device__ static void pair(double x, double y, double z, const Nb& nb, const Own& o, Acc& a,
                              const Prm&) {
    const double xx = o.x - x, xy = o.y - y, xz = o.z - z;
    const double r2 = xx * xx + xy * xy + xz * xz;
    double rinv, h_;
    const double GK = gk_pair(r2, UH ? o.hc.h : nb.h, o.hc, rinv, h_);
    const double vx = o.vx - nb.v.x, vy = o.vy - nb.v.y, vz = o.vz - nb.v.z;
    a.s += nb.v.w * (GK * (vx * xx + vy * xy + vz * xz));
  }
  __device__ static void finish(const Fields& f, int i, bool act, const Own& o, const Acc& a,
                                const Prm& p) {
    if (act) {
      const double drho = o.rho * a.s;
      if (!p.skip) f.drho[i] = drho;
      if (p.fuse) {
        const double rn = o.rho + p.dt * drho;
        f.rho_alt[i] = rn;
        const double mdj = o.m / rn;
        f.kv_alt[i] = make_double4(o.vx, o.vy, o.vz, mdj);
        (p.mdj_alt ? f.tk64_alt : f.tk64)[i].z = mdj;  // m/rho for the conduction loop
      }
    } else if (p.fuse && i < p.n) {
      f.rho_alt[i] = f.rho[i];
      f.kv_alt[i] = f.kv[i];
    }
  }
};

struct NoDrop {};
template <class Nb>
struct DropMdj {
  __device__ static void drop(Nb& nb) { nb.v.w = 0.0; }
};

// Free-surface sums (Geometry.cu:26-88) taken along by the rates pass, which
// forms the same x_ij over the same lists at the same positions: the normal
// sum_j m x_ij (every particle's mass is m) and the neighbour count, with the
// flag decided as in the pass of its own (SurfD, SurfG).  Nothing between the
// rates pass and the reference's surface pass reads the flags or normals.  A
// second traversal of the lists took 157 us on a 2.74 M-particle friction-stir
// plate in mixed precision (63 us on a 1.32 M-particle cylinder); the sums add
// 38 us to the rates pass (8 us).
template <class T>
struct SurfPrm {
  int id_free_surf;
  double ntot, totmass;
  T r2cut;  // > 0: lists carry a skin; count only pairs within the radius
  T m;
};
// normal = n N/(M cnt); flag |normal| >= 0.25 h with at most 46 neighbours
__device__ __forceinline__ void surface_finish(const Fields& f, int i, double nx, double ny,
                                               double nz, int cnt, double ntot, double totmass,
                                               int id_free_surf) {
  const double sc = ntot / (totmass * (double)cnt);
  nx *= sc;
  ny *= sc;
  nz *= sc;
  f.nrm[0][i] = nx;
  f.nrm[1][i] = ny;
  f.nrm[2][i] = nz;
  if (sqrt(nx * nx + ny * ny + nz * nz) >= 0.25 * f.h[i] && cnt <= 46 && !f.idlock[i])
    f.ID[i] = id_free_surf;
}
template <bool SF>
struct SurfSums {
  __device__ __forceinline__ void surf_merge(const SurfSums&) {}
  template <class T>
  __device__ __forceinline__ void surf_add(T, T, T, T, const SurfPrm<T>&) {}
  template <class P>
  __device__ __forceinline__ void surf_finish(const Fields&, int, const P&) const {}
};
template <>
struct SurfSums<true> {
  double nx, ny, nz;
  int cnt;
  __device__ __forceinline__ void surf_merge(const SurfSums& b) {
    nx += b.nx;
    ny += b.ny;
    nz += b.nz;
    cnt += b.cnt;
  }
  // FP32 terms are rounded to FP32 and summed in FP64
  template <class T>
  __device__ __forceinline__ void surf_add(T dx, T dy, T dz, T r2, const SurfPrm<T>& p) {
    if (p.r2cut > (T)0 && !(r2 < p.r2cut)) return;
    const T tx = p.m * dx, ty = p.m * dy, tz = p.m * dz;
    nx += tx;
    ny += ty;
    nz += tz;
    cnt++;
  }
  template <class P>
  __device__ __forceinline__ void surf_finish(const Fields& f, int i, const P& p) const {
    surface_finish(f, i, nx, ny, nz, cnt, p.ntot, p.totmass, p.id_free_surf);
  }
};

// B: strain rate -1/2 sum (m_j/rho_j) GK (v_ij (x) x_ij + x_ij (x) v_ij) and
// rotation rate -1/2 sum (m_j/rho_j) GK (v_ij (x) x_ij - x_ij (x) v_ij),
// upper triangle, xz optionally negated (InteractionAlt.cu:262-383)
// SF: the free-surface sums of the same pairs as well (SurfSums)
template <bool UH, bool SF = false>
struct RatesD : std::conditional_t<SF, NoDrop, DropMdj<typename DensD<UH>::Nb>> {
  WF_GATHER64
  static constexpr int NBATCH = 4;
  struct Prm {
    int limit;
    double xz_sign;
    SurfPrm<double> sf;
  };
  struct Own {
    double x, y, z, vx, vy, vz;
    HConst hc;
  };
  typedef typename DensD<UH>::Nb Nb;
  WF_LDS64(3, 1)
  __device__ static void lds_put(const Fields& f, int j, const Ctx& c, double2 (&q)[3],
                                 double (&r)[1]) {
    DensD<UH>::lds_put(f, j, c, q, r);
  }
  __device__ static void lds_get(const double2 (&q)[3], const double (&r)[1], double& x, double& y,
                                 double& z, Nb& nb) {
    DensD<UH>::lds_get(q, r, x, y, z, nb);
  }
  struct Acc : SurfSums<SF> {
    double dxx, dyy, dzz, dxy, dyz, dxz, wxy, wyz, wxz;
  };
  __device__ static void merge(Acc& a, const Acc& b) {
    a.dxx += b.dxx; a.dyy += b.dyy; a.dzz += b.dzz;
    a.dxy += b.dxy; a.dyz += b.dyz; a.dxz += b.dxz;
    a.wxy += b.wxy; a.wyz += b.wyz; a.wxz += b.wxz;
    a.surf_merge(b);
  }
  __device__ static void init(const Fields& f, int i, bool act, Own& o, Acc& a, const Ctx&) {
    a = Acc{};
    if (!act) return;
    o.x = f.x[0][i]; o.y = f.x[1][i]; o.z = f.x[2][i];
    o.vx = f.v[0][i]; o.vy = f.v[1][i]; o.vz = f.v[2][i];
    o.hc = hconst(f.h[i]);
  }
  __device__ static void load(const Fields& f, int j, Nb& nb) { DensD<UH>::load(f, j, nb); }
  __device__ static void pair(double x, double y, double z, const Nb& nb, const Own& o, Acc& a,
                              const Prm& p) {
    const double xx = o.x - x, xy = o.y - y, xz = o.z - z;
    const double r2 = xx * xx + xy * xy + xz * xz;
    a.surf_add(xx, xy, xz, r2, p.sf);
    double rinv, h_;
    const double w = gk_pair(r2, UH ? o.hc.h : nb.h, o.hc, rinv, h_) * nb.v.w;
    const double vx = o.vx - nb.v.x, vy = o.vy - nb.v.y, vz = o.vz - nb.v.z;
    const double ax = w * vx, ay = w * vy, az = w * vz;
    a.dxx += ax * xx;
    a.dyy += ay * xy;
    a.dzz += az * xz;
    a.dxy += ax * xy + ay * xx;
    a.dyz += ay * xz + az * xy;
    a.dxz += ax * xz + az * xx;
    a.wxy += ax * xy - ay * xx;
    a.wyz += ay * xz - az * xy;
    a.wxz += ax * xz - az * xx;
  }
  __device__ static void finish(const Fields& f, int i, bool act, const Own&, const Acc& a,
                                const Prm& p) {
    if (!act) return;
    double v[9];
    rates9(a, p, v);
    put9(f, i, v);
    a.surf_finish(f, i, p.sf);
  }
  // the strain rate (xx yy zz xy yz xz) and the rotation rate (xy yz xz; its
  // diagonal stays 0) as they are stored
  typedef double RT;
  __device__ static void rates9(const Acc& a, const Prm& p, double (&v)[9]) {
    v[0] = -a.dxx; v[1] = -a.dyy; v[2] = -a.dzz;
    v[3] = -0.5 * a.dxy; v[4] = -0.5 * a.dyz; v[5] = -0.5 * a.dxz;
    v[6] = -0.5 * a.wxy; v[7] = -0.5 * a.wyz; v[8] = -0.5 * p.xz_sign * a.wxz;
  }
  __device__ static void put9(const Fields& f, int i, const double (&v)[9]) {
#pragma unroll
    for (int k = 0; k < 6; k++) f.strrate[k][i] = v[k];
#pragma unroll
    for (int k = 0; k < 3; k++) f.rotrate[3 + k][i] = v[6 + k];
  }
};

// D: a_i = sum_j m_j (sigma_i/rho_i^2 + sigma_j/rho_j^2 + Pi_ij I) . (GK x_ij),
// Pi_ij = (alpha C mu + beta mu^2)/rho_bar for approaching pairs,
// mu = h v.x/(r^2 + 0.01 h^2) (InteractionAlt.cu:18-150).  sigma_j/rho_j^2
// comes formed in the neighbour's record.
// neighbour records (96 B each) a lane holds in flight in the FP64 accel loop
#ifndef WF_ACCEL64_NBATCH
#define WF_ACCEL64_NBATCH 2
#endif
// BV: the beta (quadratic) viscosity term is on; UC: every particle has the
// same mass and sound speed (and h), so a pair reads neither; IT: each particle
// is integrated as soon as its sum is done (IntegratePrm)
template <bool UH, bool BV = false, bool UC = false, bool IT = false>
struct AccelD {
  WF_GATHER64
  static constexpr int NBATCH = WF_ACCEL64_NBATCH;
  struct Prm {
    int limit;
    double alpha, beta;
    StatsFold fold;  // the stress pass's statistics, folded by workgroup 0
    double m_uni, cs_uni;  // UC
    IntegratePrm ip;       // IT
  };
  struct NoIn {};
  struct Own {
    double x, y, z, vx, vy, vz, di, Ci, s0, s1, s2, s3, s4, s5;
    HConst hc;
    std::conditional_t<IT, IntegrateIn, NoIn> in;
  };
  struct Nb {
    double4 v, sa, sb;  // {v, m}, sigma/rho^2 xx yy zz xy, {yz, xz, rho, Cs}
    double h;
  };
#if WF_DROP_ACCEL64
  __device__ static void drop(Nb& nb) { nb.v.w = 0.0; }
#endif
  struct Acc {
    double ax, ay, az;
  };
  __device__ static void merge(Acc& a, const Acc& b) {
    a.ax += b.ax; a.ay += b.ay; a.az += b.az;
  }
  __device__ static void init(const Fields& f, int i, bool act, Own& o, Acc& a, const Ctx&) {
    a = Acc{0, 0, 0};
    if (!act) return;
    o.x = f.x[0][i]; o.y = f.x[1][i]; o.z = f.x[2][i];
    o.vx = f.v[0][i]; o.vy = f.v[1][i]; o.vz = f.v[2][i];
    o.di = f.rho[i]; o.Ci = f.Cs[i];
    o.hc = hconst(f.h[i]);
    if constexpr (IT) integrate_load<kRec64>(f, i, o.in);
    // its own record's sigma/rho^2 (the stress pass may not have stored sigma)
    if constexpr (UC) {
      const double4 sa = f.arec64u[i], sb = f.arec64[i];
      o.s0 = sa.x; o.s1 = sa.y; o.s2 = sb.x; o.s3 = sb.y; o.s4 = sb.z; o.s5 = sb.w;
    } else {
      const double4 sa = f.arec64[rec_at(f, i, 1)], sb = f.arec64[rec_at(f, i, 2)];
      o.s0 = sa.x; o.s1 = sa.y; o.s2 = sa.z; o.s3 = sa.w; o.s4 = sb.x; o.s5 = sb.y;
    }
  }
  __device__ static void load(const Fields& f, int j, Nb& nb) {
    nb.v = gat<double4, 96>(f.arec64, j);  // rec_at(f, j, 0..2)
    nb.sa = gat<double4, 96>(f.arec64, j, 32);
    nb.sb = gat<double4, 96>(f.arec64, j, 64);
    nb.h = UH ? 0.0 : gat<double>(f.h, j);
  }
#if WF_COLOAD64
  static constexpr bool CO = true;
  __device__ static void coload(const Fields& f, int j, int sub, Nb& nb) {
    uint4 c[6];
    coload_rec<6>(f.arec64, j, sub, c);
    __builtin_memcpy(&nb.v, &c[0], 32);
    __builtin_memcpy(&nb.sa, &c[2], 32);
    __builtin_memcpy(&nb.sb, &c[4], 32);
    nb.h = UH ? 0.0 : gat<double>(f.h, j);
  }
#endif
  // UC: in LDS {x, y}, {z, rho}, {v_x, v_y}, {v_z, s_xx}, s_yy with s =
  // sigma/rho^2; gathered {s_zz, s_xy, s_yz, s_xz}
  WF_LDS64(4, 1)
  typedef double4 Rest;
  __device__ static const void* rest(const Fields& f) { return f.arec64; }
  __device__ static void lds_put(const Fields& f, int j, const Ctx&, double2 (&q)[4],
                                 double (&r)[1]) {
    const double4 v = gat<double4>(f.kv, j), s = gat<double4>(f.arec64u, j);
    q[0] = make_double2(f.x[0][j], f.x[1][j]);
    q[1] = make_double2(f.x[2][j], s.z);
    q[2] = make_double2(v.x, v.y);
    q[3] = make_double2(v.z, s.x);
    r[0] = s.y;
  }
  __device__ static void lds_get(const double2 (&q)[4], const double (&r)[1], double& x, double& y,
                                 double& z, Nb& nb) {
    x = q[0].x;
    y = q[0].y;
    z = q[1].x;
    nb.v = make_double4(q[2].x, q[2].y, q[3].x, 0.0);
    nb.sa.x = q[3].y;
    nb.sa.y = r[0];
    nb.sb.z = q[1].y;
  }
  __device__ static void rest_get(const Rest& s, Nb& nb) {
    nb.sa.z = s.x;
    nb.sa.w = s.y;
    nb.sb.x = s.z;
    nb.sb.y = s.w;
  }
  __device__ static void pair(double x, double y, double z, const Nb& nb, const Own& o, Acc& a,
                              const Prm& p) {
    const double xx = o.x - x, xy = o.y - y, xz = o.z - z;
    const double r2 = xx * xx + xy * xy + xz * xz;
    double rinv, h_;
    const double GK = gk_pair(r2, UH ? o.hc.h : nb.h, o.hc, rinv, h_);
    const double vx = o.vx - nb.v.x, vy = o.vy - nb.v.y, vz = o.vz - nb.v.z;
    const double vdx = vx * xx + vy * xy + vz * xz;
    // Monaghan viscosity on approaching pairs only: (alpha C mu + beta mu^2)
    // / rho_bar with mu = h v/e, v = min(v_ij.x_ij, 0), e = r^2 + 0.01 h^2,
    // as 2 h v (alpha C + beta mu) / (e (rho_i + rho_j)): one refined
    // reciprocal and no branch (receding pairs get v = 0)
    const double vn = fmin(vdx, 0.0);
    const double rs = o.di + nb.sb.z;
    const double inv = rcp_f64((r2 + 0.01 * h_ * h_) * rs);
    const double Cj = UC ? p.cs_uni : nb.sb.w;
    double PI;
    if constexpr (BV) {
      const double coef = (0.5 * p.alpha) * (o.Ci + Cj) + p.beta * (h_ * vn * rs * inv);
      PI = 2.0 * h_ * vn * coef * inv;
    } else {
      PI = vn * ((h_ * p.alpha) * (o.Ci + Cj)) * inv;
    }
    const double g = GK * (UC ? p.m_uni : nb.v.w);
    const double gx = g * xx, gy = g * xy, gz = g * xz;
    const double mxx = o.s0 + nb.sa.x + PI, myy = o.s1 + nb.sa.y + PI;
    const double mzz = o.s2 + nb.sa.z + PI;
    const double mxy = o.s3 + nb.sa.w, myz = o.s4 + nb.sb.x, mxz = o.s5 + nb.sb.y;
    if constexpr (UC && !BV) {
      // the order of the general loop's contraction, so that a record layout
      // does not change the sums
      a.ax += __builtin_fma(mxz, gz, __builtin_fma(mxy, gy, mxx * gx));
      a.ay += __builtin_fma(myz, gz, __builtin_fma(mxy, gx, myy * gy));
      a.az += __builtin_fma(mzz, gz, __builtin_fma(myz, gy, mxz * gx));
    } else {
      a.ax += mxx * gx + mxy * gy + mxz * gz;
      a.ay += mxy * gx + myy * gy + myz * gz;
      a.az += mxz * gx + myz * gy + mzz * gz;
    }
  }
  __device__ static void finish(const Fields& f, int i, bool act, const Own& o, const Acc& a,
                                const Prm& p) {
    if (!act) return;
    if constexpr (IT) {
      if (!p.ip.contacts || p.ip.contacts[i] == 0) {
        integrate_apply<kRec64>(f, i, a.ax, a.ay, a.az, p.ip.dt, p.ip.bc, p.ip.fr, p.ip.out,
                                o.in);
        return;
      }
    }
    f.a[0][i] = a.ax;
    f.a[1][i] = a.ay;
    f.a[2][i] = a.az;
  }
};

// What a conduction pass reads of its own particle after the pair loop, read
// before it so that the loads are in flight while the pairs are summed
struct CondIn {
  double rho, cp, qp, qf, ta;
  int bct;
  __device__ __forceinline__ void load(const Fields& f, int i) {
    rho = f.rho[i];
    cp = f.cp[i];
    qp = f.qpl[i];
    qf = f.qfric[i];
    ta = f.Ta[i];
    bct = f.BC_T[i];
  }
};
// dT_i/dt from the conduction sum q: convection (Thermal.cu:36-64), plastic
// and friction heat, fixed temperature
template <class P>
__device__ __forceinline__ double cond_rate(const Fields& f, int i, double q, double Ti,
                                            const P& p, const CondIn& in) {
  double acc = q * (1. / (in.rho * in.cp));
  if (in.bct == WF_BCT_CONVECTION) {
    const double mi = f.m[i];
    const double dS2 = pow(mi / in.rho, 0.666666666);
    const double q_conv = p.h_conv * dS2 * (p.T_inf - Ti) / mi;
    acc += 1. / in.cp * q_conv;
  }
  if (in.qp != 0.0) acc += in.qp * (1. / (in.rho * in.cp));
  if (in.qf != 0.0) acc += in.qf / (f.m[i] * in.cp);
  return in.bct == WF_BCT_FIXED ? 0.0 : acc;
}

// G: conduction dT_i/dt = 1/(rho_i cp_i) sum_j (m_j/rho_j) 4 k_i k_j/(k_i+k_j)
// (T_i - T_j) GK  (Thermal.cu:101-142, where x_ij.(GK x_ij)/r^2 = GK), then
// convection (Thermal.cu:36-64), plastic-work source and FIXED BC; optional
// fused leapfrog (Thermal.cu:16-31) writing T into T_alt and the next record.
template <bool UH>
struct CondD {
  WF_GATHER64
  static constexpr int NBATCH = 4;
  struct Prm {
    int limit;
    double T_inf, h_conv, dt;
    int leap, first;
    int skip;  // dT/dt and T_b are overwritten unread (StepParams::keep)
  };
  struct Own {
    double x, y, z, k, T, mdj;
    HConst hc;
    CondIn in;
  };
  struct Nb {
    double4 tk;  // T, k, m/rho
    double h;
  };
  __device__ static void drop(Nb& nb) { nb.tk.z = 0.0; }
  struct Acc {
    double q;
  };
  __device__ static void merge(Acc& a, const Acc& b) {
    a.q += b.q;
  }
  __device__ static void init(const Fields& f, int i, bool act, Own& o, Acc& a, const Ctx&) {
    a.q = 0.0;
    if (!act) return;
    o.x = f.x[0][i]; o.y = f.x[1][i]; o.z = f.x[2][i];
    o.k = f.k[i]; o.T = f.T[i];
    o.mdj = f.tk64[i].z;
    o.hc = hconst(f.h[i]);
    o.in.load(f, i);
  }
  __device__ static void load(const Fields& f, int j, Nb& nb) {
    nb.tk = gat<double4>(f.tk64, j);
    nb.h = UH ? 0.0 : gat<double>(f.h, j);
  }
#if WF_COLOAD64
  static constexpr bool CO = true;
  __device__ static void coload(const Fields& f, int j, int sub, Nb& nb) {
    uint4 c[2];
    coload_rec<2>(f.tk64, j, sub, c);
    __builtin_memcpy(&nb.tk, c, 32);
    nb.h = UH ? 0.0 : gat<double>(f.h, j);
  }
#endif
  // staged whole: {x, y}, {z, m/rho}, {T, k}
  WF_LDS64(3, 0)
  __device__ static void lds_put(const Fields& f, int j, const Ctx&, double2 (&q)[3],
                                 double (&)[1]) {
    const double4 tk = gat<double4>(f.tk64, j);
    q[0] = make_double2(f.x[0][j], f.x[1][j]);
    q[1] = make_double2(f.x[2][j], tk.z);
    q[2] = make_double2(tk.x, tk.y);
  }
  __device__ static void lds_get(const double2 (&q)[3], const double (&)[1], double& x, double& y,
                                 double& z, Nb& nb) {
    x = q[0].x;
    y = q[0].y;
    z = q[1].x;
    nb.tk = make_double4(q[2].x, q[2].y, q[1].y, 0.0);
  }
  __device__ static void pair(double x, double y, double z, const Nb& nb, const Own& o, Acc& a,
                              const Prm&) {
    const double xx = o.x - x, xy = o.y - y, xz = o.z - z;
    const double r2 = xx * xx + xy * xy + xz * xz;
    double rinv, h_;
    const double GK = gk_pair(r2, UH ? o.hc.h : nb.h, o.hc, rinv, h_);
    const double kj = nb.tk.y;
    double kh = 2.0 * o.k;  // equal conductivities need no division
    if (__builtin_expect(kj != o.k, 0)) kh = 4.0 * o.k * kj / (o.k + kj);
    a.q += nb.tk.z * kh * (o.T - nb.tk.x) * GK;
  }
  __device__ static void finish(const Fields& f, int i, bool act, const Own& o, const Acc& a,
                                const Prm& p) {
    if (!act) return;
    const double acc = cond_rate(f, i, a.q, o.T, p, o.in);
    if (!p.skip) f.dTdt[i] = acc;
    if (p.leap) {
      double Tn;
      if (p.first) {
        f.Ta[i] = o.T - p.dt / 2.0 * acc;
        Tn = o.T;
      } else {
        const double ta = o.in.ta;
        if (!p.skip) f.Tb[i] = ta;
        double tan = ta + acc * p.dt;
        f.Ta[i] = tan;
        Tn = (tan + ta) / 2.;
      }
      f.T_alt[i] = Tn;
      f.tk64_alt[i] = make_double4(Tn, o.k, o.mdj, 0.0);
    }
  }
};

// ===========================================================================
// Mixed precision (WF_MIXED): the same pair physics in FP32, on FP32 mirrors,
// with coordinates relative to the tile's base cell (x = xr + (c - c_tile) cs,
// c an integer grid cell), FP32 pair terms summed in FP64, and FP64 results.
// Per-particle terms stay FP64.
//
// The FP32 loops hold only the staged set's tile-frame positions in LDS
// (kStage32 particles, normally the whole set) and gather the other
// neighbour fields from packed per-particle float4/float2 mirrors, which stay
// in L1/L2 because the staged set is spatially compact.  A thread therefore
// walks its whole neighbour list without waiting at chunk boundaries for the
// busiest lane of its wavefront (with chunks of a few hundred staged
// particles a wavefront keeps only ~40-55 % of its lanes busy).

// sum of FP32 pair terms kept in FP64: with packed FP32 off, an FP64 add
// issues at the FP32 rate on gfx950, so widening each term costs two
// operations where compensated (Kahan) FP32 summation costs four, and the
// sum carries no rounding beyond the terms' own
struct KSum {
  double s;
  __device__ __forceinline__ void zero() { s = 0.0; }
  __device__ __forceinline__ void add(float y) { s += (double)y; }
  __device__ __forceinline__ void add(const KSum& o) { s += o.s; }
  __device__ __forceinline__ double val() const { return s; }
};

struct HConstF {
  float h, inv_h, C3;  // h, 1/h, 3/(pi h^4)
};
__device__ __forceinline__ HConstF hconst_f(float h) {
  const float hh = h * h;
  return HConstF{h, __builtin_amdgcn_rcpf(h), 3.f * __builtin_amdgcn_rcpf(hh * hh * (float)kPi)};
}
// FP32 cubic-spline gradient (1/r) dW/dr from r^2 (Functions.cu:76-88), the
// branch-free form of gk_pair; UH: every particle has the same h, so h_j = h_i
template <bool UH>
__device__ __forceinline__ float gk_pair_f(float r2, float hj, const HConstF& hc, float& h_) {
  const float rinv = __builtin_amdgcn_rsqf(fmaxf(r2, 1e-30f));
  const float rij = r2 * rinv;
  float inv_h = hc.inv_h, C3 = hc.C3;
  h_ = hc.h;
  if (!UH && hj != hc.h) {
    h_ = 0.5f * (hc.h + hj);
    inv_h = __builtin_amdgcn_rcpf(h_);
    C3 = 3.f * __builtin_amdgcn_rcpf(h_ * h_ * h_ * h_ * (float)kPi);
  }
  const float q = rij * inv_h;
  const float u = clamp01f(1.f - q), t = clamp01f(1.f - 0.5f * q);
  return C3 * rinv * ((u - t) * (u + t));
}

struct Ctx32 {
  int bx, by, bz;
  float cs;
};
__device__ __forceinline__ Ctx32 ctx32(const Fields& f, int t, float cs) {
  int bx, by, bz;
  unpack_cell(__float_as_int(f.p4[t * kTileP].w), bx, by, bz);
  return Ctx32{bx, by, bz, cs};
}
// position of particle j in the tile frame
__device__ __forceinline__ void pos32(const Fields& f, int j, const Ctx32& c, float& x, float& y,
                                      float& z) {
  int cx, cy, cz;
  const float4 p = gat<float4>(f.p4, j);
  unpack_cell(__float_as_int(p.w), cx, cy, cz);
  x = p.x + (float)(cx - c.bx) * c.cs;
  y = p.y + (float)(cy - c.by) * c.cs;
  z = p.z + (float)(cz - c.bz) * c.cs;
}

// staged slots per LDS pass: 1024 x 16 B (tile-frame position + index) =
// 16 KB (768 slots send the larger tiles to the chunked path: 17 % slower)
#ifndef WF_STAGE32
#define WF_STAGE32 1024
#endif
constexpr int kStage32 = WF_STAGE32;
#define WF_GATHER32                                                                \
  typedef float PT;                                                                \
  static constexpr int STAGE = kStage32;                                           \
  static constexpr int LANES = WF_LANES32;                                         \
  typedef Ctx32 Ctx;                                                               \
  template <class P>                                                               \
  __device__ static Ctx ctx(const Fields& f, int t, const P& p) {                  \
    return ctx32(f, t, p.cs);                                                      \
  }                                                                                \
  __device__ static void pos(const Fields& f, int j, const Ctx& c, float& x, float& y, \
                             float& z) {                                           \
    pos32(f, j, c, x, y, z);                                                       \
  }

// One staged particle in LDS: its position in the tile frame and its
// particle index, read together by one LDS access per pair (the index
// addresses the neighbour's packed record in global memory).
template <class PT>
struct alignas(16) StagedSlot;
template <>
struct alignas(16) StagedSlot<float> {
  float x, y, z;
  int j;
};
template <>
struct alignas(16) StagedSlot<double> {
  double x, y, z;
  int j, pad;
};

// A pair functor may stage one more 16-byte value per staged particle in LDS
// beside its position (typedef Extra, Extra extra(f, j) reads it when the set
// is staged, put(nb, e) hands it to the neighbour record): a field every pair
// needs then costs an LDS read instead of a global gather per pair.
template <class K, class = void>
struct ExtraOf {
  static constexpr bool on = false;
  typedef int type;
};
template <class K>
struct ExtraOf<K, std::void_t<typename K::Extra>> {
  static constexpr bool on = true;
  typedef typename K::Extra type;
};

// A pair functor may sum a batch's pair terms in a narrower partial sum
// (typedef Part, pzero(part), flush(acc, part)): pair() then adds into the
// partial, which is added to the functor's sums once per batch of up to
// NBATCH pairs.  Without a Part, pair() adds into the sums directly.
template <class K, class = void>
struct PartOf {
  static constexpr bool on = false;
};
template <class K>
struct PartOf<K, std::void_t<typename K::Part>> {
  static constexpr bool on = true;
};

// A pair functor whose every term scales with one neighbour weight (m_j or
// m_j/rho_j) may say how to zero it (drop(nb)): the batch then evaluates
// all of its pairs in straight-line code, entries past the list with a zero
// weight (adding exact zeros), so that the compiler keeps every record load
// ahead of the first pair and each pair waits only for its own record.
template <class K, class = void>
struct DropOf {
  static constexpr bool on = false;
};
template <class K>
struct DropOf<K, std::void_t<decltype(K::drop(std::declval<typename K::Nb&>()))>> {
  static constexpr bool on = true;
};

// waves per SIMD a pair functor asks the register allocator to leave room
// for (MIN_WAVES; 1 = no request)
template <class K, class = void>
struct WavesOf {
  static constexpr int value = 1;
};
template <class K>
struct WavesOf<K, std::void_t<decltype(K::MIN_WAVES)>> {
  static constexpr int value = K::MIN_WAVES;
};

// the value v holds in lane (this lane ^ M), M = 1, 2, 4 or 8, where the M
// lanes of an aligned group hold the same value (a butterfly's steps): by DPP,
// so that no trip through the LDS pipe is waited for.  quad_perm [1, 0, 3, 2]
// and [2, 3, 0, 1], row_half_mirror (lane 7 - i of 8), row_mirror (15 - i)
template <int M, class T>
__device__ __forceinline__ T lane_value_xor(const T& v) {
  static_assert(sizeof(T) % 4 == 0, "whole 32-bit words");
  static_assert(M == 1 || M == 2 || M == 4 || M == 8, "within a row of 16 lanes");
  constexpr int CTRL = M == 1 ? 0xB1 : M == 2 ? 0x4E : M == 4 ? 0x141 : 0x140;
  constexpr int W = sizeof(T) / 4;
  int in[W], out[W];
  __builtin_memcpy(in, &v, sizeof(T));
#pragma unroll
  for (int w = 0; w < W; w++)
    out[w] = __builtin_amdgcn_update_dpp(0, in[w], CTRL, 0xF, 0xF, false);
  T r;
  __builtin_memcpy(&r, out, sizeof(T));
  return r;
}
// the sums of a particle's L lanes merged, in every one of them
template <class K, int L, int M = 1>
__device__ __forceinline__ void merge_lanes(typename K::Acc& acc) {
  if constexpr (M < L) {
    const typename K::Acc other = lane_value_xor<M>(acc);
    K::merge(acc, other);
    merge_lanes<K, L, 2 * M>(acc);
  }
}

// A pair functor may load its neighbour records cooperatively (static
// constexpr bool CO = true, coload(f, j, sub, nb)); with two lanes per
// particle both lanes then run the same iterations of the list walk.
template <class K, class = void>
struct CoOf {
  static constexpr bool on = false;
};
template <class K>
struct CoOf<K, std::void_t<decltype(K::CO)>> {
  static constexpr bool on = K::CO;
};

// A pass whose Prm has a StatsFold (fold) folds the preceding stress pass's
// block statistics in its first workgroup, after that workgroup's tile, so
// that the fold overlaps the other workgroups instead of taking a launch.
template <class K, class = void>
struct FoldOf {
  static constexpr bool on = false;
};
template <class K>
struct FoldOf<K, std::void_t<decltype(std::declval<typename K::Prm&>().fold)>> {
  static constexpr bool on = true;
};

// One workgroup per tile, L = K::LANES consecutive lanes per particle: lanes
// L p .. L p + L - 1 all hold particle p and deal its slot list out by quads
// (lane L p + h takes the quads q with q % L == h); their sums are merged
// (butterfly over the L lanes) before lane L p writes the result.
template <class K>
__global__ __launch_bounds__(4 * kTileP) __attribute__((amdgpu_waves_per_eu(WavesOf<K>::value)))
void k_pair_gather(Fields f, TileLists tl, typename K::Prm prm) {
  constexpr int ST = K::STAGE;
  constexpr int L = K::LANES;
  static_assert(L == 1 || L == 2 || L == 4, "1, 2 or 4 lanes per particle");
  constexpr int NT = L * kTileP;  // threads per tile
  typedef StagedSlot<typename K::PT> Slot;
  __shared__ Slot st[ST];
  constexpr bool XS = ExtraOf<K>::on;
  typedef typename ExtraOf<K>::type XT;
  __shared__ XT sx[XS ? ST : 1];
  const int t = xcd_tile(blockIdx.x, gridDim.x);
  const int tid = threadIdx.x;
  const int sub = tid & (L - 1);
  const int i = t * kTileP + tid / L;
  const bool act = i < prm.limit;
  const typename K::Ctx cx = K::ctx(f, t, prm);
  typename K::Own own;
  typename K::Acc acc;
  K::init(f, i, act, own, acc, cx);
  const int ub = tl.uoff[t], ucnt = tl.ucnt[t];
  const int* __restrict__ tj = tl.tj + ub;
  const int cnt = act ? tl.count[i] : 0;
#ifndef WF_STAGE_UNROLL
#define WF_STAGE_UNROLL 8
#endif
  // staging: SU slots per thread at a time, their indices, then their
  // positions, then the LDS writes, so that each thread keeps SU index loads
  // and then SU position loads in flight instead of one dependent pair
  auto stage = [&](int c0, int m) {
    constexpr int SU = WF_STAGE_UNROLL;
    for (int s0 = tid; s0 < m; s0 += SU * NT) {
      int jj[SU];
#pragma unroll
      for (int u = 0; u < SU; u++) {
        const int s = s0 + u * NT;
        jj[u] = s < m ? tj[c0 + s] : 0;
      }
      typename K::PT x[SU], y[SU], z[SU];
#pragma unroll
      for (int u = 0; u < SU; u++)
        if (s0 + u * NT < m) K::pos(f, jj[u], cx, x[u], y[u], z[u]);
      XT e[XS ? SU : 1];
      if constexpr (XS) {
#pragma unroll
        for (int u = 0; u < SU; u++)
          if (s0 + u * NT < m) e[u] = K::extra(f, jj[u]);
      }
#pragma unroll
      for (int u = 0; u < SU; u++) {
        const int s = s0 + u * NT;
        if (s < m) {
          Slot v;
          v.x = x[u];
          v.y = y[u];
          v.z = z[u];
          v.j = jj[u];
          st[s] = v;
          if constexpr (XS) sx[s] = e[u];
        }
      }
    }
  };
  constexpr int NB = K::NBATCH;  // neighbour records held at once (4, or 2)
  if (ucnt <= ST) {
    // the whole staged set fits: one pass, a quad of four slots at a time;
    // the lane's slot word two quads ahead is fetched while the current
    // quad's records are in flight, and the next quad's particle indices
    // come from LDS
    stage(0, ucnt);
    __syncthreads();
    // lanes past the padded particle range read row 0 of the last particle
    // (their lists are empty); every slot word is loaded unconditionally
    // from a row clamped into the list, since a select between a load and a
    // constant turns into a load through a selected pointer with the
    // constant in scratch
    const uint2* __restrict__ q = tl.slotq + min((int64_t)i, tl.npad - 1);
    const int klast = max(cnt - 1, 0);
    // 32-bit word index: rows x npad stays below 2^32 (kMaxParticles)
    const unsigned np = (unsigned)tl.npad;
    auto word = [&](int k) { return q[(unsigned)(min(k, klast) >> 2) * np]; };
    auto sl_of = [](const uint2 w, int u) {
      const unsigned h = (u & 2) ? w.y : w.x;
      return (int)((u & 1) ? h >> 16 : h & 0xFFFFu);
    };
    constexpr int KS = 4 * L;  // slots from one of the lane's quads to its next
    const int k0 = 4 * sub;
    // with cooperative loads both lanes of a particle take the same number
    // of steps (a lane past its list loads for its partner and adds nothing)
    constexpr bool CO = CoOf<K>::on && L == 2;
    const int kend = CO ? (cnt + KS - 1) / KS * KS + k0 : cnt;
    uint2 w0 = word(k0);
    uint2 w1 = word(k0 + KS);
    int jn[4];
#pragma unroll
    for (int u = 0; u < 4; u++) jn[u] = k0 < cnt ? st[sl_of(w0, u)].j : 0;
    for (int k = k0; k < kend; k += KS) {
      const int nk = min(4, cnt - k);
      int jc[4];
#pragma unroll
      for (int u = 0; u < 4; u++) jc[u] = jn[u];
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (k + KS + u < cnt) jn[u] = st[sl_of(w1, u)].j;
      const uint2 w2 = word(k + 2 * KS);
#pragma unroll
      for (int u0 = 0; u0 < 4; u0 += NB) {
        // with straight-line batches (drop()) every record of the batch is
        // loaded, also for entries past the list: they repeat one of it
        // (TileLists, or the index an earlier entry held), and each pair waits
        // only for its own record;
        // otherwise only the list's entries are loaded (the FP64
        // acceleration loop is bound by its gathers)
        typename K::Nb nb[NB];
#pragma unroll
        for (int u = 0; u < NB; u++) {
          if constexpr (CO) K::coload(f, jc[u0 + u], sub, nb[u]);
          else if (DropOf<K>::on || u0 + u == 0 || u0 + u < nk) K::load(f, jc[u0 + u], nb[u]);
        }
        // the batch's staged positions are read before any pair is evaluated
        // (entries past the list repeat one of it)
        typename K::PT px[NB], py[NB], pz[NB];
        int sl[NB];
#pragma unroll
        for (int u = 0; u < NB; u++) {
          sl[u] = sl_of(w0, u0 + u);
          const Slot& sv = st[sl[u]];
          px[u] = sv.x;
          py[u] = sv.y;
          pz[u] = sv.z;
        }
        // a staged extra value is read just before its pair
        auto batch = [&](auto& sum) {
#pragma unroll
          for (int u = 0; u < NB; u++) {
            if constexpr (DropOf<K>::on) {
              if constexpr (XS) K::put(nb[u], sx[sl[u]]);
              if (u0 + u >= nk) K::drop(nb[u]);
              K::pair(px[u], py[u], pz[u], nb[u], own, sum, prm);
            } else if ((!CO && u0 + u == 0) || u0 + u < nk) {
              // (the quad's first entry is in the list unless the lane only
              // loads for its partner: k < cnt)
              if constexpr (XS) K::put(nb[u], sx[sl[u]]);
              K::pair(px[u], py[u], pz[u], nb[u], own, sum, prm);
            }
          }
        };
        if constexpr (PartOf<K>::on) {
          typename K::Part part;
          K::pzero(part);
          batch(part);
          K::flush(acc, part);
        } else {
          batch(acc);
        }
      }
      w0 = w1;
      w1 = w2;
    }
  } else {
    SlotReader sr;
    sr.init(tl, i, cnt);
    // this lane's slots: those of the quads q with q % L == sub
    auto mine = [&]() { return ((sr.k >> 2) & (L - 1)) == sub; };
    for (int c0 = 0; c0 < ucnt; c0 += ST) {
      const int m = min(ST, ucnt - c0);
      __syncthreads();
      stage(c0, m);
      __syncthreads();
      const int lim = c0 + m;
      // two neighbours per iteration while both fall in this pass: their
      // gathers are issued before either pair is evaluated
      while (sr.k < sr.cnt) {
        if (!mine()) {
          sr.skip_quad();
          continue;
        }
        const int s0 = sr.slot();
        if (s0 >= lim) break;
        sr.advance();
        const Slot& a0 = st[s0 - c0];
        typename K::Nb a;
        K::load(f, a0.j, a);
        if constexpr (XS) K::put(a, sx[s0 - c0]);
        // one or two pairs, summed like a batch of the one-pass loop
        auto eval = [&](auto&& body) {
          if constexpr (PartOf<K>::on) {
            typename K::Part part;
            K::pzero(part);
            body(part);
            K::flush(acc, part);
          } else {
            body(acc);
          }
        };
        if (sr.k < sr.cnt && mine()) {
          const int s1 = sr.slot();
          if (s1 < lim) {
            sr.advance();
            const Slot& b0 = st[s1 - c0];
            typename K::Nb b;
            K::load(f, b0.j, b);
            if constexpr (XS) K::put(b, sx[s1 - c0]);
            eval([&](auto& sum) {
              K::pair(a0.x, a0.y, a0.z, a, own, sum, prm);
              K::pair(b0.x, b0.y, b0.z, b, own, sum, prm);
            });
            continue;
          }
        }
        eval([&](auto& sum) { K::pair(a0.x, a0.y, a0.z, a, own, sum, prm); });
      }
    }
  }
  merge_lanes<K, L>(acc);
  if (sub == 0) K::finish(f, i, act, own, acc, prm);
  if constexpr (FoldOf<K>::on) {
    if (blockIdx.x == 0 && prm.fold.nb > 0) {
      __syncthreads();  // the staged set is read no more: its LDS is scratch
      block_fold_stats(prm.fold, reinterpret_cast<unsigned long long*>(st));
    }
  }
}


// ---------------------------------------------------------------------------
// The pair loops with the neighbours staged whole: everything a pair reads of
// its neighbour is in LDS, each 16-byte (and one 8- or 4-byte) entry in an
// array of its own, so a pair costs LDS reads only.  A gather of a record per
// pair costs the CU's address unit 30-40 cycles per 64 lanes and 16 bytes
// where an LDS read costs 8-20, and every particle of a tile's set is read
// once instead of once per pair that has it (about ten times).  The set is
// LDS-limited (ST entries): two workgroups a CU in the FP64 conduction +
// density and acceleration loops, three in the others, which measured more
// than the four and more of the gathering kernel.  Measured on a 759k-particle
// cylinder (ms, gathering -> staged whole): FP64 conduction + density 0.227
// -> 0.142, rates 0.123 -> 0.115, acceleration 0.266 -> 0.223, density 0.121
// -> 0.104; mixed acceleration + integration 0.158 -> 0.136, conduction +
// density 0.106 -> 0.093, rates 0.061 -> 0.057.  Tiles of 64 particles (four
// workgroups a CU, but a third more staging) were slower: FP64 step 0.66 ms
// against 0.59.
//
// A policy whose entry would not leave two workgroups a CU keeps the rest of
// it in a record of its own (typedef Rest, rest(f) the array, rest_get(rest,
// nb)), which the lane pairs gather together (coload_rec): the FP64
// acceleration stages 72 of its 104 bytes.  All of it in LDS (one workgroup a
// CU) took 0.264 ms.
//
// The lanes and their sums are those of k_pair_gather; P of the tile's
// kTileP particles make a workgroup.
template <class K, class = void>
struct HasLds {
  static constexpr bool on = false;
};
template <class K>
struct HasLds<K, std::void_t<typename K::LV>> {
  static constexpr bool on = true;
};
template <class K, class = void>
struct RestOf {
  static constexpr bool on = false;
  typedef int type;
};
template <class K>
struct RestOf<K, std::void_t<typename K::Rest>> {
  static constexpr bool on = true;
  typedef typename K::Rest type;
};
// A policy may finish its particles with whole wavefronts, a thread a particle
// (static constexpr bool TAIL = true): the sums then go through LDS, where the
// staged set was (tail_put, by the lane that has them), and tail() runs in
// every thread of the workgroup, the first P with a particle each.
// What tail() reads of its particle may be loaded ahead of the pair loop
// (static constexpr bool PRE = true; Pre, pre()).
template <class K, class = void>
struct TailOf {
  static constexpr bool on = false, pre = false;
  typedef int type;
};
template <class K>
struct TailOf<K, std::void_t<decltype(K::TAIL)>> {
  static constexpr bool on = true, pre = K::PRE;
  typedef typename K::Pre type;
};
template <class K, int L, int P, int ST>
__global__ __launch_bounds__(L * P) __attribute__((amdgpu_waves_per_eu(WavesOf<K>::value)))
void k_pair_lds(Fields f, TileLists tl, typename K::Prm prm) {
  constexpr int S = kTileP / P, NT = L * P;
  static_assert(L >= 2 && L <= 16 && (L & (L - 1)) == 0, "a power of two of lanes per particle");
  typedef typename K::LV LV;
  typedef typename K::LW LW;
  typedef typename K::PT PT;
  constexpr int NV = K::NV, NW = K::NW;
  constexpr bool R = RestOf<K>::on;
  typedef typename RestOf<K>::type Rest;
  __shared__ LV sv[NV][ST];
  __shared__ LW sw[NW > 0 ? ST : 1];
  __shared__ int sj[R ? ST : 1];
  const int b = xcd_tile(blockIdx.x, gridDim.x);
  const int t = b / S;
  const int tid = threadIdx.x;
  const int sub = tid & (L - 1);
  const int i = b * P + tid / L;
  const bool act = i < prm.limit;
  const int ub = tl.uoff[t], ucnt = tl.ucnt[t];
  const int* __restrict__ tj = tl.tj + ub;
  const int cnt = act ? tl.count[i] : 0;
  const typename K::Ctx cx = K::ctx(f, t, prm);
  typename K::Own own;
  typename K::Acc acc;
  K::init(f, i, act, own, acc, cx);
  typename TailOf<K>::type pre;
  if constexpr (TailOf<K>::pre)
    if (tid < P && b * P + tid < prm.limit) K::pre(f, prm, b * P + tid, pre);
  // SU neighbours per thread at a time: their indices, then everything the
  // pairs read of them, then the LDS writes
  auto stage = [&](int c0, int m) {
    constexpr int SU = 4;
    for (int s0 = tid; s0 < m; s0 += SU * NT) {
      int jj[SU];
#pragma unroll
      for (int u = 0; u < SU; u++) jj[u] = s0 + u * NT < m ? tj[c0 + s0 + u * NT] : 0;
      LV q[SU][NV];
      LW r[SU][1];
#pragma unroll
      for (int u = 0; u < SU; u++) K::lds_put(f, jj[u], cx, q[u], r[u]);
#pragma unroll
      for (int u = 0; u < SU; u++) {
        const int s = s0 + u * NT;
        if (s < m) {
#pragma unroll
          for (int v = 0; v < NV; v++) sv[v][s] = q[u][v];
          if constexpr (NW > 0) sw[s] = r[u][0];
          if constexpr (R) sj[s] = jj[u];
        }
      }
    }
  };
  auto fetch = [&](int sl, PT& x, PT& y, PT& z, typename K::Nb& nb) {
    LV q[NV];
    LW r[1] = {};
#pragma unroll
    for (int v = 0; v < NV; v++) q[v] = sv[v][sl];
    if constexpr (NW > 0) r[0] = sw[sl];
    K::lds_get(q, r, x, y, z, nb);
  };
  // body(sum) adds the pairs of a quad, through the policy's partial sums if
  // it has them
  auto quad = [&](auto&& body) {
    if constexpr (PartOf<K>::on) {
      typename K::Part part;
      K::pzero(part);
      body(part);
      K::flush(acc, part);
    } else {
      body(acc);
    }
  };
  if (ucnt <= ST) {
    stage(0, ucnt);
    __syncthreads();
    // lanes past the padded particle range read row 0 of the last particle
    // (their lists are empty); rows are clamped into the list
    const uint2* __restrict__ q = tl.slotq + min((int64_t)i, tl.npad - 1);
    const int klast = max(cnt - 1, 0);
    // 32-bit word index: rows x npad stays below 2^32 (kMaxParticles)
    const unsigned np = (unsigned)tl.npad;
    auto word = [&](int k) { return q[(unsigned)(min(k, klast) >> 2) * np]; };
    auto sl_of = [](const uint2 w, int u) {
      const unsigned h = (u & 2) ? w.y : w.x;
      return (int)((u & 1) ? h >> 16 : h & 0xFFFFu);
    };
    constexpr int KS = 4 * L;  // slots from one of the lane's quads to its next
    const int k0 = 4 * sub;
    // with a gathered rest both lanes of a pair run the same steps (coload_rec)
    const int kend = R ? (cnt + KS - 1) / KS * KS + k0 : cnt;
    uint2 w0 = word(k0), w1 = word(k0 + KS);
    int jn[4];
    if constexpr (R) {
#pragma unroll
      for (int u = 0; u < 4; u++) jn[u] = k0 + u < cnt ? sj[sl_of(w0, u)] : 0;
    }
    for (int k = k0; k < kend; k += KS) {
      const int nk = min(4, cnt - k);
      int jc[4];
      if constexpr (R) {
#pragma unroll
        for (int u = 0; u < 4; u++) jc[u] = jn[u];
#pragma unroll
        for (int u = 0; u < 4; u++)
          if (k + KS + u < cnt) jn[u] = sj[sl_of(w1, u)];
      }
      const uint2 w2 = word(k + 2 * KS);
      Rest rr[4];
      if constexpr (R) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
          uint4 c[sizeof(Rest) / 16];
          coload_rec<sizeof(Rest) / 16>(K::rest(f), jc[u], sub & 1, c);
          __builtin_memcpy(&rr[u], c, sizeof(Rest));
        }
      }
      quad([&](auto& sum) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
          PT x, y, z;
          typename K::Nb nb;
          if constexpr (DropOf<K>::on) {
            // entries past the list repeat one of it (TileLists) and add exact
            // zeros (drop): another particle's value, were it not finite, would
            // reach a particle that does not list it as 0 x NaN
            fetch(sl_of(w0, u), x, y, z, nb);
            if (u >= nk) K::drop(nb);
            K::pair(x, y, z, nb, own, sum, prm);
          } else if (u < nk) {
            fetch(sl_of(w0, u), x, y, z, nb);
            if constexpr (R) K::rest_get(rr[u], nb);
            K::pair(x, y, z, nb, own, sum, prm);
          }
        }
      });
      w0 = w1;
      w1 = w2;
    }
  } else {
    // A larger set: its first ST entries are staged, what a pair reads of one
    // beyond comes from memory.  Rows ascend, so that is the end of some lists.
    // Staging the set in passes instead made such a tile take more than twice
    // as long, which showed in every domain of a few rounds of workgroups: mixed
    // step with a 0.4 dx skin at 61,748 particles 80.9 -> 63.0 us, with the
    // positions off the lattice at 20,400 77.6 -> 49.9, sets left uncompacted
    // (~1,230 particles) at 801,536 629 -> 500 us (gathering: 70.3, 58.0, 732);
    // FP64 92.9 -> 82.4, 77.0 -> 62.7, 1,156 -> 885 (101, 80.4, 1,281).
    stage(0, ST);
    __syncthreads();
    const uint2* __restrict__ q = tl.slotq + min((int64_t)i, tl.npad - 1);
    const int klast = max(cnt - 1, 0);
    const unsigned np = (unsigned)tl.npad;
    auto word = [&](int k) { return q[(unsigned)(min(k, klast) >> 2) * np]; };
    constexpr int KS = 4 * L;
    uint2 w0 = word(4 * sub);
    for (int k = 4 * sub; k < cnt; k += KS) {
      const uint2 w1 = word(k + KS);
      const int nk = min(4, cnt - k);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (u >= nk) break;
        const unsigned h = (u & 2) ? w0.y : w0.x;
        const int sl = (int)((u & 1) ? h >> 16 : h & 0xFFFFu);
        quad([&](auto& sum) {
          PT x, y, z;
          typename K::Nb nb;
          if (sl < ST) {
            fetch(sl, x, y, z, nb);
            if constexpr (R) K::rest_get(gat<Rest>(K::rest(f), sj[sl]), nb);
          } else {
            const int j = tj[sl];
            LV e[NV];
            LW r[1] = {};
            K::lds_put(f, j, cx, e, r);
            K::lds_get(e, r, x, y, z, nb);
            if constexpr (R) K::rest_get(gat<Rest>(K::rest(f), j), nb);
          }
          K::pair(x, y, z, nb, own, sum, prm);
        });
      }
      w0 = w1;
    }
  }
  merge_lanes<K, L>(acc);
  if constexpr (TailOf<K>::on) {
    __syncthreads();  // the staged set is read no more
    if (sub == 0) K::template tail_put<P>(f, i, act, acc, prm, &sv[0][0], tid / L);
    __syncthreads();
    K::template tail<P>(f, b * P + tid, prm, &sv[0][0], b, pre);
  } else {
    if (sub == 0) K::finish(f, i, act, own, acc, prm);
  }
  if constexpr (FoldOf<K>::on) {
    if (blockIdx.x == 0 && prm.fold.nb > 0) {
      __syncthreads();  // the staged set is read no more: its LDS is scratch
      block_fold_stats(prm.fold, reinterpret_cast<unsigned long long*>(&sv[0][0]));
    }
  }
}

// A: density rate (InteractionAlt.cu:166-246), fused density update writes
// the next {v, m/rho} mirror
template <bool UH>
struct DensG {
  WF_GATHER32
  static constexpr int NBATCH = 4;
  struct Prm {
    int limit, n;
    double dt;
    int fuse;
    float cs;
    int mdj_alt;  // write m/rho into the next conduction record (fused with conduction)
    int skip;     // drho is overwritten unread (StepParams::keep): don't store it
  };
  struct Own {
    float x, y, z, vx, vy, vz;
    HConstF hc;
    double rho, m;  // of the update after the loop
  };
  struct Nb {
    float4 v;  // v, m/rho
    float h;
  };
  __device__ static void drop(Nb& nb) { nb.v.w = 0.f; }
  typedef KSum Acc;
  typedef float Part;  // a batch's terms in FP32, then added to the FP64 sum
  __device__ static void pzero(Part& q) { q = 0.f; }
  __device__ static void flush(Acc& a, const Part& q) { a.add(q); }
  __device__ static void merge(Acc& a, const Acc& b) {
    a.add(b);
  }
  __device__ static void init(const Fields& f, int i, bool act, Own& o, Acc& a, const Ctx32& c) {
    a.zero();
    if (!act) return;
    pos32(f, i, c, o.x, o.y, o.z);
    const float4 v = f.v4[i];
    o.vx = v.x; o.vy = v.y; o.vz = v.z;
    o.hc = hconst_f(f.h32[i]);
    o.rho = f.rho[i];
    o.m = f.m[i];
  }
  __device__ static void load(const Fields& f, int j, Nb& nb) {
    nb.v = gat<float4>(f.v4, j);
    nb.h = UH ? 0.f : gat<float>(f.h32, j);
  }
  // staged whole: {x, y, z, m/rho}, {v, -}
  WF_LDS32(2, 0)
  __device__ static void lds_put(const Fields& f, int j, const Ctx& c, float4 (&q)[2],
                                 float (&)[1]) {
    float x, y, z;
    pos32(f, j, c, x, y, z);
    q[1] = gat<float4>(f.v4, j);
    q[0] = make_float4(x, y, z, q[1].w);
  }
  __device__ static void lds_get(const float4 (&q)[2], const float (&)[1], float& x, float& y,
                                 float& z, Nb& nb) {
    x = q[0].x;
    y = q[0].y;
    z = q[0].z;
    nb.v = make_float4(q[1].x, q[1].y, q[1].z, q[0].w);
  }
  __device__ static void pair(float x, float y, float z, const Nb& nb, const Own& o, Part& a,
                              const Prm&) {
    const float xx = o.x - x, xy = o.y - y, xz = o.z - z;
    const float r2 = xx * xx + xy * xy + xz * xz;
    float h_;
    const float GK = gk_pair_f<UH>(r2, nb.h, o.hc, h_);
    const float vx = o.vx - nb.v.x, vy = o.vy - nb.v.y, vz = o.vz - nb.v.z;
    a = __builtin_fmaf(nb.v.w, GK * (vx * xx + vy * xy + vz * xz), a);
  }
  __device__ static void finish(const Fields& f, int i, bool act, const Own& o, const Acc& a,
                                const Prm& p) {
    if (act) {
      const double rho = o.rho;
      const double drho = rho * a.val();
      if (!p.skip) f.drho[i] = drho;
      if (p.fuse) {
        const double rn = rho + p.dt * drho;
        f.rho_alt[i] = rn;
        const float mdj = (float)(o.m / rn);
        f.v4_alt[i] = make_float4(o.vx, o.vy, o.vz, mdj);
        (p.mdj_alt ? f.tk4_alt : f.tk4)[i].z = mdj;  // m/rho for the conduction loop
      }
    } else if (p.fuse && i < p.n) {
      f.rho_alt[i] = f.rho[i];
      f.v4_alt[i] = f.v4[i];
    }
  }
};

// B: strain and rotation rates (InteractionAlt.cu:262-383).  With
// a = w v_ij (w = (m_j/rho_j) GK) the rates are sums of the nine products
// a_k x_l: the diagonal takes a_x x_x, a_y x_y, a_z x_z, each off-diagonal
// pair (k, l) the sum (strain) and the difference (rotation) of a_k x_l and
// a_l x_k.  The loop sums the nine products (one FMA each) and forms the
// sums and differences once per particle.  Summing four pairs' products in
// FP32 before adding them to FP64 was as fast but doubled the plastic-strain
// and temperature error of a 3,000-step Johnson-Cook run against FP64
// (5.6e-5 vs 2.8e-5).
// SF: the free-surface sums of the same pairs as well (SurfSums)
template <bool UH, bool SF = false>
struct RatesG {
  WF_GATHER32
  static constexpr int NBATCH = 4;
  struct Prm {
    int limit;
    double xz_sign;
    float cs;
    SurfPrm<float> sf;
  };
  typedef typename DensG<UH>::Own Own;
  typedef typename DensG<UH>::Nb Nb;
  // the neighbour's {v, m/rho} is staged in LDS with its position
  typedef float4 Extra;
  __device__ static Extra extra(const Fields& f, int j) { return gat<float4>(f.v4, j); }
  __device__ static void put(Nb& nb, const Extra& e) { nb.v = e; }
  __device__ static void load(const Fields& f, int j, Nb& nb) {
    nb.h = UH ? 0.f : gat<float>(f.h32, j);
  }
  WF_LDS32(2, 0)
  __device__ static void lds_put(const Fields& f, int j, const Ctx& c, float4 (&q)[2],
                                 float (&r)[1]) {
    DensG<UH>::lds_put(f, j, c, q, r);
  }
  __device__ static void lds_get(const float4 (&q)[2], const float (&r)[1], float& x, float& y,
                                 float& z, Nb& nb) {
    DensG<UH>::lds_get(q, r, x, y, z, nb);
  }
  // products a_k x_l: xx, yy, zz, then (x y, y x), (y z, z y), (x z, z x)
  // each product of two FP32 factors is exact in FP64 and added by one FP64
  // FMA: 6 conversions and 9 FMAs a pair.  Widening each FP32 product and
  // adding it costs 27 operations, and this loop is bound by its vector ALU:
  // on a 759k-particle cylinder 0.082 -> 0.066 ms, with the same error
  // against the FP64 rates (4.7e-7 relative L2; the FP32 factors set it)
  struct Acc : SurfSums<SF> {
    double xx, yy, zz, xy, yx, yz, zy, xz, zx;
  };
  __device__ static void merge(Acc& a, const Acc& b) {
    a.xx += b.xx; a.yy += b.yy; a.zz += b.zz;
    a.xy += b.xy; a.yx += b.yx; a.yz += b.yz;
    a.zy += b.zy; a.xz += b.xz; a.zx += b.zx;
    a.surf_merge(b);
  }
  __device__ static void init(const Fields& f, int i, bool act, Own& o, Acc& a, const Ctx32& c) {
    a = Acc{};
    if (!act) return;
    pos32(f, i, c, o.x, o.y, o.z);
    const float4 v = f.v4[i];
    o.vx = v.x; o.vy = v.y; o.vz = v.z;
    o.hc = hconst_f(f.h32[i]);
  }
  __device__ static void pair(float x, float y, float z, const Nb& nb, const Own& o, Acc& a,
                              const Prm& p) {
    const float xx = o.x - x, xy = o.y - y, xz = o.z - z;
    const float r2 = xx * xx + xy * xy + xz * xz;
    a.surf_add(xx, xy, xz, r2, p.sf);
    float h_;
    const float w = gk_pair_f<UH>(r2, nb.h, o.hc, h_) * nb.v.w;
    const float vx = o.vx - nb.v.x, vy = o.vy - nb.v.y, vz = o.vz - nb.v.z;
    const double ax = w * vx, ay = w * vy, az = w * vz;
    const double dx = xx, dy = xy, dz = xz;
    a.xx = __builtin_fma(ax, dx, a.xx);
    a.yy = __builtin_fma(ay, dy, a.yy);
    a.zz = __builtin_fma(az, dz, a.zz);
    a.xy = __builtin_fma(ax, dy, a.xy);
    a.yx = __builtin_fma(ay, dx, a.yx);
    a.yz = __builtin_fma(ay, dz, a.yz);
    a.zy = __builtin_fma(az, dy, a.zy);
    a.xz = __builtin_fma(ax, dz, a.xz);
    a.zx = __builtin_fma(az, dx, a.zx);
  }
  __device__ static void finish(const Fields& f, int i, bool act, const Own&, const Acc& a,
                                const Prm& p) {
    if (!act) return;
    float v[9];
    rates9(a, p, v);
    put9(f, i, v);
    a.surf_finish(f, i, p.sf);
  }
  typedef float RT;
  __device__ static void rates9(const Acc& a, const Prm& p, float (&v)[9]) {
    v[0] = (float)-a.xx; v[1] = (float)-a.yy; v[2] = (float)-a.zz;
    v[3] = (float)(-0.5 * (a.xy + a.yx));
    v[4] = (float)(-0.5 * (a.yz + a.zy));
    v[5] = (float)(-0.5 * (a.xz + a.zx));
    v[6] = (float)(-0.5 * (a.xy - a.yx));
    v[7] = (float)(-0.5 * (a.yz - a.zy));
    v[8] = (float)(-0.5 * p.xz_sign * (a.xz - a.zx));
  }
  __device__ static void put9(const Fields& f, int i, const float (&v)[9]) {
#pragma unroll
    for (int k = 0; k < 6; k++) f.strrate32[k][i] = v[k];
#pragma unroll
    for (int k = 0; k < 3; k++) f.rotrate32[3 + k][i] = v[6 + k];
  }
};

// B and C in one pass: the rates pass R that runs its particles' stress update
// (stress_particle) as soon as their sums are done, which saves a launch and
// the rates' way through memory (rates_stress_blocks says where); a lane a
// particle and whole wavefronts, because the surrogate's matrix instructions
// take all 64 lanes.
// AHEAD: with a tile dealt out to several workgroups, at most one a CU, there
// are registers to load what the update reads before the pair loop.  FP64
// step, us: 2,000 bilinear particles 22.2 -> 21.5, 8,272 Johnson-Cook 33.2 ->
// 33.0; not with whole tiles (20,640: 35.7 -> 36.0) nor in mixed precision
// (8,272: 27.0 -> 27.5).
template <class R, int REC, bool S32, bool AHEAD>
struct RatesStress : R {
  static constexpr bool TAIL = true, PRE = AHEAD;
  typedef StressIn Pre;
  // 160 registers of 168 (unasked: 170, two a SIMD)
  static constexpr int MIN_WAVES = AHEAD ? 1 : 3;
  struct Prm : R::Prm {
    StepParams sp;
    RetArgs ra;
    BlockStats* bs;  // one entry a workgroup
  };
  __device__ static void pre(const Fields& f, const Prm& p, int i, Pre& in) {
    stress_load<true, true, S32>(f, p.sp, i, in);
  }
  typedef typename R::RT RT;
  template <int P>
  __device__ static void tail_put(const Fields& f, int i, bool act, const typename R::Acc& a,
                                  const Prm& p, void* lds, int q) {
    RT v[9];
    R::rates9(a, p, v);
    if (act) a.surf_finish(f, i, p.sf);
    RT* sh = reinterpret_cast<RT*>(lds);
#pragma unroll
    for (int k = 0; k < 9; k++) sh[k * P + q] = v[k];
  }
  template <int P>
  __device__ static void tail(const Fields& f, int i, const Prm& p, void* lds, int b, Pre& in) {
    constexpr int NW = P >= 64 ? P / 64 : 1;  // wavefronts that update particles
    BlockStats st{0ull, 0ull, 0ull, 0ull};
    if (threadIdx.x < 64 * NW) {
      const RT* sh = reinterpret_cast<const RT*>(lds) + threadIdx.x;
      auto rates = [&](double (&d)[6], double (&w)[3]) {
        RT v[9];
#pragma unroll
        for (int k = 0; k < 9; k++) v[k] = sh[k * P];
#pragma unroll
        for (int k = 0; k < 6; k++) d[k] = v[k];
#pragma unroll
        for (int k = 0; k < 3; k++) w[k] = v[6 + k];
      };
      const bool active = (int)threadIdx.x < P && i < p.limit;
      if (!AHEAD && active) pre(f, p, i, in);
      stress_particle<true, true, REC, S32>(f, p.sp, p.ra, i, active, in, rates, st);
      if (p.sp.keep && active) {
        RT v[9];
#pragma unroll
        for (int k = 0; k < 9; k++) v[k] = sh[k * P];
        R::put9(f, i, v);
      }
    }
    stress_block_stats(st, NW, reinterpret_cast<BlockStats*>((RT*)lds + 9 * P), p.bs + b);
  }
};

// D: acceleration with Monaghan viscosity (InteractionAlt.cu:18-150)
#ifndef WF_ACCEL32_NBATCH
#define WF_ACCEL32_NBATCH 4
#endif
#ifndef WF_ACCEL32_WAVES
#define WF_ACCEL32_WAVES 1
#endif
// BV: the beta (quadratic) viscosity term is on; IT: each particle is
// integrated as soon as its sum is done (IntegratePrm), its integration
// inputs loaded before the pair loop
// UC: every particle has the same sound speed (and h)
template <bool UH, bool BV = false, bool IT = false, bool UC = false>
struct AccelG {
  WF_GATHER32
  static constexpr int NBATCH = WF_ACCEL32_NBATCH;
  static constexpr int MIN_WAVES = WF_ACCEL32_WAVES;
  struct Prm {
    int limit;
    float alpha32, beta32;
    float cs;
    IntegratePrm ip;  // integrate each particle after its sum (IT)
    StatsFold fold;   // the stress pass's statistics, folded by workgroup 0
    float cs_uni;     // UC
  };
  struct NoIn {};
  struct Own {
    float x, y, z, vx, vy, vz, di, Ci, s0, s1, s2, s3, s4, s5;
    HConstF hc;
    std::conditional_t<IT, IntegrateIn, NoIn> in;
  };
  struct Nb {
    float4 v, sa, sb;  // {v, m}, sigma/rho^2 {xx, yy, zz, xy}, {yz, xz, rho, Cs}
    float h;
  };
  __device__ static void drop(Nb& nb) { nb.v.w = 0.f; }
  struct Acc {
    KSum ax, ay, az;
  };
  // a batch's pair terms summed in FP32, then added to the FP64 sums
  struct Part {
    float ax, ay, az;
  };
  __device__ static void pzero(Part& q) { q = Part{0.f, 0.f, 0.f}; }
  __device__ static void flush(Acc& a, const Part& q) {
    a.ax.add(q.ax); a.ay.add(q.ay); a.az.add(q.az);
  }
  __device__ static void merge(Acc& a, const Acc& b) {
    a.ax.add(b.ax); a.ay.add(b.ay); a.az.add(b.az);
  }
  __device__ static void init(const Fields& f, int i, bool act, Own& o, Acc& a, const Ctx32& c) {
    a.ax.zero(); a.ay.zero(); a.az.zero();
    if (!act) return;
    pos32(f, i, c, o.x, o.y, o.z);
    const float4 v = f.v4[i], sa = f.arec[rec32_at(i, 0)], sb = f.arec[rec32_at(i, 1)];
    o.vx = v.x; o.vy = v.y; o.vz = v.z;
    o.s0 = sa.x; o.s1 = sa.y; o.s2 = sa.z; o.s3 = sa.w;
    o.s4 = sb.x; o.s5 = sb.y; o.di = sb.z; o.Ci = sb.w;
    o.hc = hconst_f(f.h32[i]);
    if constexpr (IT) integrate_load<kRec32>(f, i, o.in);
  }
  // the neighbour's {v, m} (m = (m/rho) rho, formed once per staged
  // particle) is staged in LDS with its position, so a pair gathers only the
  // 32-byte stress record
  typedef float4 Extra;
  __device__ static Extra extra(const Fields& f, int j) {
    float4 v = gat<float4>(f.v4, j);
    v.w *= gat<float4, 32>(f.arec, j, 16).z;  // rec32_at(j, 1)
    return v;
  }
  __device__ static void put(Nb& nb, const Extra& e) { nb.v = e; }
  // UC: staged whole: {x, y, z, rho}, {v, s_xx}, {s_yy, s_zz, s_xy, s_yz},
  // {s_xz, m} with s = sigma/rho^2 (56 bytes: 960 leave three workgroups a CU)
  typedef float4 LV;
  typedef float2 LW;
  static constexpr int NV = 3, NW = 1, SET = 960;
  __device__ static void lds_put(const Fields& f, int j, const Ctx& c, float4 (&q)[3],
                                 float2 (&r)[1]) {
    const float4 v = gat<float4>(f.v4, j);
    const float4 sa = gat<float4, 32>(f.arec, j), sb = gat<float4, 32>(f.arec, j, 16);
    float x, y, z;
    pos32(f, j, c, x, y, z);
    q[0] = make_float4(x, y, z, sb.z);
    q[1] = make_float4(v.x, v.y, v.z, sa.x);
    q[2] = make_float4(sa.y, sa.z, sa.w, sb.x);
    r[0] = make_float2(sb.y, v.w * sb.z);  // m = (m/rho) rho, as extra() forms it
  }
  __device__ static void lds_get(const float4 (&q)[3], const float2 (&r)[1], float& x, float& y,
                                 float& z, Nb& nb) {
    x = q[0].x;
    y = q[0].y;
    z = q[0].z;
    nb.v = make_float4(q[1].x, q[1].y, q[1].z, r[0].y);
    nb.sa = make_float4(q[1].w, q[2].x, q[2].y, q[2].z);
    nb.sb = make_float4(q[2].w, r[0].x, q[0].w, 0.f);
  }
  __device__ static void load(const Fields& f, int j, Nb& nb) {
    nb.sa = gat<float4, 32>(f.arec, j);  // rec32_at(j, 0..1)
    nb.sb = gat<float4, 32>(f.arec, j, 16);
    nb.h = UH ? 0.f : gat<float>(f.h32, j);
  }

  __device__ static void pair(float x, float y, float z, const Nb& nb, const Own& o, Part& a,
                              const Prm& p) {
    const float xx = o.x - x, xy = o.y - y, xz = o.z - z;
    const float r2 = xx * xx + xy * xy + xz * xz;
    float h_;
    const float GK = gk_pair_f<UH>(r2, nb.h, o.hc, h_);
    const float vx = o.vx - nb.v.x, vy = o.vy - nb.v.y, vz = o.vz - nb.v.z;
    const float vdx = vx * xx + vy * xy + vz * xz;
    // Monaghan viscosity on approaching pairs only: (alpha C mu + beta mu^2)
    // / rho_bar with mu = h v/e, v = min(v_ij.x_ij, 0), e = r^2 + 0.01 h^2,
    // as 2 h v (alpha C + beta mu) / (e (rho_i + rho_j)) = v h alpha (C_i +
    // C_j) / (e (rho_i + rho_j)) without beta: one reciprocal and no branch
    // (receding pairs get v = 0)
    const float vn = fminf(vdx, 0.f);
    const float rs = o.di + nb.sb.z;
    const float inv = __builtin_amdgcn_rcpf((r2 + 0.01f * h_ * h_) * rs);
    const float Cj = UC ? p.cs_uni : nb.sb.w;
    float PI;
    if constexpr (BV) {
      const float coef =
          (0.5f * p.alpha32) * (o.Ci + Cj) + p.beta32 * (h_ * vn * rs * inv);
      PI = 2.f * h_ * vn * coef * inv;
    } else {
      PI = vn * ((h_ * p.alpha32) * (o.Ci + Cj)) * inv;
    }
    const float g = GK * nb.v.w;
    const float gx = g * xx, gy = g * xy, gz = g * xz;
    const float mxx = o.s0 + nb.sa.x + PI, myy = o.s1 + nb.sa.y + PI;
    const float mzz = o.s2 + nb.sa.z + PI;
    const float mxy = o.s3 + nb.sa.w, myz = o.s4 + nb.sb.x, mxz = o.s5 + nb.sb.y;
    a.ax = __builtin_fmaf(mxz, gz, __builtin_fmaf(mxy, gy, __builtin_fmaf(mxx, gx, a.ax)));
    a.ay = __builtin_fmaf(myz, gz, __builtin_fmaf(myy, gy, __builtin_fmaf(mxy, gx, a.ay)));
    a.az = __builtin_fmaf(mzz, gz, __builtin_fmaf(myz, gy, __builtin_fmaf(mxz, gx, a.az)));
  }
  __device__ static void finish(const Fields& f, int i, bool act, const Own& o, const Acc& a,
                                const Prm& p) {
    if (!act) return;
    if constexpr (IT) {
      if (!p.ip.contacts || p.ip.contacts[i] == 0) {
        integrate_apply<kRec32>(f, i, a.ax.val(), a.ay.val(), a.az.val(), p.ip.dt, p.ip.bc,
                                p.ip.fr, p.ip.out, o.in);
        return;
      }
    }
    f.a[0][i] = a.ax.val();
    f.a[1][i] = a.ay.val();
    f.a[2][i] = a.az.val();
  }
};

// conduction (Thermal.cu:101-142), fused convection, plastic-work heat and
// leapfrog; the next {T, k} mirror is written
template <bool UH>
struct CondG {
  WF_GATHER32
  static constexpr int NBATCH = 4;
  struct Prm {
    int limit;
    double T_inf, h_conv, dt;
    int leap, first;
    float cs;
    int skip;  // dT/dt and T_b are overwritten unread (StepParams::keep)
  };
  struct Own {
    float x, y, z, k, T, mdj;
    HConstF hc;
    CondIn in;
    double Ti;
  };
  struct Nb {
    float4 tk;  // T, k, m/rho
    float h;
  };
  __device__ static void drop(Nb& nb) { nb.tk.z = 0.f; }
  typedef KSum Acc;
  typedef float Part;  // a batch's terms in FP32, then added to the FP64 sum
  __device__ static void pzero(Part& q) { q = 0.f; }
  __device__ static void flush(Acc& a, const Part& q) { a.add(q); }
  __device__ static void merge(Acc& a, const Acc& b) {
    a.add(b);
  }
  __device__ static void init(const Fields& f, int i, bool act, Own& o, Acc& a, const Ctx32& c) {
    a.zero();
    if (!act) return;
    pos32(f, i, c, o.x, o.y, o.z);
    const float4 tk = f.tk4[i];
    o.T = tk.x;
    o.k = tk.y;
    o.mdj = tk.z;
    o.hc = hconst_f(f.h32[i]);
    o.in.load(f, i);
    o.Ti = f.T[i];
  }
  // the neighbour's {T, k, m/rho} is staged in LDS with its position (the
  // pass writes only the next record, tk4_alt)
  typedef float4 Extra;
  __device__ static Extra extra(const Fields& f, int j) { return gat<float4>(f.tk4, j); }
  __device__ static void put(Nb& nb, const Extra& e) { nb.tk = e; }
  __device__ static void load(const Fields& f, int j, Nb& nb) {
    nb.h = UH ? 0.f : gat<float>(f.h32, j);
  }
  // staged whole: {x, y, z, m/rho}, {T, k, -, -}
  WF_LDS32(2, 0)
  __device__ static void lds_put(const Fields& f, int j, const Ctx& c, float4 (&q)[2],
                                 float (&)[1]) {
    float x, y, z;
    pos32(f, j, c, x, y, z);
    q[1] = gat<float4>(f.tk4, j);
    q[0] = make_float4(x, y, z, q[1].z);
  }
  __device__ static void lds_get(const float4 (&q)[2], const float (&)[1], float& x, float& y,
                                 float& z, Nb& nb) {
    x = q[0].x;
    y = q[0].y;
    z = q[0].z;
    nb.tk = make_float4(q[1].x, q[1].y, q[0].w, 0.f);
  }
  __device__ static void pair(float x, float y, float z, const Nb& nb, const Own& o, Part& a,
                              const Prm&) {
    const float xx = o.x - x, xy = o.y - y, xz = o.z - z;
    const float r2 = xx * xx + xy * xy + xz * xz;
    float h_;
    const float GK = gk_pair_f<UH>(r2, nb.h, o.hc, h_);
    const float kj = nb.tk.y;
    const float kh = (kj == o.k) ? 2.f * o.k : 4.f * o.k * kj * __builtin_amdgcn_rcpf(o.k + kj);
    a = __builtin_fmaf(nb.tk.z * kh, (o.T - nb.tk.x) * GK, a);
  }
  __device__ static void finish(const Fields& f, int i, bool act, const Own& o, const Acc& a,
                                const Prm& p) {
    if (!act) return;
    const double Ti = o.Ti, acc = cond_rate(f, i, a.val(), Ti, p, o.in);
    if (!p.skip) f.dTdt[i] = acc;
    if (p.leap) {
      double Tn;
      if (p.first) {
        f.Ta[i] = Ti - p.dt / 2.0 * acc;
        Tn = Ti;
      } else {
        const double ta = o.in.ta;
        if (!p.skip) f.Tb[i] = ta;
        double tan = ta + acc * p.dt;
        f.Ta[i] = tan;
        Tn = (tan + ta) / 2.;
      }
      f.T_alt[i] = Tn;
      f.tk4_alt[i] = make_float4((float)Tn, o.k, o.mdj, 0.f);
    }
  }
};

// ---------------------------------------------------------------------------
// S: free-surface normal n_i = sum_j m_j x_ij * N/(M nb_i) and the surface
// flag |n_i| >= 0.25 h_i with nb_i <= 46 (Geometry.cu:26-88).  Rigid
// triangles are not particles here, so every list entry counts.
#ifndef WF_STAGE_SURF
#define WF_STAGE_SURF 1024
#endif
template <bool UM>
struct SurfD {
  // FP64 positions; its own staging size (a pair costs little here, so the
  // chunked path for large staged sets weighs more)
  typedef double PT;
  static constexpr int STAGE = WF_STAGE_SURF;
#ifndef WF_LANES_SURF
#define WF_LANES_SURF 2
#endif
  static constexpr int LANES = WF_LANES_SURF;
  typedef NoCtx Ctx;
  template <class P>
  __device__ static Ctx ctx(const Fields&, int, const P&) {
    return Ctx{};
  }
  __device__ static void pos(const Fields& f, int j, const Ctx&, double& x, double& y,
                             double& z) {
    x = f.x[0][j];
    y = f.x[1][j];
    z = f.x[2][j];
  }
  static constexpr int NBATCH = 4;
  struct Prm {
    int limit;
    int id_free_surf;
    double ntot, totmass;
    double r2cut;  // > 0: lists carry a skin; count only pairs within the radius
    double m_uni;  // every particle's mass (UM)
  };
  struct Own {
    double x, y, z;
  };
  struct Nb {
    double m;
  };
  struct Acc {
    double nx, ny, nz;
    int cnt;
  };
  __device__ static void merge(Acc& a, const Acc& b) {
    a.nx += b.nx; a.ny += b.ny; a.nz += b.nz;
    a.cnt += b.cnt;
  }
  __device__ static void init(const Fields& f, int i, bool act, Own& o, Acc& a, const NoCtx&) {
    a.nx = a.ny = a.nz = 0.0;
    a.cnt = 0;
    if (!act) return;
    o.x = f.x[0][i]; o.y = f.x[1][i]; o.z = f.x[2][i];
  }
  __device__ static void load(const Fields& f, int j, Nb& nb) { nb.m = UM ? 0.0 : f.m[j]; }
  __device__ static void pair(double x, double y, double z, const Nb& nb, const Own& o, Acc& a,
                              const Prm& p) {
    const double dx = o.x - x, dy = o.y - y, dz = o.z - z;
    if (p.r2cut > 0.0 && !(dx * dx + dy * dy + dz * dz < p.r2cut)) return;
    const double mj = UM ? p.m_uni : nb.m;
    a.nx += mj * dx;
    a.ny += mj * dy;
    a.nz += mj * dz;
    a.cnt++;
  }
  __device__ static void finish(const Fields& f, int i, bool act, const Own&, const Acc& a,
                                const Prm& p) {
    if (!act) return;
    surface_finish(f, i, a.nx, a.ny, a.nz, a.cnt, p.ntot, p.totmass, p.id_free_surf);
  }
};

static inline int ntiles(int n) { return (n + kTileP - 1) / kTileP; }

// the same in mixed precision: FP32 tile-frame positions, each FP32 term
// m_j x_ij summed in FP64 and the flag decided in FP64 from those sums (a
// flag can differ from the FP64 pass only for |n| within ~1e-7 of 0.25 h)
template <bool UM>
struct SurfG {
  WF_GATHER32
  static constexpr int NBATCH = 4;
  struct Prm {
    int limit;
    int id_free_surf;
    double ntot, totmass;
    float r2cut;  // > 0: lists carry a skin; count only pairs within the radius
    float m_uni;  // every particle's mass (UM)
    float cs;
  };
  struct Own {
    float x, y, z;
  };
  struct Nb {
    float m;
  };
  struct Acc {
    KSum nx, ny, nz;
    int cnt;
  };
  __device__ static void merge(Acc& a, const Acc& b) {
    a.nx.add(b.nx); a.ny.add(b.ny); a.nz.add(b.nz);
    a.cnt += b.cnt;
  }
  __device__ static void init(const Fields& f, int i, bool act, Own& o, Acc& a, const Ctx32& c) {
    a.nx.zero(); a.ny.zero(); a.nz.zero();
    a.cnt = 0;
    if (!act) return;
    pos32(f, i, c, o.x, o.y, o.z);
  }
  __device__ static void load(const Fields& f, int j, Nb& nb) {
    nb.m = UM ? 0.f : (float)f.m[j];
  }
  __device__ static void pair(float x, float y, float z, const Nb& nb, const Own& o, Acc& a,
                              const Prm& p) {
    const float dx = o.x - x, dy = o.y - y, dz = o.z - z;
    if (p.r2cut > 0.f && !(dx * dx + dy * dy + dz * dz < p.r2cut)) return;
    const float mj = UM ? p.m_uni : nb.m;
    a.nx.add(mj * dx);
    a.ny.add(mj * dy);
    a.nz.add(mj * dz);
    a.cnt++;
  }
  __device__ static void finish(const Fields& f, int i, bool act, const Own&, const Acc& a,
                                const Prm& p) {
    if (!act) return;
    surface_finish(f, i, a.nx.val(), a.ny.val(), a.nz.val(), a.cnt, p.ntot, p.totmass,
                   p.id_free_surf);
  }
};

}  // namespace wf

namespace wf {
// neighbour record of a fused pass, and the first pass's staged extra value
// (if it has one) forwarded to the fused functor
template <class A, class B>
struct CondDensNb {
  typename A::Nb a;
  typename B::Nb b;
};
template <class A, class Nb, bool = ExtraOf<A>::on>
struct FusedExtra {};
template <class A, class Nb>
struct FusedExtra<A, Nb, true> {
  typedef typename A::Extra Extra;
  __device__ static Extra extra(const Fields& f, int j) { return A::extra(f, j); }
  __device__ static void put(Nb& nb, const Extra& e) { A::put(nb.a, e); }
};

// Conduction of one step fused with the density pass of the next: both read
// the positions after integration and the same neighbour lists, and neither
// reads what the other writes (the density pass puts the new m/rho into the
// next conduction record), so one traversal of the lists serves both.  Each
// sum runs over the list in the same order as in its own kernel.
// the fused pass sums a batch in partial sums when both passes do
template <class A, class B, bool = PartOf<A>::on && PartOf<B>::on>
struct FusedPart {};
template <class A, class B>
struct FusedPart<A, B, true> {
  struct Part {
    typename A::Part a;
    typename B::Part b;
  };
  __device__ static void pzero(Part& q) {
    A::pzero(q.a);
    B::pzero(q.b);
  }
  template <class Acc>
  __device__ static void flush(Acc& s, const Part& q) {
    A::flush(s.a, q.a);
    B::flush(s.b, q.b);
  }
};

// and evaluates a batch in straight-line code when both passes can
template <class A, class B, bool = DropOf<A>::on && DropOf<B>::on>
struct FusedDrop {};
template <class A, class B>
struct FusedDrop<A, B, true> {
  __device__ static void drop(CondDensNb<A, B>& nb) {
    A::drop(nb.a);
    B::drop(nb.b);
  }
};

template <class A, class B>
struct CondDens : FusedExtra<A, CondDensNb<A, B>>, FusedPart<A, B>, FusedDrop<A, B> {
  typedef typename A::PT PT;
  static constexpr int STAGE = A::STAGE;
  static constexpr int LANES = A::LANES;
  static_assert(A::LANES == B::LANES, "fused passes share the lane split");
  static constexpr int NBATCH = A::NBATCH < B::NBATCH ? A::NBATCH : B::NBATCH;
  typedef typename A::Ctx Ctx;
  struct Prm {
    int limit;  // particles of the conduction pass (>= the density pass's)
    typename A::Prm a;
    typename B::Prm b;
    // (may be null) the plastic-zone trigger's largest squared hot
    // displacement, as FP64 bits, and skin^2: when 4 d2 > skin^2 a rebuild
    // starts the next step, and the density half writes nothing
    const unsigned long long* pz_d2;
    double pz_skin2;
  };
  struct Own {
    typename A::Own a;
    typename B::Own b;
  };
  typedef CondDensNb<A, B> Nb;
  struct Acc {
    typename A::Acc a;
    typename B::Acc b;
  };
  template <class P>
  __device__ static Ctx ctx(const Fields& f, int t, const P& p) {
    return A::ctx(f, t, p.a);
  }
  __device__ static void pos(const Fields& f, int j, const Ctx& c, PT& x, PT& y, PT& z) {
    A::pos(f, j, c, x, y, z);
  }
  __device__ static void init(const Fields& f, int i, bool act, Own& o, Acc& a, const Ctx& c) {
    A::init(f, i, act, o.a, a.a, c);
    B::init(f, i, act, o.b, a.b, c);
  }
  __device__ static void load(const Fields& f, int j, Nb& nb) {
    A::load(f, j, nb.a);
    B::load(f, j, nb.b);
  }
  static constexpr bool CO = CoOf<A>::on && CoOf<B>::on;
  __device__ static void coload(const Fields& f, int j, int sub, Nb& nb) {
    if constexpr (CO) {
      A::coload(f, j, sub, nb.a);
      B::coload(f, j, sub, nb.b);
    }
  }
  // staged whole: the density pass's entries and T, k (the m/rho of the two
  // records is the same value): FP64 {x, y}, {z, m/rho}, {v_x, v_y}, {T, k},
  // v_z, FP32 {x, y, z, m/rho}, {v, T}, k
  static constexpr bool F64 = std::is_same<PT, double>::value;
  typedef std::conditional_t<F64, double2, float4> LV;
  typedef PT LW;
  static constexpr int NV = F64 ? 4 : 2, NW = 1, SET = 1024;
  __device__ static void lds_put(const Fields& f, int j, const Ctx& c, LV (&q)[NV], PT (&r)[1]) {
    if constexpr (F64) {
      const double4 v = gat<double4>(f.kv, j);
      q[0] = make_double2(f.x[0][j], f.x[1][j]);
      q[1] = make_double2(f.x[2][j], v.w);
      q[2] = make_double2(v.x, v.y);
      q[3] = gat<double2, 32>(f.tk64, j);
      r[0] = v.z;
    } else {
      const float4 v = gat<float4>(f.v4, j), tk = gat<float4>(f.tk4, j);
      float x, y, z;
      pos32(f, j, c, x, y, z);
      q[0] = make_float4(x, y, z, v.w);
      q[1] = make_float4(v.x, v.y, v.z, tk.x);
      r[0] = tk.y;
    }
  }
  __device__ static void lds_get(const LV (&q)[NV], const PT (&r)[1], PT& x, PT& y, PT& z,
                                 Nb& nb) {
    x = q[0].x;
    y = q[0].y;
    if constexpr (F64) {
      z = q[1].x;
      nb.b.v = make_double4(q[2].x, q[2].y, r[0], q[1].y);
      nb.a.tk = make_double4(q[3].x, q[3].y, q[1].y, 0.0);
    } else {
      z = q[0].z;
      nb.b.v = make_float4(q[1].x, q[1].y, q[1].z, q[0].w);
      nb.a.tk = make_float4(q[1].w, r[0], q[0].w, 0.f);
    }
  }
  // S: the sums (Acc) or the batch's partial sums (Part)
  template <class S>
  __device__ static void pair(PT x, PT y, PT z, const Nb& nb, const Own& o, S& a,
                              const Prm& p) {
    A::pair(x, y, z, nb.a, o.a, a.a, p.a);
    B::pair(x, y, z, nb.b, o.b, a.b, p.b);
  }
  __device__ static void merge(Acc& a, const Acc& b) {
    A::merge(a.a, b.a);
    B::merge(a.b, b.b);
  }
  __device__ static void finish(const Fields& f, int i, bool act, const Own& o, const Acc& a,
                                const Prm& p) {
    A::finish(f, i, act, o.a, a.a, p.a);
    if (p.pz_d2 && 4.0 * __longlong_as_double((long long)*p.pz_d2) > p.pz_skin2) return;
    B::finish(f, i, i < p.b.limit, o.b, a.b, p.b);
  }
};
template <bool UH>
using CondDensD = CondDens<CondD<UH>, DensD<UH>>;
template <bool UH>
using CondDensG = CondDens<CondG<UH>, DensG<UH>>;

template <bool UH>
using RatesDU = RatesD<UH>;
template <bool UH>
using RatesGU = RatesG<UH>;

LaunchEvents g_next_launch = {nullptr, nullptr};

template <class K>
static void launch_timed(void (*kernel)(Fields, TileLists, typename K::Prm), dim3 grid, dim3 block,
                         hipStream_t s, const Fields& f, const TileLists& tl,
                         const typename K::Prm& p) {
  if (g_next_launch.start) {
    hipExtLaunchKernelGGL(kernel, grid, block, 0, s, g_next_launch.start, g_next_launch.stop, 0, f,
                          tl, p);
    g_next_launch = LaunchEvents{nullptr, nullptr};
  } else {
    hipLaunchKernelGGL(kernel, grid, block, 0, s, f, tl, p);
  }
}
// One pair pass over nt tiles, the neighbours staged whole (LDS) or gathered
// (with its dispatch timestamps in g_next_launch's events when those are set).
//
// A domain of few tiles leaves most of the 256 CUs idle and its passes last as
// long as one tile's chain of loads and pairs, so a tile is dealt out to 8, 4
// or 2 workgroups as long as they fit one a CU: each stages the whole set
// (which costs the idle CUs nothing) and has 16, 8 or 4 lanes a particle
// instead of 2.  Past one a CU the repeated staging costs more than the shorter
// chain gains: Johnson-Cook step, us, with 1 / 2 / 4 / 8 workgroups a tile
// (FP64; mixed): 17 tiles 44.4 / 38.0 / 34.0 / 33.4; 34.8 / 30.5 / 28.5 /
// 26.3; 41 tiles 45.1 / 38.6 / 35.7 / 37.5; 35.3 / 31.2 / 29.2 / 30.0; 65
// tiles 45.4 / 38.7 / 40.3 / 45.2; 34.9 / 30.8 / 31.4 / 31.8; 142 tiles 46.9 /
// 48.1 / 51.5 / 60.7; 35.6 / 35.4 / 35.4 / 42.7.
constexpr int kCus = 256;
static int pair_split(int nt) {
  return 8 * nt <= kCus ? 8 : 4 * nt <= kCus ? 4 : 2 * nt <= kCus ? 2 : 1;
}
// Up to two tiles a CU, 1,024 staged entries cost no loop a workgroup a CU (an
// entry has at most 76 bytes) and send fewer tiles to memory.
constexpr int kSetMax = 1024;
template <class K, bool LDS = true>
static void launch_pair(hipStream_t s, int nt, const Fields& f, const TileLists& tl,
                        const typename K::Prm& p) {
  if constexpr (LDS && HasLds<K>::on) {
    constexpr int kThreads = 2 * kTileP;
    const int split = pair_split(nt);
    auto go = [&](auto kernel) {
      launch_timed<K>(kernel, dim3(nt * split), dim3(kThreads), s, f, tl, p);
    };
    if (split == 8) go(k_pair_lds<K, 16, kTileP / 8, kSetMax>);
    else if (split == 4) go(k_pair_lds<K, 8, kTileP / 4, kSetMax>);
    else if (split == 2) go(k_pair_lds<K, 4, kTileP / 2, kSetMax>);
    else if (nt <= 2 * kCus) go(k_pair_lds<K, 2, kTileP, kSetMax>);
    else go(k_pair_lds<K, 2, kTileP, K::SET>);
  } else {
    launch_timed<K>(k_pair_gather<K>, dim3(nt), dim3(kTileP * K::LANES), s, f, tl, p);
  }
}

// launch policy POL with every particle's h equal (UH) or not
template <template <bool> class POL, class... A>
static void launch_gather(hipStream_t s, const Fields& f, const TileLists& tl, int grid, bool uh,
                          A... args) {
  if (uh) launch_pair<POL<true>>(s, grid, f, tl, typename POL<true>::Prm{args...});
  else launch_pair<POL<false>, false>(s, grid, f, tl, typename POL<false>::Prm{args...});
}

void launch_surface_mixed(hipStream_t s, const Fields& f, const TileLists& tl, int solid,
                          double ntot, double totmass, int id_free_surf, double r2cut, bool um,
                          double m_value, float cs32) {
  if (solid <= 0) return;
  const float r2 = (float)r2cut;
  if (um) {
    const SurfG<true>::Prm p{solid, id_free_surf, ntot, totmass, r2, (float)m_value, cs32};
    launch_pair<SurfG<true>>(s, ntiles(solid), f, tl, p);
  } else {
    const SurfG<false>::Prm p{solid, id_free_surf, ntot, totmass, r2, 0.f, cs32};
    launch_pair<SurfG<false>, false>(s, ntiles(solid), f, tl, p);
  }
}

void launch_surface_tiled(hipStream_t s, const Fields& f, const TileLists& tl, int solid,
                          double ntot, double totmass, int id_free_surf, double r2cut, bool um,
                          double m_value) {
  if (solid <= 0) return;
  if (um) {
    const SurfD<true>::Prm p{solid, id_free_surf, ntot, totmass, r2cut, m_value};
    launch_pair<SurfD<true>>(s, ntiles(solid), f, tl, p);
  } else {
    const SurfD<false>::Prm p{solid, id_free_surf, ntot, totmass, r2cut, 0.0};
    launch_pair<SurfD<false>, false>(s, ntiles(solid), f, tl, p);
  }
}

void launch_dens_tiled(hipStream_t s, const Fields& f, const TileLists& tl, int n, int solid,
                       double dt, bool fuse, bool uh) {
  if (n <= 0) return;
  launch_gather<DensD>(s, f, tl, ntiles(n), uh, solid, n, dt, fuse ? 1 : 0);
}
static double xz_sign(int quirks) { return (quirks & WF_Q_ROT_XZ_SIGN) ? -1.0 : 1.0; }
void launch_rates_tiled(hipStream_t s, const Fields& f, const TileLists& tl, int solid,
                        int quirks, bool uh, const SurfaceArgs* sf) {
  if (solid <= 0) return;
  const double xz = xz_sign(quirks);
  if (sf) {
    typedef RatesD<true, true> K;
    const SurfPrm<double> sp{sf->id_free_surf, sf->ntot, sf->totmass, sf->r2cut, sf->m};
    launch_pair<K>(s, ntiles(solid), f, tl, K::Prm{solid, xz, sp});
  } else {
    launch_gather<RatesDU>(s, f, tl, ntiles(solid), uh, solid, xz, SurfPrm<double>{});
  }
}
void launch_accel_tiled(hipStream_t s, const Fields& f, const TileLists& tl, int solid,
                        double alpha, double beta, bool uh, double m_uni, double cs_uni,
                        const StatsFold& fold) {
  if (solid <= 0) return;
  auto go = [&](auto tag, auto lds) {
    typedef decltype(tag) K;
    const typename K::Prm p{solid, alpha, beta, fold, m_uni, cs_uni, IntegratePrm{}};
    launch_pair<K, lds()>(s, ntiles(solid), f, tl, p);
  };
  const std::true_type yes;
  const std::false_type no;
  if (f.arec64u)
    beta != 0.0 ? go(AccelD<true, true, true>{}, yes) : go(AccelD<true, false, true>{}, yes);
  else if (uh)
    beta != 0.0 ? go(AccelD<true, true>{}, no) : go(AccelD<true, false>{}, no);
  else
    beta != 0.0 ? go(AccelD<false, true>{}, no) : go(AccelD<false, false>{}, no);
}
void launch_accel_integrate_tiled(hipStream_t s, const Fields& f, const TileLists& tl, int solid,
                                  double alpha, double beta, double m_uni, double cs_uni,
                                  double dt, const BcTable& bc, const IntegrateOut& out,
                                  const int* contacts, const StatsFold& fold) {
  if (solid <= 0) return;
  auto go = [&](auto tag) {
    typedef decltype(tag) K;
    launch_pair<K>(s, ntiles(solid), f, tl,
                   typename K::Prm{solid, alpha, beta, fold, m_uni, cs_uni,
                                   IntegratePrm{dt, bc, Frame32{}, out, contacts}});
  };
  beta != 0.0 ? go(AccelD<true, true, true, true>{}) : go(AccelD<true, false, true, true>{});
}
// uc: every particle has the same h and sound speed cs_uni
template <bool IT>
static void accel_mixed(hipStream_t s, const Fields& f, const TileLists& tl, int solid,
                        double alpha, double beta, float cs32, bool uh, bool uc, double cs_uni,
                        const IntegratePrm& ip, const StatsFold& fold) {
  if (solid <= 0) return;
  auto go = [&](auto tag, auto lds) {
    typedef decltype(tag) K;
    launch_pair<K, lds()>(s, ntiles(solid), f, tl,
                          typename K::Prm{solid, (float)alpha, (float)beta, cs32, ip, fold,
                                          (float)cs_uni});
  };
  const std::true_type yes;
  const std::false_type no;
  if (uc)
    beta != 0.0 ? go(AccelG<true, true, IT, true>{}, yes) : go(AccelG<true, false, IT, true>{}, yes);
  else if (uh)
    beta != 0.0 ? go(AccelG<true, true, IT>{}, no) : go(AccelG<true, false, IT>{}, no);
  else
    beta != 0.0 ? go(AccelG<false, true, IT>{}, no) : go(AccelG<false, false, IT>{}, no);
}
void launch_accel_integrate_mixed(hipStream_t s, const Fields& f, const TileLists& tl, int solid,
                                  double alpha, double beta, float cs32, bool uh, bool uc,
                                  double cs_uni, double dt, const BcTable& bc, const Frame32& fr,
                                  const IntegrateOut& out, const int* contacts,
                                  const StatsFold& fold) {
  accel_mixed<true>(s, f, tl, solid, alpha, beta, cs32, uh, uc, cs_uni,
                    IntegratePrm{dt, bc, fr, out, contacts}, fold);
}
void launch_cond_tiled(hipStream_t s, const Fields& f, const TileLists& tl, int n, double T_inf,
                       double h_conv, double dt, bool leap, bool first, bool uh, bool keep) {
  if (n <= 0) return;
  launch_gather<CondD>(s, f, tl, ntiles(n), uh, n, T_inf, h_conv, dt, leap ? 1 : 0,
                       first ? 1 : 0, keep ? 0 : 1);
}
void launch_dens_mixed(hipStream_t s, const Fields& f, const TileLists& tl, int n, int solid,
                       double dt, bool fuse, float cs32, bool uh) {
  if (n <= 0) return;
  launch_gather<DensG>(s, f, tl, ntiles(n), uh, solid, n, dt, fuse ? 1 : 0, cs32);
}
void launch_rates_mixed(hipStream_t s, const Fields& f, const TileLists& tl, int solid,
                        int quirks, float cs32, bool uh, const SurfaceArgs* sf) {
  if (solid <= 0) return;
  const double xz = xz_sign(quirks);
  if (sf) {
    typedef RatesG<true, true> K;
    const SurfPrm<float> sp{sf->id_free_surf, sf->ntot, sf->totmass, (float)sf->r2cut,
                            (float)sf->m};
    launch_pair<K>(s, ntiles(solid), f, tl, K::Prm{solid, xz, cs32, sp});
  } else {
    launch_gather<RatesGU>(s, f, tl, ntiles(solid), uh, solid, xz, cs32, SurfPrm<float>{});
  }
}
// The Newton return map is a long dependent chain that only half of the
// workgroup's wavefronts run, so with more workgroups than one round of three
// a CU the separate pass, all lanes busy and three wavefronts a SIMD, hides it
// better.  Step, us, separate -> fused: Johnson-Cook FP64 at 147 tiles 48.0 ->
// 45.2, 736 tiles 92.9 -> 91.0, 1,489 tiles 150.8 -> 154.7, 5,931 tiles 594 ->
// 617; mixed 34.9 -> 33.0, 60.1 -> 58.1, 94.8 -> 99.2, 351 -> 386; bilinear
// FP64 at 16 tiles 27.5 -> 25.5, 162 tiles 42.2 -> 39.3, 1,598 tiles 152.7 ->
// 149.1, and with what only a caller reads unstored (StepParams::keep) 6,515
// tiles 570.7 -> 557.5.
int rates_stress_blocks(int solid, bool jc_newton) {
  const int nt = ntiles(solid), split = pair_split(nt);
  if (jc_newton && (nt > 768 || kTileP / split < 64)) return 0;
  return nt * split;
}
void launch_rates_stress(hipStream_t s, const Fields& f, const TileLists& tl, bool mixed,
                         float cs32, const SurfaceArgs* sf, const StepParams& sp, BlockStats* bs,
                         const RetArgs& ra) {
  const int solid = sp.solid;
  if (solid <= 0) return;
  const double xz = xz_sign(sp.quirks);
  auto go = [&](auto tag, const auto& rp) {
    typedef decltype(tag) K;
    typename K::Prm p;
    static_cast<std::decay_t<decltype(rp)>&>(p) = rp;
    p.sp = sp;
    p.ra = ra;
    p.bs = bs;
    launch_pair<K>(s, ntiles(solid), f, tl, p);
  };
  auto pick = [&](auto rates, auto mx, const auto& rp) {
    typedef decltype(rates) R;
    if constexpr (mx()) {
      go(RatesStress<R, kRec32, true, false>{}, rp);
    } else {
      if (pair_split(ntiles(solid)) > 1) go(RatesStress<R, kRec64, false, true>{}, rp);
      else go(RatesStress<R, kRec64, false, false>{}, rp);
    }
  };
  const std::true_type yes;
  const std::false_type no;
  if (mixed) {
    SurfPrm<float> sp32{};
    if (sf) sp32 = {sf->id_free_surf, sf->ntot, sf->totmass, (float)sf->r2cut, (float)sf->m};
    if (sf) pick(RatesG<true, true>{}, yes, RatesG<true, true>::Prm{solid, xz, cs32, sp32});
    else pick(RatesG<true>{}, yes, RatesG<true>::Prm{solid, xz, cs32, sp32});
  } else {
    SurfPrm<double> sp64{};
    if (sf) sp64 = {sf->id_free_surf, sf->ntot, sf->totmass, sf->r2cut, sf->m};
    if (sf) pick(RatesD<true, true>{}, no, RatesD<true, true>::Prm{solid, xz, sp64});
    else pick(RatesD<true>{}, no, RatesD<true>::Prm{solid, xz, sp64});
  }
}
void launch_accel_mixed(hipStream_t s, const Fields& f, const TileLists& tl, int solid,
                        double alpha, double beta, float cs32, bool uh, bool uc, double cs_uni,
                        const StatsFold& fold) {
  accel_mixed<false>(s, f, tl, solid, alpha, beta, cs32, uh, uc, cs_uni, IntegratePrm{}, fold);
}
void launch_cond_mixed(hipStream_t s, const Fields& f, const TileLists& tl, int n, double T_inf,
                       double h_conv, double dt, bool leap, bool first, float cs32, bool uh,
                       bool keep) {
  if (n <= 0) return;
  launch_gather<CondG>(s, f, tl, ntiles(n), uh, n, T_inf, h_conv, dt, leap ? 1 : 0,
                       first ? 1 : 0, cs32, keep ? 0 : 1);
}
void launch_cond_dens_tiled(hipStream_t s, const Fields& f, const TileLists& tl, int n,
                            int solid, double T_inf, double h_conv, double dt, bool leap,
                            bool first, bool uh, const unsigned long long* pz_d2,
                            double pz_skin2, bool keep, bool keep_next) {
  if (n <= 0) return;
  auto go = [&](auto tag, auto split) {
    typedef decltype(tag) K;
    const typename K::Prm p{n, {n, T_inf, h_conv, dt, leap ? 1 : 0, first ? 1 : 0, keep ? 0 : 1},
                            {solid, n, dt, 1, 1, keep_next ? 0 : 1}, pz_d2, pz_skin2};
    launch_pair<K, split()>(s, ntiles(n), f, tl, p);
  };
  if (uh) go(CondDensD<true>{}, std::true_type{});
  else go(CondDensD<false>{}, std::false_type{});
}
void launch_cond_dens_mixed(hipStream_t s, const Fields& f, const TileLists& tl, int n,
                            int solid, double T_inf, double h_conv, double dt, bool leap,
                            bool first, float cs32, bool uh, const unsigned long long* pz_d2,
                            double pz_skin2, bool keep, bool keep_next) {
  if (n <= 0) return;
  auto go = [&](auto tag, auto split) {
    typedef decltype(tag) K;
    const typename K::Prm p{
        n, {n, T_inf, h_conv, dt, leap ? 1 : 0, first ? 1 : 0, cs32, keep ? 0 : 1},
        {solid, n, dt, 1, cs32, 1, keep_next ? 0 : 1}, pz_d2, pz_skin2};
    launch_pair<K, split()>(s, ntiles(n), f, tl, p);
  };
  if (uh) go(CondDensG<true>{}, std::true_type{});
  else go(CondDensG<false>{}, std::false_type{});
}
}  // namespace wf
