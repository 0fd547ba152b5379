// wf_kernels.hip — FP64 per-particle kernels of the SPH pipeline (gfx950):
// pressure + Jaumann stress + return map + energy, BC + integration,
// leapfrog, reductions and reorder helpers.  One thread per particle over
// Morton-sorted SoA planes, so every load and store is coalesced.  The pair
// loops are in wf_pair.hip.
#include "wf_stress.hpp"

namespace wf {

static inline int grid_for(int n) { return (n + kBlock - 1) / kBlock; }

__global__ __launch_bounds__(kBlock) void k_update_density(Fields f, int solid, double dt) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < solid) f.rho[i] += dt * f.drho[i];
}

// ---------------------------------------------------------------------------
// Pressure, PressureKernelExt + EOS case 0 (Mechanical.cu:289-298,
// Functions.cu:211-213) with PresEq = P0 = 0.
__global__ __launch_bounds__(kBlock) void k_pressure(Fields f, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) f.p[i] = 0.0 + (f.Cs[i] * f.Cs[i]) * (f.rho[i] - f.rho0[i]);
}

// C: the stress pass, one thread per particle (stress_particle)
template <bool FUSE_P, bool ENERGY, int REC, bool S32>
__global__ __launch_bounds__(kBlock) void k_stress(Fields f, StepParams p, BlockStats* bs,
                                                   RetArgs ra) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  __shared__ BlockStats wst[kBlock / 64];
  auto rates = [&](double (&d)[6], double (&w)[3]) {
#pragma unroll
    for (int k = 0; k < 6; k++) d[k] = S32 ? (double)f.strrate32[k][i] : f.strrate[k][i];
    // the rotation rate's diagonal planes hold zeros
#pragma unroll
    for (int k = 0; k < 3; k++) w[k] = S32 ? (double)f.rotrate32[3 + k][i] : f.rotrate[3 + k][i];
  };
  StressIn in;
  if (i < p.solid) stress_load<FUSE_P, ENERGY, S32>(f, p, i, in);
  BlockStats st;
  stress_particle<FUSE_P, ENERGY, REC, S32>(f, p, ra, i, i < p.solid, in, rates, st);
  stress_block_stats(st, kBlock / 64, wst, bs + blockIdx.x);
}

// Rebuild trigger of WF_REBUILD_PLASTIC_ZONE: the largest squared
// displacement from the last build over the particles with eps_p > ep_hot.
// A max of non-negative doubles is the max of their bit patterns, so the
// result does not depend on the order of the atomics.
__global__ __launch_bounds__(kBlock) void k_hot_disp(Fields f, const double* __restrict__ xb0,
                                                     const double* __restrict__ xb1,
                                                     const double* __restrict__ xb2, int n,
                                                     double ep_hot,
                                                     unsigned long long* d2_bits) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned long long b = 0ull;
  if (i < n && f.pl_strain[i] > ep_hot) {
    const double dx = f.x[0][i] - xb0[i], dy = f.x[1][i] - xb1[i], dz = f.x[2][i] - xb2[i];
    b = (unsigned long long)__double_as_longlong(dx * dx + dy * dy + dz * dz);
  }
  b = wave_max_u64(b);
  if (lane_id() == 0 && b) atomicMax(d2_bits, b);
}

// one block folds the per-block statistics into the run counters (used
// where no acceleration pass follows the stress pass to do it); one
// 256-thread block reading one entry at a time took 20 us for the 10.7k
// blocks of a 2.7M-particle step
constexpr int kFoldThreads = 1024;
__global__ __launch_bounds__(kFoldThreads) void k_fold_stats(const BlockStats* bs, int nb,
                                                             Counters* ctr) {
  __shared__ unsigned long long sh[4 * kFoldThreads / 64];
  block_fold_stats(StatsFold{bs, nb, ctr}, sh);
}

// ---------------------------------------------------------------------------
// F: velocity BCs + UpdatePosFraser + UpdateVel + BCs in one pass
// (SolverFraser.cu:273-281; Mechanical.cu:142-191,572-584)
template <int REC>
__global__ __launch_bounds__(kBlock) void k_integrate(Fields f, int n, double dt, BcTable bc,
                                                     Frame32 fr) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  // in place: each thread reads and writes only its own particle
  const IntegrateOut o{{f.x[0], f.x[1], f.x[2]}, f.p4, f.v4, f.kv, false};
  integrate_particle<REC>(f, i, f.a[0][i], f.a[1][i], f.a[2][i], dt, bc, fr, o);
}

// every FP32 mirror from the FP64 state; the integer cell of each particle is
// (re)chosen here and kept until the next refresh
__global__ __launch_bounds__(kBlock) void k_mirror32(Fields f, int n, Frame32 fr) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int c[3];
  float xr[3];
  for (int a = 0; a < 3; a++) {
    double u = floor((f.x[a][i] - fr.org[a]) / fr.cs);
    int lim = a < 2 ? 2047 : 1023;
    c[a] = (int)fmin(fmax(u, 0.0), (double)lim);
    xr[a] = (float)(f.x[a][i] - (fr.org[a] + c[a] * fr.cs));
  }
  f.p4[i] = make_float4(xr[0], xr[1], xr[2], __int_as_float(pack_cell(c[0], c[1], c[2])));
  const double rho = f.rho[i];
  f.h32[i] = (float)f.h[i];
  const float4 v4 = make_float4((float)f.v[0][i], (float)f.v[1][i], (float)f.v[2][i],
                                (float)(f.m[i] / rho));
  f.v4[i] = v4;
  f.v4_alt[i] = v4;
  const double ir2 = 1.0 / (rho * rho);
  f.arec[rec32_at(i, 0)] =
      make_float4((float)(f.sigma32[0][i] * ir2), (float)(f.sigma32[1][i] * ir2),
                  (float)(f.sigma32[2][i] * ir2), (float)(f.sigma32[3][i] * ir2));
  f.arec[rec32_at(i, 1)] = make_float4((float)(f.sigma32[4][i] * ir2),
                                          (float)(f.sigma32[5][i] * ir2), (float)rho,
                                          (float)f.Cs[i]);
  const float4 tk = make_float4((float)f.T[i], (float)f.k[i], v4.w, 0.f);
  f.tk4[i] = tk;
  f.tk4_alt[i] = tk;
}

// every FP64 neighbour record from the FP64 state
__global__ __launch_bounds__(kBlock) void k_records64(Fields f, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double rho = f.rho[i], mdj = f.m[i] / rho, ir2 = 1.0 / (rho * rho);
  const double4 kv = make_double4(f.v[0][i], f.v[1][i], f.v[2][i], mdj);
  f.kv[i] = kv;
  f.kv_alt[i] = kv;
  if (!f.arec64u)
    f.arec64[rec_at(f, i, 0)] = make_double4(f.v[0][i], f.v[1][i], f.v[2][i], f.m[i]);
  accel_record64(f, i, f.sigma[0][i] * ir2, f.sigma[1][i] * ir2, f.sigma[2][i] * ir2,
                 f.sigma[3][i] * ir2, f.sigma[4][i] * ir2, f.sigma[5][i] * ir2, rho, f.Cs[i]);
  const double4 tk = make_double4(f.T[i], f.k[i], mdj, 0.0);
  f.tk64[i] = tk;
  f.tk64_alt[i] = tk;
}

__global__ __launch_bounds__(kBlock) void k_apply_bc(Fields f, int n, int zone, double vx,
                                                     double vy, double vz) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || f.ID[i] != zone) return;
  f.a[0][i] = 0.0; f.a[1][i] = 0.0; f.a[2][i] = 0.0;
  f.v[0][i] = vx; f.v[1][i] = vy; f.v[2][i] = vz;
  f.va[0][i] = vx; f.va[1][i] = vy; f.va[2][i] = vz;
}

// ApplyAxiSymmBC (Domain_d.cu:665-689): the radial projection computed there
// is overwritten by zeros, so a particle meeting the condition loses its
// in-plane acceleration
__global__ __launch_bounds__(kBlock) void k_axisymm_bc(Fields f, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double ax = f.a[0][i], ay = f.a[1][i];
  if (sqrt(ax * ax + ay * ay) > 1.0e-3 && f.x[0][i] > f.h[i] / 2.0 && ax > 1.0e-2) {
    f.a[0][i] = 0.0;
    f.a[1][i] = 0.0;
  }
}

__global__ __launch_bounds__(kBlock) void k_update_pos(Fields f, int n, double dt) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int c = 0; c < 3; c++) {
    double u_ = f.v[c][i] * dt + ((f.a[c][i] * 0.5) * dt) * dt;
    f.x[c][i] += u_;
    f.u[c][i] += u_;
  }
}

__global__ __launch_bounds__(kBlock) void k_update_vel(Fields f, int n, double dt) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int c = 0; c < 3; c++) f.v[c][i] += f.a[c][i] * dt;
}

__global__ __launch_bounds__(kBlock) void k_leapfrog(Fields f, int n, double dt, int first) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (first) {
    f.Ta[i] = f.T[i] - dt / 2.0 * f.dTdt[i];
  } else {
    f.Tb[i] = f.Ta[i];
    f.Ta[i] += f.dTdt[i] * dt;
    f.T[i] = (f.Ta[i] + f.Tb[i]) / 2.;
  }
}

// Deterministic FP64 sum: fixed-shape block partials, then one block.
__global__ __launch_bounds__(kBlock) void k_sum_partial(const double* v, int n, double* partial) {
  __shared__ double sh[kBlock / 64];
  double acc = 0.0;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) acc += v[i];
  acc = wave_sum_f64(acc);
  if (lane_id() == 0) sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < kBlock / 64; w++) t += sh[w];
    partial[blockIdx.x] = t;
  }
}
__global__ void k_sum_final(const double* partial, int nb, double* out) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    double t = 0.0;
    for (int b = 0; b < nb; b++) t += partial[b];
    *out = t;
  }
}

// ---- generic reorder helpers ----------------------------------------------
__global__ void k_gather_f64(double* dst, const double* src, const int* idx, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[idx[i]];
}
__global__ void k_gather_i32(int* dst, const int* src, const int* idx, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[idx[i]];
}
__global__ void k_scatter_f64(double* dst, const double* src, const int* idx, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[idx[i]] = src[i];
}
__global__ void k_scatter_i32(int* dst, const int* src, const int* idx, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[idx[i]] = src[i];
}
__global__ void k_fill_f64(double* dst, double v, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = v;
}

// ---- launchers --------------------------------------------------------------
void launch_update_density(hipStream_t s, const Fields& f, const StepParams& p, double dt) {
  if (p.solid <= 0) return;
  hipLaunchKernelGGL(k_update_density, dim3(grid_for(p.solid)), dim3(kBlock), 0, s, f, p.solid,
                     dt);
}
void launch_pressure(hipStream_t s, const Fields& f, const StepParams& p) {
  if (p.n <= 0) return;
  hipLaunchKernelGGL(k_pressure, dim3(grid_for(p.n)), dim3(kBlock), 0, s, f, p.n);
}
template <bool S32>
static void launch_stress_t(hipStream_t s, const Fields& f, const StepParams& p,
                            BlockStats* bs, bool fuse_pressure, bool energy, int rec,
                            const RetArgs& ra) {
  dim3 g(grid_for(p.solid)), b(kBlock);
  if (rec == kRec32)
    hipLaunchKernelGGL((k_stress<true, true, kRec32, true>), g, b, 0, s, f, p, bs, ra);
  else if (rec == kRec64)
    hipLaunchKernelGGL((k_stress<true, true, kRec64, false>), g, b, 0, s, f, p, bs, ra);
  else if (fuse_pressure && energy)
    hipLaunchKernelGGL((k_stress<true, true, kRecNone, S32>), g, b, 0, s, f, p, bs, ra);
  else if (fuse_pressure)
    hipLaunchKernelGGL((k_stress<true, false, kRecNone, S32>), g, b, 0, s, f, p, bs, ra);
  else if (energy)
    hipLaunchKernelGGL((k_stress<false, true, kRecNone, S32>), g, b, 0, s, f, p, bs, ra);
  else
    hipLaunchKernelGGL((k_stress<false, false, kRecNone, S32>), g, b, 0, s, f, p, bs, ra);
}
void launch_stress(hipStream_t s, const Fields& f, const StepParams& p, BlockStats* bs,
                   bool fuse_pressure, bool energy, int rec, bool s32, const RetArgs& ra) {
  if (p.solid <= 0) return;
  if (s32) launch_stress_t<true>(s, f, p, bs, fuse_pressure, energy, rec, ra);
  else launch_stress_t<false>(s, f, p, bs, fuse_pressure, energy, rec, ra);
}
void launch_hot_disp(hipStream_t s, const Fields& f, const double* const xb[3], int n,
                     double ep_hot, unsigned long long* d2_bits) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_hot_disp, dim3(grid_for(n)), dim3(kBlock), 0, s, f, xb[0], xb[1], xb[2],
                     n, ep_hot, d2_bits);
}
void launch_fold_stats(hipStream_t s, const BlockStats* bs, int nblocks, Counters* ctr) {
  if (nblocks <= 0) return;
  hipLaunchKernelGGL(k_fold_stats, dim3(1), dim3(kFoldThreads), 0, s, bs, nblocks, ctr);
}
void launch_apply_bc(hipStream_t s, const Fields& f, int n, int zone, double vx, double vy,
                     double vz) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_apply_bc, dim3(grid_for(n)), dim3(kBlock), 0, s, f, n, zone, vx, vy, vz);
}
void launch_axisymm_bc(hipStream_t s, const Fields& f, int n) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_axisymm_bc, dim3(grid_for(n)), dim3(kBlock), 0, s, f, n);
}
void launch_update_pos(hipStream_t s, const Fields& f, int n, double dt) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_update_pos, dim3(grid_for(n)), dim3(kBlock), 0, s, f, n, dt);
}
void launch_update_vel(hipStream_t s, const Fields& f, int n, double dt) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_update_vel, dim3(grid_for(n)), dim3(kBlock), 0, s, f, n, dt);
}
void launch_integrate(hipStream_t s, const Fields& f, int n, double dt, const BcTable& bc,
                      int rec, const Frame32& fr) {
  if (n <= 0) return;
  const dim3 g(grid_for(n)), b(kBlock);
  if (rec == kRec32)
    hipLaunchKernelGGL(k_integrate<kRec32>, g, b, 0, s, f, n, dt, bc, fr);
  else if (rec == kRec64)
    hipLaunchKernelGGL(k_integrate<kRec64>, g, b, 0, s, f, n, dt, bc, fr);
  else
    hipLaunchKernelGGL(k_integrate<kRecNone>, g, b, 0, s, f, n, dt, bc, fr);
}
void launch_records64(hipStream_t s, const Fields& f, int n) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_records64, dim3(grid_for(n)), dim3(kBlock), 0, s, f, n);
}
void launch_mirror32(hipStream_t s, const Fields& f, int n, const Frame32& fr) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_mirror32, dim3(grid_for(n)), dim3(kBlock), 0, s, f, n, fr);
}
void launch_leapfrog(hipStream_t s, const Fields& f, int n, double dt, bool first) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_leapfrog, dim3(grid_for(n)), dim3(kBlock), 0, s, f, n, dt, first ? 1 : 0);
}
void launch_sum(hipStream_t s, const double* v, int n, double* partial, int nblocks,
                double* out) {
  hipLaunchKernelGGL(k_sum_partial, dim3(nblocks), dim3(kBlock), 0, s, v, n, partial);
  hipLaunchKernelGGL(k_sum_final, dim3(1), dim3(64), 0, s, partial, nblocks, out);
}
void launch_gather_f64(hipStream_t s, double* dst, const double* src, const int* idx, int n) {
  if (n > 0) hipLaunchKernelGGL(k_gather_f64, dim3(grid_for(n)), dim3(kBlock), 0, s, dst, src, idx, n);
}
void launch_gather_i32(hipStream_t s, int* dst, const int* src, const int* idx, int n) {
  if (n > 0) hipLaunchKernelGGL(k_gather_i32, dim3(grid_for(n)), dim3(kBlock), 0, s, dst, src, idx, n);
}
void launch_scatter_f64(hipStream_t s, double* dst, const double* src, const int* idx, int n) {
  if (n > 0) hipLaunchKernelGGL(k_scatter_f64, dim3(grid_for(n)), dim3(kBlock), 0, s, dst, src, idx, n);
}
void launch_scatter_i32(hipStream_t s, int* dst, const int* src, const int* idx, int n) {
  if (n > 0) hipLaunchKernelGGL(k_scatter_i32, dim3(grid_for(n)), dim3(kBlock), 0, s, dst, src, idx, n);
}
void launch_fill_f64(hipStream_t s, double* dst, double v, int n) {
  if (n > 0) hipLaunchKernelGGL(k_fill_f64, dim3(grid_for(n)), dim3(kBlock), 0, s, dst, v, n);
}

}  // namespace wf
