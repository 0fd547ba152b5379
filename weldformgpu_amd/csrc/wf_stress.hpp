// wf_stress.hpp — the stress update of one particle (pressure, Jaumann rate,
// return map, energy, neighbour records) as the stress kernel and the rates
// pass that finishes its own particles both run it.
#pragma once
#include "wf_mlp.hpp"

namespace wf {

struct T9 {
  double xx, xy, xz, yx, yy, yz, zx, zy, zz;
};

// tensor3 operator*, tensor3.cu:241-255 as written (first column A*B, the
// others A*B^T) or the true product.
__device__ __forceinline__ T9 tmul(const T9& a, const T9& b, bool quirk) {
  T9 r;
  r.xx = a.xx * b.xx + a.xy * b.yx + a.xz * b.zx;
  r.yx = a.yx * b.xx + a.yy * b.yx + a.yz * b.zx;
  r.zx = a.zx * b.xx + a.zy * b.yx + a.zz * b.zx;
  if (quirk) {
    r.xy = a.xx * b.yx + a.xy * b.yy + a.xz * b.yz;
    r.xz = a.xx * b.zx + a.xy * b.zy + a.xz * b.zz;
    r.yy = a.yx * b.yx + a.yy * b.yy + a.yz * b.yz;
    r.yz = a.yx * b.zx + a.yy * b.zy + a.yz * b.zz;
    r.zy = a.zx * b.yx + a.zy * b.yy + a.zz * b.yz;
    r.zz = a.zx * b.zx + a.zy * b.zy + a.zz * b.zz;
  } else {
    r.xy = a.xx * b.xy + a.xy * b.yy + a.xz * b.zy;
    r.xz = a.xx * b.xz + a.xy * b.yz + a.xz * b.zz;
    r.yy = a.yx * b.xy + a.yy * b.yy + a.yz * b.zy;
    r.yz = a.yx * b.xz + a.yy * b.yz + a.yz * b.zz;
    r.zy = a.zx * b.xy + a.zy * b.yy + a.zz * b.zy;
    r.zz = a.zx * b.xz + a.zy * b.yz + a.zz * b.zz;
  }
  return r;
}

// particle i's FP64 acceleration record from s = sigma/rho^2, in the layout
// in force (the general one's {v, m} is written by the caller)
__device__ __forceinline__ void accel_record64(const Fields& f, int i, double s0, double s1,
                                               double s2, double s3, double s4, double s5,
                                               double rho, double cs) {
  if (f.arec64u) {
    f.arec64u[i] = make_double4(s0, s1, rho, 0.0);
    f.arec64[i] = make_double4(s2, s3, s4, s5);
  } else {
    f.arec64[rec_at(f, i, 1)] = make_double4(s0, s1, s2, s3);
    f.arec64[rec_at(f, i, 2)] = make_double4(s4, s5, rho, cs);
  }
}

// Safeguarded Newton for the Johnson-Cook radial return,
// r(g) = s_trial - 3G g - (A + B (ep+g)^n) rt = 0 on [0, hi], from g0, with
// rt = rate factor x thermal factor and hi = (s_trial - s_y(ep)) / (3G).
// On convergence *xn holds (ep+g)^n of the returned g (the final yield
// stress needs it), else it is left alone.
__device__ __forceinline__ double jc_newton(const MatParams& mp, double s_trial, double G,
                                            double ep, double rt, double hi, double g0,
                                            double tol, int max_iter, int* iters, double* xn_out) {
  double lo = 0.0;
  if (!(hi > 0.0)) {
    *iters = 0;
    return 0.0;
  }
  double g = g0;
  if (!(g > lo) || !(g < hi)) g = (g0 >= hi) ? hi : lo;
  int it = 0;
  for (; it < max_iter; it++) {
    // one pow per iterate: s_y = (A + B x^n) rt, H = n B x^n / x rt
    const double x = ep + g;
    const double xn = pow(x, mp.n);
    const double r = s_trial - 3.0 * G * g - (mp.A + mp.B * xn) * rt;
    if (fabs(r) <= tol * s_trial) {
      *xn_out = xn;
      break;
    }
    if (r > 0.0) lo = g;
    else hi = g;
    const double H = x > 0.0 ? mp.n * mp.B * (xn / x) * rt : HUGE_VAL;
    double gn = g + r / (3.0 * G + H);
    if (!(gn > lo && gn < hi)) gn = 0.5 * (lo + hi);
    g = gn;
  }
  *iters = it;
  return g;
}

// What the stress update reads of its particle, so that a pass may load it
// ahead.  Everything is read before the update's first store: the stores
// could alias the fields, so a read behind one waits for its own trip to
// memory.  Eleven trips in a row before, the strain's six among them: a
// 759k-particle Johnson-Cook step went from 601 to 594 us (FP64) and from
// 361 to 351 us (mixed).
struct StressIn {
  double rho, cs, p, G, T, sigma_y, ep, m, eint;  // p: rho0 with FUSE_P
  double strain[6], s[6];
};
template <bool FUSE_P, bool ENERGY, bool S32>
__device__ __forceinline__ void stress_load(const Fields& f, const StepParams& p, int i,
                                            StressIn& in) {
  in.rho = f.rho[i];
  in.cs = p.uniform ? p.Cs : f.Cs[i];
  in.p = !FUSE_P ? f.p[i] : p.uniform ? p.rho0 : f.rho0[i];
  in.G = p.uniform ? p.G : f.G[i];
  in.T = f.T[i];
  in.sigma_y = f.sigma_y[i];
  in.ep = f.pl_strain[i];
#pragma unroll
  for (int k = 0; k < 6; k++) in.strain[k] = f.strain[k][i];
  if (ENERGY) {
    in.m = p.uniform ? p.m : f.m[i];
    in.eint = f.eint[i];
  }
#pragma unroll
  for (int k = 0; k < 6; k++) in.s[k] = S32 ? (double)f.ss32[k][i] : f.ss[k][i];
}

// ---------------------------------------------------------------------------
// C: Jaumann stress update + return map, StressStrainOne (Mechanical.cu:458-554),
// optionally with the pressure (FUSE_P), the per-particle internal-energy
// increment (ENERGY, Energy.cu:5-19 with per-particle indexing) and the
// packed FP32 or FP64 neighbour records of the pair loops (REC).
//
// The Johnson-Cook Newton return map (an extension: the reference re-evaluates
// the yield stress explicitly, Mechanical.cu:504-508) is solved in place, in
// three phases per wavefront: every lane forms its elastic predictor; if any
// lane yields, the whole wavefront evaluates the surrogate MLP on its 64
// feature rows (BF16 MFMA, wf_mlp.hpp) for an initial plastic increment and
// the yielding lanes run the FP64 Newton from it (from 0 without the
// surrogate) to the same residual; then every lane finishes and writes its
// state once.  The solved increment is logged as a training sample.
// S32: sigma, the deviatoric stress and the rates are stored in FP32
// (mixed precision); the arithmetic is FP64 either way.
//
// Whole wavefronts must call it (the surrogate's matrix instructions take all
// 64 lanes); lanes without a particle pass active = false.  rates(d, w) gives
// the particle's strain rate (xx yy zz xy yz xz) and rotation rate (xy yz xz);
// st receives its share of the block statistics (wave_iters: unset).
// in: what stress_load read of it.
template <bool FUSE_P, bool ENERGY, int REC, bool S32, class RATES>
__device__ __forceinline__ void stress_particle(const Fields& f, const StepParams& p,
                                                const RetArgs& ra, int i, bool active,
                                                const StressIn& in, const RATES& rates,
                                                BlockStats& st) {
  st = BlockStats{0ull, 0ull, 0ull, 0ull};
  const MatParams& mp = p.mat;
  const double dt = p.dt;
  T9 S{}, D{};
  double sig_trial = 0.0, sigy = 0.0, ep = 0.0, sigeq = 0.0, dep = 0.0, scale = 1.0;
  double esr = 0.0, T = 0.0, rt = 1.0, gmax = 0.0;
  double G = 0.0, rho_i = 0.0, cs_i = 0.0, p_i = 0.0, m_i = 0.0, eint = 0.0;
  bool newton = false;  // a yielding Johnson-Cook particle under the Newton return map
  if (active) {
    const bool qp = (p.quirks & WF_Q_TENSOR_PRODUCT) != 0;
    rho_i = in.rho;
    cs_i = in.cs;
    p_i = in.p;
    G = in.G;
    T = in.T;
    sigy = in.sigma_y;
    ep = in.ep;
    if (ENERGY) {
      m_i = in.m;
      eint = in.eint;
    }
    S.xx = in.s[0]; S.yy = in.s[1]; S.zz = in.s[2];
    S.xy = S.yx = in.s[3]; S.yz = S.zy = in.s[4]; S.xz = S.zx = in.s[5];
    double d6[6], w3[3];
    rates(d6, w3);
    D.xx = d6[0]; D.yy = d6[1]; D.zz = d6[2];
    D.xy = D.yx = d6[3]; D.yz = D.zy = d6[4]; D.xz = D.zx = d6[5];
    T9 W;
    W.xx = W.yy = W.zz = 0.0;  // antisymmetric
    W.xy = w3[0]; W.yz = w3[1]; W.xz = w3[2];
    W.yx = -W.xy; W.zy = -W.yz; W.zx = -W.xz;
#pragma unroll
    for (int k = 0; k < 6; k++) f.strain[k][i] = in.strain[k] + d6[k] * dt;
    if (FUSE_P) {
      p_i = 0.0 + (cs_i * cs_i) * (rho_i - p_i);
    }
    T9 WT = {W.xx, W.yx, W.zx, W.xy, W.yy, W.zy, W.xz, W.yz, W.zz};
    T9 SRT = tmul(S, WT, qp);
    T9 RS = tmul(W, S, qp);
    if (REC == kRec64 && !f.arec64u)
      f.arec64[rec_at(f, i, 0)] = make_double4(f.v[0][i], f.v[1][i], f.v[2][i], f.m[i]);
    const double tr3 = 1.0 / 3.0 * (D.xx + D.yy + D.zz);
    const double g2 = 2.0 * G;
    // S = dt*(2G(D - tr/3 I) + SRT + RS) + S   (Mechanical.cu:490)
    S.xx = ((D.xx - tr3) * g2 + SRT.xx + RS.xx) * dt + S.xx;
    S.yy = ((D.yy - tr3) * g2 + SRT.yy + RS.yy) * dt + S.yy;
    S.zz = ((D.zz - tr3) * g2 + SRT.zz + RS.zz) * dt + S.zz;
    S.xy = (D.xy * g2 + SRT.xy + RS.xy) * dt + S.xy;
    S.yx = (D.yx * g2 + SRT.yx + RS.yx) * dt + S.yx;
    S.xz = (D.xz * g2 + SRT.xz + RS.xz) * dt + S.xz;
    S.zx = (D.zx * g2 + SRT.zx + RS.zx) * dt + S.zx;
    S.yz = (D.yz * g2 + SRT.yz + RS.yz) * dt + S.yz;
    S.zy = (D.zy * g2 + SRT.zy + RS.zy) * dt + S.zy;

    esr = sqrt(0.5 * ((D.xx - D.yy) * (D.xx - D.yy) + (D.yy - D.zz) * (D.yy - D.zz) +
                      (D.zz - D.xx) * (D.zz - D.xx)) +
               3.0 * (D.xy * D.xy + D.yz * D.yz + D.zx * D.zx));
    const double J2 = 0.5 * (S.xx * S.xx + 2.0 * S.xy * S.yx + 2.0 * S.xz * S.zx +
                             S.yy * S.yy + 2.0 * S.yz * S.zy + S.zz * S.zz);
    sig_trial = sqrt(3.0 * J2);
    sigeq = sig_trial;
    if (p.return_map == WF_RETURN_REFERENCE) {
      if (sigy < sig_trial) scale = sigy / sig_trial;
      if (mp.model == WF_MAT_HOLLOMON) sigy = hollomon_yield(mp, ep);
      else if (mp.model == WF_MAT_JOHNSON_COOK)
        sigy = jc_yield(mp, ep, jc_rate_factor(mp, esr), 1.0 - pow(jc_theta(mp, T), mp.m));
      if (sig_trial > sigy) {
        dep = (sig_trial - sigy) / (3. * G);
        ep += dep;
        sigeq = sigy;
        if (mp.model == WF_MAT_BILINEAR) sigy += dep * mp.Ep;
      }
    } else {
      double rate_f = 1.0, therm_f = 1.0;
      if (mp.model == WF_MAT_HOLLOMON) sigy = hollomon_yield(mp, ep);
      else if (mp.model == WF_MAT_JOHNSON_COOK) {
        rate_f = jc_rate_factor(mp, esr);
        therm_f = 1.0 - pow(jc_theta(mp, T), mp.m);
        sigy = jc_yield(mp, ep, rate_f, therm_f);
      }
      if (sig_trial > sigy) {
        double g = 0.0;
        if (mp.model == WF_MAT_BILINEAR) {
          g = (sig_trial - sigy) / (3.0 * G + mp.Ep);
          sigy = sigy + mp.Ep * g;
        } else if (mp.model == WF_MAT_JOHNSON_COOK) {
          newton = true;  // solved below, with the rest of the wavefront
          rt = rate_f * therm_f;
          gmax = (sig_trial - sigy) / (3.0 * G);
        } else {
          double lo = 0.0, hi = (sig_trial - sigy) / (3.0 * G);
          for (int it = 0; it < 200; it++) {
            double mid = 0.5 * (lo + hi);
            double r = sig_trial - 3.0 * G * mid - hollomon_yield(mp, ep + mid);
            if (r > 0) lo = mid;
            else hi = mid;
          }
          g = 0.5 * (lo + hi);
          sigy = hollomon_yield(mp, ep + g);
        }
        if (!newton) {
          scale = (sig_trial - 3.0 * G * g) / sig_trial;
          dep = g;
          ep += g;
          sigeq = sig_trial - 3.0 * G * g;
        }
      }
    }
  }
  // wave-uniform: the MFMA needs all 64 lanes
  if (__ballot(newton) != 0ull) {
    float f0, f1, f2, f3;
    mlp_features(newton ? sig_trial : 1.0, mp.A, ep, esr, newton ? jc_theta(mp, T) : 0.0, f0,
                 f1, f2, f3);
    double g0 = 0.0;
    if (ra.use_mlp) {
      MlpWave mw;
      mlp_wave_load_packed((const uint4*)ra.mlp_pack, mw);
      const float y = mlp_wave_eval(mw, f0, f1, f2, f3);
      if (isfinite(y)) g0 = fmin(fmax((double)y, 0.0), 1.0) * gmax;
    }
    if (newton) {
      int it = 0;
      double xn = -1.0;  // (ep+g)^n >= 0 once the Newton has converged
      const double g = jc_newton(mp, sig_trial, G, ep, rt, gmax, g0, p.newton_tol,
                                 p.newton_max_iter, &it, &xn);
      st.iters = (unsigned long long)it;
      st.calls = 1ull;
      scale = (sig_trial - 3.0 * G * g) / sig_trial;
      dep = g;
      sigeq = sig_trial - 3.0 * G * g;
      // training sample (one slot per particle: deterministic)
      f.mlx[0][i] = f0;
      f.mlx[1][i] = f1;
      f.mlx[2][i] = f2;
      f.mlx[3][i] = f3;
      f.mly[i] = gmax > 0.0 ? (float)(g / gmax) : 0.f;
      f.mlstep[i] = (int)ra.step;
      ep += g;  // the same rounding as the Newton's ep + g
      sigy = (mp.A + mp.B * (xn >= 0.0 ? xn : pow(ep, mp.n))) * rt;
    }
  }
  if (active) {
    if (scale != 1.0) {
      S.xx *= scale; S.yy *= scale; S.zz *= scale;
      S.xy *= scale; S.yz *= scale; S.xz *= scale;
    }
    const double sv[6] = {S.xx, S.yy, S.zz, S.xy, S.yz, S.xz};
#pragma unroll
    for (int k = 0; k < 6; k++) {
      if (S32) f.ss32[k][i] = (float)sv[k];
      else f.ss[k][i] = sv[k];
    }
    f.sigma_y[i] = sigy;
    f.pl_strain[i] = ep;
    f.qpl[i] = p.taylor_quinney * sigeq * dep / dt;
    const double pi = p_i;
    // sigma = -p I + S (Mechanical.cu:540); store upper triangle
    const double sg[6] = {-pi + S.xx, -pi + S.yy, -pi + S.zz, S.xy, S.yz, S.xz};
    if (REC == kRec32) {  // sigma/rho^2, rho and Cs for the FP32 acceleration loop
      const double rho = rho_i, ir2 = 1.0 / (rho * rho);
      f.arec[rec32_at(i, 0)] = make_float4((float)(sg[0] * ir2), (float)(sg[1] * ir2),
                                           (float)(sg[2] * ir2), (float)(sg[3] * ir2));
      f.arec[rec32_at(i, 1)] =
          make_float4((float)(sg[4] * ir2), (float)(sg[5] * ir2), (float)rho, (float)cs_i);
    }
    if (REC == kRec64) {  // the same in FP64 for the FP64 acceleration loop
      const double rho = rho_i, ir2 = 1.0 / (rho * rho);
      accel_record64(f, i, sg[0] * ir2, sg[1] * ir2, sg[2] * ir2, sg[3] * ir2, sg[4] * ir2,
                     sg[5] * ir2, rho, cs_i);
    }
    if (ENERGY) {
      double de = m_i / rho_i *
                  (S.xx * D.xx + S.yy * D.yy + S.zz * D.zz +
                   2.0 * (S.xy * D.xy + S.yz * D.yz + S.xz * D.xz));
      f.eint[i] = eint + de * dt;
    }
    // the conditional stores come last: a branch amid the arithmetic changes
    // which products the compiler contracts
    if (p.keep) {
      if (FUSE_P) f.p[i] = p_i;
      f.esr[i] = esr;
      f.sigma_eq[i] = sigeq;
#pragma unroll
      for (int k = 0; k < 6; k++) {
        if (S32) f.sigma32[k][i] = (float)sg[k];
        else f.sigma[k][i] = sg[k];
      }
    }
    st.ep_bits = (unsigned long long)__double_as_longlong(ep > 0.0 ? ep : 0.0);
  }
}

// The workgroup's statistics from its threads' (st, zero in those without a
// particle): nw wavefronts took part (the first ones); wst: LDS for them.
// Every thread of the workgroup must call it.
__device__ __forceinline__ void stress_block_stats(const BlockStats& st, int nw, BlockStats* wst,
                                                   BlockStats* out) {
  const int lane = lane_id(), w = threadIdx.x >> 6;
  if (w < nw) {
    const unsigned long long mx = wave_max_u64(st.ep_bits);
    const unsigned long long sit = wave_sum_u64(st.iters);
    const unsigned long long sc = wave_sum_u64(st.calls);
    const unsigned long long wmax = wave_max_u64(st.iters);
    if (lane == 0) wst[w] = BlockStats{mx, sit, sc, wmax};
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    BlockStats b{0ull, 0ull, 0ull, 0ull};
    for (int u = 0; u < nw; u++) {
      b.ep_bits = wst[u].ep_bits > b.ep_bits ? wst[u].ep_bits : b.ep_bits;
      b.iters += wst[u].iters;
      b.calls += wst[u].calls;
      b.wave_iters += wst[u].wave_iters;
    }
    *out = b;
  }
}

}  // namespace wf
