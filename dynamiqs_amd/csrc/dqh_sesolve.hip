// Schrodinger equation d psi / dt = -i H(t) psi (sesolve) with adaptive Tsit5 or
// Dopri5, for gfx950. k_sesolve: any Hamiltonian; k_sesolve_const (below): constant ones
// up to n = 128.
//
// One workgroup integrates one instance (its own adaptive step): one wave for
// np <= 64, four waves up to np = 1024. The FP64 state, the FP32 stage input and the
// seven FP32 stages live in LDS. The vector field is a GEMV with G = -i H read as
// G^T (stored transposed, so that consecutive rows are consecutive addresses) from
// global memory, where a batch that shares H finds it in L2. In the one-wave
// kernel each row is split over 64 / np lane groups (strided columns) and reduced
// with cross-lane shuffles, so that every lane works for np = 16 and 32; the
// four-wave kernel gives each thread whole rows. Piecewise-constant and modulated
// terms are separate products combined with their coefficients in FP64. The
// controller, error norm (RMS over the n entries), FSAL, step snapping, jump
// handling and dense-output saves are those of the mesolve kernels.
#include <hip/hip_runtime.h>

#include <cmath>
#include <string>

#include "dqh.h"
#include "dqh_common.h"
#include "dqh_mfma.h"
#include "dqh_tsit5_tableau.h"
#include "dqh_wave.h"

namespace dqh {
namespace se {

// workgroup size T (one wave or four)
template <int T>
struct SeCfg {
  static constexpr int kW = T / 64;
};

template <int T>
__device__ __forceinline__ double bsum(double v, double *red) {
  constexpr int kW = SeCfg<T>::kW;
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < kW; ++w) s += red[w];
  return s;
}

__device__ __forceinline__ int segment_of(const double *times, int nseg, double t) {
  int lo = 0, hi = nseg;  // searchsorted(times, t, 'right') - 1
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (times[mid] <= t)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo - 1;
}

// coefficients of the time-dependent terms: PWC values of segment seg (zero outside)
// and the modulated f_j(tau) from their piecewise-cubic tables. The loops have
// compile-time bounds so that the coefficients stay in registers.
struct Coef {
  double2 c[8 + DQH_MAX_MOD];
  int npwc, nmod;
};

__device__ __forceinline__ void coefficients(const dqh_me_inst &p, int seg, double tau, Coef &cf) {
  cf.npwc = (int)p.npwc;
  cf.nmod = (int)p.nmod;
  const int nv = (int)p.nseg - 1;
  const double *vals = gp<const double>(p.pwc_vals);
  const bool inside = seg >= 0 && seg < nv;
#pragma unroll
  for (int j = 0; j < 8; ++j)
    cf.c[j] = (j < cf.npwc && inside) ? make_double2(vals[2 * (j * nv + seg)], vals[2 * (j * nv + seg) + 1])
                                      : make_double2(0.0, 0.0);
  if (cf.nmod > 0) {
    const int64_t nint = p.mod_nint;
    int64_t i = (int64_t)floor((tau - p.mod_t0) / p.mod_dt);
    i = i < 0 ? 0 : (i >= nint ? nint - 1 : i);
    const double x = tau - (p.mod_t0 + (double)i * p.mod_dt);
    const double2 *tab = gp<const double2>(p.mod_coef);
#pragma unroll
    for (int j = 0; j < DQH_MAX_MOD; ++j) {
      double re = 0.0, im = 0.0;
      if (j < cf.nmod) {
        const double2 *q = tab + ((size_t)j * nint + i) * 4;
        re = q[0].x;
        im = q[0].y;
        for (int m = 1; m < 4; ++m) {
          re = re * x + q[m].x;
          im = im * x + q[m].y;
        }
      }
      cf.c[8 + j] = make_double2(re, im);
    }
  }
}

// sum over j = j0, j0 + js, ... of M[i][j] ys[j] with M^T stored, so that
// consecutive rows (lanes) read consecutive elements (FP32 products and sums)
__device__ __forceinline__ float2 row_dot(const float2 *MT, int np, int i, const float2 *ys, int j0, int js) {
  float ar = 0.f, ai = 0.f;
  for (int j = j0; j < np; j += js) {
    const float2 g = MT[(size_t)j * np + i];
    const float2 v = ys[j];
    ar = fmaf(g.x, v.x, fmaf(-g.y, v.y, ar));
    ai = fmaf(g.x, v.y, fmaf(g.y, v.x, ai));
  }
  return make_float2(ar, ai);
}

// out = G(t) ys, G = -i H(t) = G0 + sum_k c_k G_k: one product per term, combined
// with the coefficients in FP64. G0^T is p.Hnh, the PWC terms' p.Hpwc and the
// modulated terms' p.Hmod. Lane group q of the one-wave kernel sums the columns
// j = q (mod 64 / np) of row i; the groups are reduced with shuffles.
template <int T>
__device__ __forceinline__ void field(const dqh_me_inst &p, const Coef &cf, const float2 *ys, float2 *out) {
  const int np = (int)p.np;
  const size_t nn = (size_t)np * np;
  const float2 *G0 = gp<const float2>(p.Hnh);
  const float2 *Gp = gp<const float2>(p.Hpwc);
  const float2 *Gm = gp<const float2>(p.Hmod);
  const int nq = T == 64 ? 64 / np : 1;  // np <= 64 in the one-wave kernel
  const int q = T == 64 ? (int)threadIdx.x / np : 0;
  for (int i0 = 0; i0 < np; i0 += T) {
    const int i = T == 64 ? (int)threadIdx.x - q * np : i0 + (int)threadIdx.x;
    const bool row = q < nq && i < np;
    double re = 0.0, im = 0.0;
    if (row) {
      const float2 a = row_dot(G0, np, i, ys, q, nq);
      re = a.x;
      im = a.y;
#pragma unroll
      for (int k = 0; k < 8 + DQH_MAX_MOD; ++k) {
        const bool on = k < 8 ? k < cf.npwc : k - 8 < cf.nmod;
        const double2 c = cf.c[k];
        if (on && (c.x != 0.0 || c.y != 0.0)) {
          const float2 r = row_dot(k < 8 ? Gp + (size_t)k * nn : Gm + (size_t)(k - 8) * nn, np, i, ys, q, nq);
          re += c.x * r.x - c.y * r.y;
          im += c.x * r.y + c.y * r.x;
        }
      }
    }
    if (T == 64) {
      for (int o = np; o < np * nq; o <<= 1) {
        re += __shfl_xor(re, o, 64);
        im += __shfl_xor(im, o, 64);
      }
    }
    if (row && q == 0) out[i] = make_float2((float)re, (float)im);
  }
  __syncthreads();
}

// save y + h sum_j w_j k_j (state and <psi|E|psi>) at save index isave
template <int T, int MAXNP>
__device__ void save_at(const dqh_me_inst &p, const double2 *y, float2 (*k)[MAXNP], double h, const double *w,
                        bool interp, int isave, double2 *v, double *red) {
  const int n = (int)p.n, np = (int)p.np, nE = (int)p.nE, ntsave = (int)p.ntsave;
  for (int i = threadIdx.x; i < np; i += T) {
    double re = y[i].x, im = y[i].y;
    if (interp)
      for (int j = 0; j < 7; ++j) {
        re += h * w[j] * k[j][i].x;
        im += h * w[j] * k[j][i].y;
      }
    v[i] = make_double2(re, im);
    if ((p.flags & DQH_FLAG_SAVE_STATES) && i < n)
      gp<float2>(p.states)[(size_t)isave * n + i] = make_float2((float)re, (float)im);
  }
  __syncthreads();
  const float2 *ET = gp<const float2>(p.EopsT);
  for (int qe = 0; qe < nE; ++qe) {
    // <v|E|v> = sum_i conj(v_i) sum_j E[i][j] v_j with E^T stored: E[i][j] = ET[j][i]
    double ar = 0.0, ai = 0.0;
    for (int i = threadIdx.x; i < np; i += T) {
      double sr = 0.0, si = 0.0;
      for (int j = 0; j < np; ++j) {
        const float2 e = ET[(size_t)qe * np * np + (size_t)j * np + i];
        sr += e.x * v[j].x - e.y * v[j].y;
        si += e.x * v[j].y + e.y * v[j].x;
      }
      ar += v[i].x * sr + v[i].y * si;
      ai += v[i].x * si - v[i].y * sr;
    }
    const double sr = bsum<T>(ar, red), si = bsum<T>(ai, red);
    if (threadIdx.x == 0) gp<float2>(p.expects)[(size_t)qe * ntsave + isave] = make_float2((float)sr, (float)si);
  }
  __syncthreads();
}

// MAXNP: the largest padded dimension the LDS arrays hold (64, 256 or 1024; the
// 1024 variant takes 112 KB of LDS, one workgroup per CU)
template <int T, int MAXNP>
__global__ __launch_bounds__(T) void k_sesolve(const dqh_me_inst *__restrict__ insts) {
  constexpr int kMaxNp = MAXNP;
  __shared__ double red[SeCfg<T>::kW];
  __shared__ double2 y[kMaxNp], y1[kMaxNp], vsave[kMaxNp];
  __shared__ float2 ys[kMaxNp];
  __shared__ float2 k[7][kMaxNp];
  const dqh_me_inst &p = insts[blockIdx.x];
  const RKTab &rk = rk_tab(p.flags);
  const int n = (int)p.n, np = (int)p.np, ntsave = (int)p.ntsave, nseg = (int)p.nseg;
  const bool pwc = p.npwc > 0, smooth = p.nmod > 0;
  const double *tsave = gp<const double>(p.tsave);
  const double *ptimes = gp<const double>(p.pwc_times);
  int64_t *stats = gp<int64_t>(p.stats);
  if (np > kMaxNp || n <= 0 || n > np || p.npwc > 8 || p.nmod > DQH_MAX_MOD || (p.npwc > 0 && nseg < 2) ||
      ((p.flags & DQH_FLAG_EULER) && (!p.step_t || p.max_steps < 0))) {
    if (threadIdx.x == 0) stats[3] = DQH_UNSUPPORTED;
    return;
  }
  const double rtol = p.rtol, atol = p.atol, inv_n = 1.0 / (double)n, t_end = p.t1;
  const double w0[7] = {0, 0, 0, 0, 0, 0, 0};
  const double2 *y0 = gp<const double2>(p.y);
  for (int i = threadIdx.x; i < np; i += T) {
    y[i] = i < n ? y0[i] : make_double2(0.0, 0.0);
    for (int j = 0; j < 7; ++j) k[j][i] = make_float2(0.f, 0.f);
  }
  __syncthreads();
  double t = p.t0;
  int isave = 0, status = 0;
  int64_t nsteps = 0, nacc = 0, nrej = 0, nrhs = 0;
  while (isave < ntsave && tsave[isave] <= t) {
    save_at<T, MAXNP>(p, y, k, 0.0, w0, false, isave, vsave, red);
    ++isave;
  }
  if (p.flags & DQH_FLAG_EULER) {
    // fixed steps between the boundaries step_t[0..max_steps]: y <- y + h G(t) y with
    // the operators at the step start, linear interpolation to the save times
    const double *st = gp<const double>(p.step_t);
    Coef cf;
    double wl[7] = {0, 0, 0, 0, 0, 0, 0};
    for (int64_t m = 0; m < p.max_steps; ++m) {
      const double ta = st[m], tb = st[m + 1], h = tb - ta;
      coefficients(p, pwc ? segment_of(ptimes, nseg, ta) : -1, ta, cf);
      for (int i = threadIdx.x; i < np; i += T) ys[i] = make_float2((float)y[i].x, (float)y[i].y);
      __syncthreads();
      field<T>(p, cf, ys, k[0]);
      ++nrhs;
      while (isave < ntsave && tsave[isave] <= tb + 1e-12 * fmax(1.0, fabs(tb))) {
        wl[0] = fmin(fmax((tsave[isave] - ta) / h, 0.0), 1.0);
        save_at<T, MAXNP>(p, y, k, h, wl, true, isave, vsave, red);
        ++isave;
      }
      for (int i = threadIdx.x; i < np; i += T)
        y[i] = make_double2(y[i].x + h * (double)k[0][i].x, y[i].y + h * (double)k[0][i].y);
      __syncthreads();
      ++nsteps;
      ++nacc;
    }
  } else {
    int seg = pwc ? segment_of(ptimes, nseg, t) : -1;
    Coef cf;
    coefficients(p, seg, t, cf);
    for (int i = threadIdx.x; i < np; i += T) ys[i] = make_float2((float)y[i].x, (float)y[i].y);
    __syncthreads();
    field<T>(p, cf, ys, k[0]);
    ++nrhs;
    // initial step (Hairer-Norsett-Wanner II.4), scale atol + rtol |y0|
    double dt;
    {
      double s0 = 0.0, s1 = 0.0;
      for (int i = threadIdx.x; i < n; i += T) {
        const double ay2 = y[i].x * y[i].x + y[i].y * y[i].y;
        const double sc = atol + rtol * sqrt(ay2);
        s0 += ay2 / (sc * sc);
        s1 += ((double)k[0][i].x * k[0][i].x + (double)k[0][i].y * k[0][i].y) / (sc * sc);
      }
      const double d0 = sqrt(bsum<T>(s0, red) * inv_n), d1 = sqrt(bsum<T>(s1, red) * inv_n);
      const double h0 = (d0 < 1e-5 || d1 < 1e-5) ? 1e-6 : 0.01 * d0 / d1;
      for (int i = threadIdx.x; i < np; i += T)
        ys[i] = make_float2((float)(y[i].x + h0 * k[0][i].x), (float)(y[i].y + h0 * k[0][i].y));
      __syncthreads();
      if (smooth) coefficients(p, seg, t + h0, cf);
      field<T>(p, cf, ys, k[1]);
      ++nrhs;
      double s2 = 0.0;
      for (int i = threadIdx.x; i < n; i += T) {
        const double sc = atol + rtol * sqrt(y[i].x * y[i].x + y[i].y * y[i].y);
        const double dr = (double)k[1][i].x - k[0][i].x, di = (double)k[1][i].y - k[0][i].y;
        s2 += (dr * dr + di * di) / (sc * sc);
      }
      const double d2 = sqrt(bsum<T>(s2, red) * inv_n) / h0;
      const double md = fmax(d1, d2);
      const double h1 = md <= 1e-15 ? fmax(1e-6, h0 * 1e-3) : ctrl_pow(0.01 / md, kInitExp);
      dt = fmin(100.0 * h0, h1);
    }
    bool need_k0 = false;
    while (t < t_end) {
      if (nsteps >= p.max_steps) {
        status = DQH_MAX_STEPS;
        break;
      }
      if (pwc) {
        const int s = segment_of(ptimes, nseg, t);
        if (s != seg) seg = s;
      }
      if (need_k0) {
        coefficients(p, seg, t, cf);
        for (int i = threadIdx.x; i < np; i += T) ys[i] = make_float2((float)y[i].x, (float)y[i].y);
        __syncthreads();
        field<T>(p, cf, ys, k[0]);
        ++nrhs;
        need_k0 = false;
      }
      double h = dt, target = t_end;
      bool target_jump = false;
      if (pwc) {
        const int m = segment_of(ptimes, nseg, t) + 1;
        if (m < nseg && ptimes[m] < t_end) {
          target = ptimes[m];
          target_jump = true;
        }
      }
      bool made_jump = false;
      double t_new = t + h;
      if (snaps_to(t, h, target)) {
        h = target - t;
        t_new = target;
        made_jump = target_jump;
      }
      if (!(h > 0.0) || !(h > 1e-14 * fmax(1.0, fabs(t)))) {
        status = DQH_NONFINITE;
        break;
      }
      if (!smooth) coefficients(p, seg, t, cf);
      for (int s = 1; s < 7; ++s) {
        for (int i = threadIdx.x; i < np; i += T) {
          double re = y[i].x, im = y[i].y;
          for (int j = 0; j < s; ++j) {
            re += h * rk.A[s][j] * k[j][i].x;
            im += h * rk.A[s][j] * k[j][i].y;
          }
          if (s == 6) y1[i] = make_double2(re, im);
          ys[i] = make_float2((float)re, (float)im);
        }
        __syncthreads();
        if (smooth) coefficients(p, seg, t + rk.C[s] * h, cf);
        field<T>(p, cf, ys, k[s]);
        ++nrhs;
      }
      double ssum = 0.0;
      for (int i = threadIdx.x; i < n; i += T) {
        double er = 0.0, ei = 0.0;
        for (int j = 0; j < 7; ++j) {
          er += rk.E[j] * k[j][i].x;
          ei += rk.E[j] * k[j][i].y;
        }
        er *= h;
        ei *= h;
        const double sc = atol + rtol * fmax(sqrt(y[i].x * y[i].x + y[i].y * y[i].y),
                                             sqrt(y1[i].x * y1[i].x + y1[i].y * y1[i].y));
        ssum += (er * er + ei * ei) / (sc * sc);
      }
      const double norm = sqrt(bsum<T>(ssum, red) * inv_n);
      const bool finite = isfinite(norm), keep = finite && norm < 1.0;
      double factor = !finite ? p.factormin : (norm == 0.0 ? p.factormax : p.safety * ctrl_pow(norm, -0.2));
      factor = fmin(fmax(factor, keep ? 1.0 : p.factormin), p.factormax);
      ++nsteps;
      if (keep) {
        if (threadIdx.x == 0 && nacc < p.step_log_cap) gp<double>(p.step_log)[nacc] = t_new;
        ++nacc;
        while (isave < ntsave && tsave[isave] <= t_new) {
          const double th = (tsave[isave] - t) / h;
          double w[7];
          for (int j = 0; j < 7; ++j) w[j] = th * (rk.R[j][0] + th * (rk.R[j][1] + th * (rk.R[j][2] + th * rk.R[j][3])));
          save_at<T, MAXNP>(p, y, k, h, w, true, isave, vsave, red);
          ++isave;
        }
        for (int i = threadIdx.x; i < np; i += T) {
          y[i] = y1[i];
          k[0][i] = k[6][i];
        }
        __syncthreads();
        t = t_new;
        need_k0 = made_jump;
      } else {
        ++nrej;
      }
      dt = factor * h;
    }
  }
  while (isave < ntsave) {
    save_at<T, MAXNP>(p, y, k, 0.0, w0, false, isave, vsave, red);
    ++isave;
  }
  for (int i = threadIdx.x; i < n; i += T) {
    const float2 v = make_float2((float)y[i].x, (float)y[i].y);
    gp<float2>(p.final_state)[i] = v;
    if (!(p.flags & DQH_FLAG_SAVE_STATES)) gp<float2>(p.states)[i] = v;
  }
  if (threadIdx.x == 0) {
    stats[0] = nsteps;
    stats[1] = nacc;
    stats[2] = nrej;
    stats[3] = status;
    stats[4] = nrhs;
  }
}

// Constant Hamiltonians up to n = 128: four lanes per row, each with a quarter of the row's
// columns of G = -i H in registers, and the state and stages of the row in registers too
// (alike in its four lanes). The stage input goes through LDS (two copies alternate, one
// barrier per stage), the four partial sums are added within the quad. Up to n = 64 the first
// expectation operator is in registers as well. Bound by the latency of a stage. A call,
// against reading G from the caches at every stage: 48 solves of n = 64 (50 saves, Dopri5)
// 2.45 -> 1.1 ms, 3000 two-level solves 2.0 -> 1.9 ms (the host's share), up to 7 times
// less at 64 < n <= 128.
template <int NR, int TAB>
__global__ __launch_bounds__(4 * NR) void k_sesolve_const(const dqh_me_inst *__restrict__ insts) {
  constexpr int T = 4 * NR, CP = NR / 8;  // column pairs per lane: 8 c + 2 q, 8 c + 2 q + 1
  __shared__ __align__(16) float2 ys[2][NR];
  __shared__ __align__(16) double2 vs[2][NR];
  __shared__ double red[4 * (T / 64)];
  constexpr RKTab rk = kRKTabs[TAB];
  const dqh_me_inst &p = insts[blockIdx.x];
  const int n = (int)p.n, np = (int)p.np, nE = (int)p.nE, ntsave = (int)p.ntsave;
  const int tid = (int)threadIdx.x, i = tid >> 2, q = tid & 3;
  int64_t *stats = gp<int64_t>(p.stats);
  if (n <= 0 || n > NR || n > np || p.npwc != 0 || p.nmod != 0 || (p.flags & DQH_FLAG_EULER) ||
      ((p.flags & DQH_FLAG_DOPRI5) != 0) != (TAB == 1)) {
    if (tid == 0) stats[3] = DQH_UNSUPPORTED;
    return;
  }
  const double *tsave = gp<const double>(p.tsave);
  const double rtol = p.rtol, atol = p.atol, inv_n = 1.0 / (double)n, t_end = p.t1;
  const bool row = i < n, one = row && q == 0, save_states = (p.flags & DQH_FLAG_SAVE_STATES) != 0;
  // matrices are stored transposed: consecutive rows are consecutive addresses
  auto load = [&](const float2 *M, float2 (&g)[2 * CP]) {
#pragma unroll
    for (int c = 0; c < 2 * CP; ++c) {
      const int j = 8 * (c >> 1) + 2 * q + (c & 1);
      g[c] = row && j < n ? M[(size_t)j * np + i] : make_float2(0.f, 0.f);
    }
  };
  constexpr bool kKeepE = NR <= 64;
  float2 g[2 * CP], E0[kKeepE ? 2 * CP : 1];
  load(gp<const float2>(p.Hnh), g);
  const float2 *ET = gp<const float2>(p.EopsT);
  if constexpr (kKeepE) {
    if (nE > 0) load(ET, E0);
  }
  double2 y = row ? gp<const double2>(p.y)[i] : make_double2(0.0, 0.0), y1 = make_double2(0.0, 0.0);
  float2 k[7];
#pragma unroll
  for (int s = 0; s < 7; ++s) k[s] = make_float2(0.f, 0.f);
  int cur = 0, par = 0;
  auto field = [&](double2 v) -> float2 {
    float2 *b = ys[cur];
    cur ^= 1;
    if (q == 0) b[i] = make_float2((float)v.x, (float)v.y);
    __syncthreads();
    const float4 *b4 = reinterpret_cast<const float4 *>(b);
    float ar = 0.f, ai = 0.f, br = 0.f, bi = 0.f;
#pragma unroll
    for (int c = 0; c < CP; ++c) {
      if (c > 0 && c % 8 == 0) asm volatile("" ::: "memory");  // at most 8 reads in flight, for their registers
      const float4 x = b4[4 * c + q];
      ar = fmaf(g[2 * c].x, x.x, fmaf(-g[2 * c].y, x.y, ar));
      ai = fmaf(g[2 * c].x, x.y, fmaf(g[2 * c].y, x.x, ai));
      br = fmaf(g[2 * c + 1].x, x.z, fmaf(-g[2 * c + 1].y, x.w, br));
      bi = fmaf(g[2 * c + 1].x, x.w, fmaf(g[2 * c + 1].y, x.z, bi));
    }
    return make_float2(quad_sum(ar + br), quad_sum(ai + bi));
  };
  int vcur = 0;
  // y + h sum_j w_j k_j (state and <psi|E|psi>) at save index isave (h = 0: the state itself,
  // whatever the stages of a rejected step hold)
  auto save = [&](double h, const double (&w)[7], int isave) {
    double re = 0.0, im = 0.0;
    if (h != 0.0) {
#pragma unroll
      for (int j = 0; j < 7; ++j) {
        re += w[j] * (double)k[j].x;
        im += w[j] * (double)k[j].y;
      }
    }
    const double2 v = make_double2(y.x + h * re, y.y + h * im);
    if (save_states && one) gp<float2>(p.states)[(size_t)isave * n + i] = make_float2((float)v.x, (float)v.y);
    if (nE == 0) return;
    double2 *vb = vs[vcur];
    vcur ^= 1;
    if (q == 0) vb[i] = v;
    __syncthreads();
    for (int e = 0; e < nE; ++e) {
      double sr = 0.0, si = 0.0;
      const float2 *M = ET + (size_t)e * np * np;
      bool kept = false;
      if constexpr (kKeepE) kept = e == 0;
#pragma unroll
      for (int c = 0; c < 2 * CP; ++c) {
        if (c > 0 && c % 8 == 0) asm volatile("" ::: "memory");
        int qq = q;
        float2 m = make_float2(0.f, 0.f);
        if constexpr (kKeepE) m = E0[c];
        asm volatile("" : "+v"(m.x), "+v"(m.y), "+v"(qq));  // addresses and FP64 values are formed here, not kept
        const int j = 8 * (c >> 1) + 2 * qq + (c & 1);
        // rows and columns past n meet a zero of v: any element in range will do there
        if (!kept) m = M[min(j, np - 1) * np + min(i, np - 1)];
        const double2 x = vb[j];
        sr += m.x * x.x - m.y * x.y;
        si += m.x * x.y + m.y * x.x;
      }
      double s[2] = {v.x * sr + v.y * si, v.x * si - v.y * sr};
      block_sums<T>(s, red, par);
      if (tid == 0) gp<float2>(p.expects)[(size_t)e * ntsave + isave] = make_float2((float)s[0], (float)s[1]);
    }
  };
  const double w0[7] = {0, 0, 0, 0, 0, 0, 0};
  double t = p.t0;
  int isave = 0, status = 0;
  int64_t nsteps = 0, nacc = 0, nrej = 0, nrhs = 0;
  double next_save = ntsave > 0 ? tsave[0] : 0.0;
  auto advance = [&]() {
    ++isave;
    if (isave < ntsave) next_save = tsave[isave];
  };
  while (isave < ntsave && next_save <= t) {
    save(0.0, w0, isave);
    advance();
  }
  k[0] = field(y);
  ++nrhs;
  // initial step (Hairer-Norsett-Wanner II.4), scale atol + rtol |y0|
  double dt;
  {
    const double ay2 = y.x * y.x + y.y * y.y, sc = atol + rtol * sqrt(ay2), u = one ? 1.0 / (sc * sc) : 0.0;
    double s[2] = {u * ay2, u * ((double)k[0].x * k[0].x + (double)k[0].y * k[0].y)};
    block_sums<T>(s, red, par);
    const double d0 = sqrt(s[0] * inv_n), d1 = sqrt(s[1] * inv_n);
    const double h0 = (d0 < 1e-5 || d1 < 1e-5) ? 1e-6 : 0.01 * d0 / d1;
    k[1] = field(make_double2(y.x + h0 * k[0].x, y.y + h0 * k[0].y));
    ++nrhs;
    const double dr = (double)k[1].x - k[0].x, di = (double)k[1].y - k[0].y;
    double s2[1] = {u * (dr * dr + di * di)};
    block_sums<T>(s2, red, par);
    const double d2 = sqrt(s2[0] * inv_n) / h0;
    const double md = fmax(d1, d2);
    const double h1 = md <= 1e-15 ? fmax(1e-6, h0 * 1e-3) : ctrl_pow(0.01 / md, kInitExp);
    dt = fmin(100.0 * h0, h1);
  }
  while (t < t_end) {
    if (nsteps >= p.max_steps) {
      status = DQH_MAX_STEPS;
      break;
    }
    double h = dt, t_new = t + h;
    if (snaps_to(t, h, t_end)) {
      h = t_end - t;
      t_new = t_end;
    }
    if (!(h > 0.0) || !(h > 1e-14 * fmax(1.0, fabs(t)))) {
      status = DQH_NONFINITE;
      break;
    }
#pragma unroll
    for (int s = 1; s < 7; ++s) {
      CTab *w = weights<TAB>();
      double re = 0.0, im = 0.0;
#pragma unroll
      for (int j = 0; j < s; ++j) {
        if (rk.A[s][j] != 0.0) {  // compile-time
          re += w->A[s][j] * (double)k[j].x;
          im += w->A[s][j] * (double)k[j].y;
        }
      }
      y1 = make_double2(y.x + h * re, y.y + h * im);
      k[s] = field(y1);
    }
    nrhs += 6;
    CTab *we = weights<TAB>();
    double er = 0.0, em = 0.0;
#pragma unroll
    for (int j = 0; j < 7; ++j) {
      if (rk.E[j] != 0.0) {
        er += we->E[j] * (double)k[j].x;
        em += we->E[j] * (double)k[j].y;
      }
    }
    er *= h;
    em *= h;
    const double sc = atol + rtol * sqrt(fmax(y.x * y.x + y.y * y.y, y1.x * y1.x + y1.y * y1.y));
    double ss[1] = {one ? (er * er + em * em) / (sc * sc) : 0.0};
    block_sums<T>(ss, red, par);
    const double norm = sqrt(ss[0] * inv_n);
    const bool finite = isfinite(norm), keep = finite && norm < 1.0;
    double factor = !finite ? p.factormin : (norm == 0.0 ? p.factormax : p.safety * ctrl_pow(norm, -0.2));
    factor = fmin(fmax(factor, keep ? 1.0 : p.factormin), p.factormax);
    ++nsteps;
    if (keep) {
      if (tid == 0 && nacc < p.step_log_cap) gp<double>(p.step_log)[nacc] = t_new;
      ++nacc;
      while (isave < ntsave && next_save <= t_new) {
        const double th = (next_save - t) / h;
        CTab *wr = weights<TAB>();
        double w[7];
#pragma unroll
        for (int j = 0; j < 7; ++j)
          w[j] = th * (wr->R[j][0] + th * (wr->R[j][1] + th * (wr->R[j][2] + th * wr->R[j][3])));
        save(h, w, isave);
        advance();
      }
      y = y1;
      k[0] = k[6];
      t = t_new;
    } else {
      ++nrej;
    }
    dt = factor * h;
  }
  while (isave < ntsave) {
    save(0.0, w0, isave);
    advance();
  }
  if (one) {
    const float2 v = make_float2((float)y.x, (float)y.y);
    gp<float2>(p.final_state)[i] = v;
    if (!save_states) gp<float2>(p.states)[i] = v;
  }
  if (tid == 0) {
    stats[0] = nsteps;
    stats[1] = nacc;
    stats[2] = nrej;
    stats[3] = status;
    stats[4] = nrhs;
  }
}

template <int TAB>
void launch_const(const dqh_me_inst *d, int64_t ninst, int64_t n, hipStream_t st) {
  const dim3 g((unsigned)ninst);
  if (n <= 16)
    hipLaunchKernelGGL((k_sesolve_const<16, TAB>), g, dim3(64), 0, st, d);
  else if (n <= 32)
    hipLaunchKernelGGL((k_sesolve_const<32, TAB>), g, dim3(128), 0, st, d);
  else if (n <= 64)
    hipLaunchKernelGGL((k_sesolve_const<64, TAB>), g, dim3(256), 0, st, d);
  else
    hipLaunchKernelGGL((k_sesolve_const<128, TAB>), g, dim3(512), 0, st, d);
}

}  // namespace se
}  // namespace dqh

extern "C" int dqh_sesolve_tsit5_const(const dqh_me_inst *d_insts, int64_t ninst, int64_t n, int64_t flags, void *stream) {
  if (!d_insts || ninst <= 0 || ninst > (1 << 30) || n <= 0 || n > 128)
    return dqh::fail(DQH_BAD_ARG, "dqh_sesolve_tsit5_const: bad arguments");
  if (flags & DQH_FLAG_DOPRI5)
    dqh::se::launch_const<1>(d_insts, ninst, n, (hipStream_t)stream);
  else
    dqh::se::launch_const<0>(d_insts, ninst, n, (hipStream_t)stream);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return dqh::fail(DQH_HIP_ERROR, std::string("dqh_sesolve_tsit5_const: ") + hipGetErrorString(err));
  return DQH_OK;
}

extern "C" int dqh_sesolve_tsit5(const dqh_me_inst *d_insts, int64_t ninst, int64_t np_max, void *stream) {
  if (!d_insts || ninst <= 0 || ninst > (1 << 30) || np_max <= 0 || np_max > 1024)
    return dqh::fail(DQH_BAD_ARG, "dqh_sesolve_tsit5: bad arguments");
  if (np_max <= 64)
    hipLaunchKernelGGL((dqh::se::k_sesolve<64, 64>), dim3((unsigned)ninst), dim3(64), 0, (hipStream_t)stream, d_insts);
  else if (np_max <= 256)
    hipLaunchKernelGGL((dqh::se::k_sesolve<256, 256>), dim3((unsigned)ninst), dim3(256), 0, (hipStream_t)stream,
                       d_insts);
  else
    hipLaunchKernelGGL((dqh::se::k_sesolve<256, 1024>), dim3((unsigned)ninst), dim3(256), 0, (hipStream_t)stream,
                       d_insts);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return dqh::fail(DQH_HIP_ERROR, std::string("dqh_sesolve_tsit5: ") + hipGetErrorString(err));
  return DQH_OK;
}
