// Adaptive Tsit5 / Dopri5 for small master equations whose operators have few nonzero
// diagonals (gfx950), n < 128: one workgroup per instance.
//
// The vector field G rho + rho G^dag + sum_k L_k rho L_k^dag of such operators is a
// stencil, f[i][j] = sum_t C_t(i, j) rho[i + a_t][j + b_t]: one shift (o, 0) and one
// (0, o) per off-diagonal o of G, one (p, q) per pair of diagonals of a jump operator,
// equal shifts merged. A driven oscillator has 5 shifts and a driven Kerr oscillator
// with two-photon loss 6, against (1 + 2K) n multiply-adds per element of the dense
// products, so the matrix cores have nothing to do here and a step is bound by the
// latency of its dependent stages (n <= 32) and by FP64 issue and LDS reads (n = 64).
//
// k_tsit5_diag, n <= 64 and at most 12 shifts: a thread owns NE elements of the upper
// triangle (u = thread + NTH q, row by row, of the n (n + 1) / 2 that exist: no work on
// padding). Its coefficients C_t, the FP64 diagonal generator g = d_i + conj(d_j), the FP64
// state, the candidate and the seven FP32 stages stay in registers for the whole solve. The
// stage input goes to LDS in FP32 (both triangles), the neighbours come back with one
// 8-byte read per shift, and the FP64 diagonal term takes the thread's own input unrounded.
// Two LDS copies alternate, so a stage costs one barrier, and the stages are unrolled with
// the tableau's weights in scalar registers. With several elements per thread the saves
// form one element at a time, slots are recomputed and uniform doubles are scalar: without
// that the three elements of n = 64 spilled 340 registers in every step.
// Measured against the resident dense body: oscillator n = 16, 85 steps and 101 saves 1.20
// -> 0.31 ms; 128 driven Kerr oscillators n = 64 (2 jump operators, about 440 steps) 57.4 ->
// 4.5 ms (7.3 with the spills); the solves of a gradient at n = 32, 64 control vectors, 6.4
// -> 1.3 ms (500 saves of the backward solve: 1.19 -> 1.00 ms with the weights of all saves
// of a step formed at once, one per lane). The controller, step clipping, FSAL, saving and
// the precision of the operators and stages are those of the dense kernels.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <utility>
#include <vector>

#include "dqh.h"
#include "dqh_common.h"
#include "dqh_mfma.h"
#include "dqh_tsit5_tableau.h"
#include "dqh_wave.h"

namespace dqh {
namespace diag {

constexpr int kMaxShift = 12;  // shifts of the stencil (register coefficients per element)
constexpr int kMaxPart = 48;   // contributions to the shifts' coefficients
constexpr int kMaxOff = 16;    // off-diagonals of the generator

// A contribution to a coefficient: kind 0 G_x[i] (row diagonal x of the generator),
// kind 1 conj(G_x[j]), kind 2 L_x[i] conj(L_y[j]) (x, y: rows of the jump-operator table).
struct Part {
  uint8_t kind, x, y, pad;
};

struct Pattern {
  int32_t nterm, nH, nLrow, nzero;  // shifts, off-diagonals of G, jump-operator rows, parts of shift (0, 0)
  int32_t guard;                    // largest |a LD + b|
  int32_t a[kMaxShift], b[kMaxShift];
  int32_t first[kMaxShift + 1];  // parts of shift t: part[first[t]] .. part[first[t + 1] - 1]
  Part part[kMaxPart];
  Part zero[kMaxPart];
  // the same for the table form: off-diagonals of G, and the pairs of jump-operator rows
  // (kind 2 parts) with their shifts, (0, 0) excepted
  int32_t offH[kMaxOff];
  int32_t npair;
  Part pair[kMaxPart];
  int16_t pa[kMaxPart], pb[kMaxPart];
};

// LDS: two copies of the stage input (rows of LD = n | 1 float2, one slot that elements
// past the end write, a guard of G zeros before, between and after them so that a shift
// may leave the matrix: its coefficient is zero there), the generator's off-diagonals and
// the jump operators' rows (n each), its diagonal (FP64), partial sums.
__host__ __device__ inline int row_stride(int n) { return n | 1; }
__host__ __device__ inline int copy_stride(int n, int guard) { return n * row_stride(n) + 1 + guard; }
template <int NTH>
__host__ __device__ inline size_t lds_bytes(int n, int nH, int nLrow, int guard) {
  return (size_t)(2 * copy_stride(n, guard) + guard + (nH + nLrow) * n) * sizeof(float2) +
         (size_t)n * sizeof(double2) + (size_t)(4 * (NTH / 64)) * sizeof(double);
}

// a double that is the same in all lanes, in scalar registers where several elements per
// thread need the vector ones (ON); a single element is bound by latency instead
template <bool ON>
__device__ __forceinline__ double uniform(double x) {
  if constexpr (!ON) return x;
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

template <int NTH, int NE, int T, int TAB>
__global__ __launch_bounds__(NTH) void k_tsit5_diag(const dqh_me_inst *__restrict__ insts, Pattern pat) {
  extern __shared__ __align__(16) char smem[];
  const dqh_me_inst &p = insts[blockIdx.x];
  constexpr RKTab rk = kRKTabs[TAB];
  const int n = (int)p.n, np = (int)p.np, nE = (int)p.nE, ntsave = (int)p.ntsave, nseg = (int)p.nseg;
  const int LD = row_stride(n), tid = (int)threadIdx.x;
  const int npwc = (int)p.npwc;
  const bool pwc = npwc > 0;
  double2 *dcur = reinterpret_cast<double2 *>(smem);  // n: diagonal of the current generator
  double *red = reinterpret_cast<double *>(dcur + n);  // 4 NW
  const int CS = copy_stride(n, pat.guard);
  float2 *ysA = reinterpret_cast<float2 *>(red + 4 * (NTH / 64)) + pat.guard;
  float2 *Gt = ysA + 2 * CS;        // nH x n: G[i][i + o] of the current generator
  float2 *Lt = Gt + pat.nH * n;     // nLrow x n: L[i][i + p]
  int64_t *stats = gp<int64_t>(p.stats);
  if (n > 64 || n * (n + 1) / 2 > NTH * NE || p.nmod != 0 || (pwc && nseg < 2) ||
      (p.flags & (DQH_FLAG_GLOBAL | DQH_FLAG_LMOD | DQH_FLAG_DOPRI8 | DQH_FLAG_EULER)) ||
      ((p.flags & DQH_FLAG_DOPRI5) != 0) != (TAB == 1)) {
    if (tid == 0) stats[3] = DQH_UNSUPPORTED;
    return;
  }
  const double *tsave = gp<const double>(p.tsave);
  const double *ptimes = gp<const double>(p.pwc_times);
  const double rtol = p.rtol, atol = p.atol, t_end = p.t1;
  const double inv_nn = uniform<(NE > 1)>(1.0 / ((double)n * n));
  const bool save_states = (p.flags & DQH_FLAG_SAVE_STATES) != 0;

  // owned elements, packed i | j << 8 (i <= j; -1 past the end): their slots in a copy are
  // formed where they are used, or the registers would not hold the stages
  const int NU = n * (n + 1) / 2;
  int ij[NE];
#pragma unroll
  for (int q = 0; q < NE; ++q) {
    int rem = tid + NTH * q, i = 0;
    ij[q] = -1;
    if (rem < NU) {
      while (rem >= n - i) {
        rem -= n - i;
        ++i;
      }
      ij[q] = i | ((i + rem) << 8);
    }
  }
  // row and column of element q; past the end 0, 0
  auto at = [&](int q, int &i, int &j) {
    int x = ij[q];
    if constexpr (NE > 1) asm volatile("" : "+v"(x));
    const int z = x < 0 ? 0 : x;
    i = z & 255;
    j = z >> 8;
    return x >= 0;
  };
  for (int e = tid; e < 2 * CS + pat.guard; e += NTH) (ysA - pat.guard)[e] = make_float2(0.f, 0.f);
  for (int e = tid; e < pat.nLrow * n; e += NTH) {
    const int r = e / n, i = e - r * n;
    Lt[e] = gp<const float2>(p.Dops)[(size_t)r * np + i];
  }

  // Gt, dcur <- the constant generator plus the PWC terms of segment seg
  const float2 *G0 = gp<const float2>(p.Hnh);
  const double2 *d0g = gp<const double2>(p.hdiag);
  const float2 *Hp = gp<const float2>(p.Hpwc);
  const double *vals = gp<const double>(p.pwc_vals);
  float cr[T][NE], ci[T][NE];
  double gr[NE], gi[NE];
  auto build = [&](int seg) {
    const int nv = nseg - 1;
    const bool inside = pwc && seg >= 0 && seg < nv;
    for (int e = tid; e < (pat.nH + 1) * n; e += NTH) {
      const int r = e / n, i = e - r * n;
      double re, im;
      if (r < pat.nH) {
        const float2 o = G0[(size_t)r * np + i];
        re = o.x;
        im = o.y;
      } else {
        re = d0g[i].x;
        im = d0g[i].y;
      }
      if (inside) {
        for (int j = 0; j < npwc; ++j) {
          const double vr = vals[2 * (j * nv + seg)], vi = vals[2 * (j * nv + seg) + 1];
          const float2 o = Hp[((size_t)j * (pat.nH + 1) + r) * np + i];
          re += vr * o.x - vi * o.y;
          im += vr * o.y + vi * o.x;
        }
      }
      if (r < pat.nH)
        Gt[e] = make_float2((float)re, (float)im);
      else
        dcur[i] = make_double2(re, im);
    }
    __syncthreads();
    int z = 0;  // keeps the pattern's scalar loads here
    asm volatile("" : "+s"(z));
    auto coef = [&](const Part &s, int i, int j) -> float2 {
      if (s.kind == 0) return Gt[s.x * n + i];
      if (s.kind == 1) {
        const float2 c = Gt[s.x * n + j];
        return make_float2(c.x, -c.y);
      }
      const float2 a = Lt[s.x * n + i], c = Lt[s.y * n + j];
      return make_float2(a.x * c.x + a.y * c.y, a.y * c.x - a.x * c.y);
    };
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      int i, j;
      const bool on = at(q, i, j);
#pragma unroll
      for (int t = 0; t < T; ++t) {
        float ar = 0.f, ai = 0.f;
        for (int s = pat.first[t + z]; s < pat.first[t + 1 + z]; ++s) {
          const float2 c = coef(pat.part[s], i, j);
          ar += c.x;
          ai += c.y;
        }
        cr[t][q] = on ? ar : 0.f;
        ci[t][q] = on ? ai : 0.f;
      }
      const double2 da = dcur[i], db = dcur[j];
      double r = da.x + db.x, m = da.y - db.y;
      for (int s = z; s < pat.nzero; ++s) {
        // products of the jump operators' main diagonals, in FP64
        const float2 a = Lt[pat.zero[s].x * n + i], c = Lt[pat.zero[s].y * n + j];
        r += (double)a.x * c.x + (double)a.y * c.y;
        m += (double)a.y * c.x - (double)a.x * c.y;
      }
      gr[q] = on ? r : 0.0;
      gi[q] = on ? m : 0.0;
    }
  };

  // state
  double2 y[NE], y1[NE];
  float2 k[7][NE];
  {
    const double2 *y0 = gp<const double2>(p.y);
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      int i, j;
      y[q] = at(q, i, j) ? y0[(size_t)i * np + j] : make_double2(0.0, 0.0);
      if (i == j) y[q].y = 0.0;
      y1[q] = make_double2(0.0, 0.0);
#pragma unroll
      for (int s = 0; s < 7; ++s) k[s][q] = make_float2(0.f, 0.f);
    }
  }
  int cur = 0;  // LDS copy of the next stage input
  int sh[T];
#pragma unroll
  for (int t = 0; t < T; ++t) sh[t] = t < pat.nterm ? pat.a[t] * LD + pat.b[t] : 0;

  // out = f(v): v (FP64) to LDS in FP32 on both triangles, one barrier, the stencil in
  // FP32 and the diagonal term in FP64
  auto field = [&](const double2 (&v)[NE], float2 (&out)[NE]) {
    float2 *b = ysA + cur * CS;
    cur ^= 1;
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      const float2 x = make_float2((float)v[q].x, (float)v[q].y);
      int i, j;
      const bool on = at(q, i, j);
      b[on ? j * LD + i : n * LD] = make_float2(x.x, -x.y);
      b[on ? i * LD + j : n * LD] = x;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      int i, j;
      const bool on = at(q, i, j);
      const int e = on ? i * LD + j : n * LD;
      float2 x[T];
#pragma unroll
      for (int t = 0; t < T; ++t) x[t] = b[e + sh[t]];
      float fr = 0.f, fi = 0.f;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        fr = fmaf(cr[t][q], x[t].x, fmaf(-ci[t][q], x[t].y, fr));
        fi = fmaf(cr[t][q], x[t].y, fmaf(ci[t][q], x[t].x, fi));
      }
      const double re = (double)fr + (gr[q] * v[q].x - gi[q] * v[q].y);
      const double im = (double)fi + (gr[q] * v[q].y + gi[q] * v[q].x);
      // the diagonal of a Hermitian field is real
      out[q] = make_float2((float)re, i == j ? 0.f : (float)im);
      if constexpr (NE > 2) __builtin_amdgcn_sched_barrier(0);  // one element's neighbours in registers at a time
    }
  };

  // the FP64 conversions of the stages are made anew in every combination: kept from one
  // to the next (as common subexpressions) they would not fit the registers
  auto pin_stages = [&](int m) {
#pragma unroll
    for (int j = 0; j < 7; ++j) {
      if (j < m) {
#pragma unroll
        for (int q = 0; q < NE; ++q) asm volatile("" : "+v"(k[j][q].x), "+v"(k[j][q].y));
      }
    }
  };

  int par = 0;
  // y + h sum_j w_j k_j at save index isave (h = 0: the state itself, whatever the stages of
  // a rejected step hold): states on both triangles, Tr(E rho) over the owned elements and
  // their mirror images. One element at a time and formed anew for every
  // operator: kept, the values would not fit beside the stages.
  auto save = [&](double h, const double (&w)[7], int isave) {
    float2 *st = gp<float2>(p.states) + (size_t)isave * n * n;
    auto value = [&](int q) {
      if (h == 0.0) return y[q];
      double re = 0.0, im = 0.0;
#pragma unroll
      for (int j = 0; j < 7; ++j) {
        float2 x = k[j][q];
        if constexpr (NE > 1) asm volatile("" : "+v"(x.x), "+v"(x.y));
        re += w[j] * (double)x.x;
        im += w[j] * (double)x.y;
      }
      return make_double2(y[q].x + h * re, y[q].y + h * im);
    };
    double2 single = make_double2(0.0, 0.0);
    if constexpr (NE == 1) single = value(0);
    if (save_states) {
#pragma unroll
      for (int q = 0; q < NE; ++q) {
        const double2 v = NE == 1 ? single : value(q);
        int i, j;
        if (at(q, i, j)) {
          st[(size_t)i * n + j] = make_float2((float)v.x, (float)v.y);
          if (i != j) st[(size_t)j * n + i] = make_float2((float)v.x, (float)-v.y);
        }
        if constexpr (NE > 1) __builtin_amdgcn_sched_barrier(0);
      }
    }
    const float2 *ET = gp<const float2>(p.EopsT);
    for (int e = 0; e < nE; ++e) {
      const float2 *E = ET + (size_t)e * np * np;
      double s[2] = {0.0, 0.0};
#pragma unroll
      for (int q = 0; q < NE; ++q) {
        const double2 v = NE == 1 ? single : value(q);
        int i, j;
        if (at(q, i, j)) {
          const float2 o = E[(size_t)i * np + j];
          s[0] += o.x * v.x - o.y * v.y;
          s[1] += o.x * v.y + o.y * v.x;
          if (i != j) {
            const float2 m = E[(size_t)j * np + i];
            s[0] += m.x * v.x + m.y * v.y;
            s[1] += m.y * v.x - m.x * v.y;
          }
        }
        if constexpr (NE > 1) __builtin_amdgcn_sched_barrier(0);
      }
      block_sums<NTH>(s, red, par);
      if (tid == 0) gp<float2>(p.expects)[(size_t)e * ntsave + isave] = make_float2((float)s[0], (float)s[1]);
    }
  };
  // weight of element q in a sum over the full matrix
  auto weight = [&](int q) {
    int i, j;
    return at(q, i, j) ? (i == j ? 1.0 : 2.0) : 0.0;
  };
  const double w0[7] = {0, 0, 0, 0, 0, 0, 0};

  double t = p.t0;
  int isave = 0, status = 0;
  int64_t nsteps = 0, nacc = 0, nrej = 0, nrhs = 0;
  // NE = 1: the save times sbase .. sbase + 63, one per lane, and how many are due by x
  const int lane = tid & 63;
  int sbase = 0;
  double ts = NE == 1 && lane < ntsave ? tsave[lane] : 0.0;
  auto due = [&](double x) {
    const int i = sbase + lane;
    return (int)__popcll(__ballot(i >= isave && i < ntsave && ts <= x));
  };
  double next_save = ntsave > 0 ? tsave[0] : 0.0;
  auto advance = [&]() {
    ++isave;
    if (isave < ntsave) next_save = uniform<(NE > 1)>(tsave[isave]);
  };
  // segment of t (searchsorted right, -1 before the first breakpoint) and the breakpoint
  // after it; t only grows, so both move forward
  int seg = -1;
  double next_break = pwc ? ptimes[0] : 0.0;
  auto locate = [&]() {
    bool moved = false;
    while (seg + 1 < nseg && next_break <= t) {
      ++seg;
      moved = true;
      if (seg + 1 < nseg) next_break = ptimes[seg + 1];
    }
    return moved;
  };
  if (pwc) locate();
  __syncthreads();  // the LDS tables and the zeroed copies
  build(seg);
  while (isave < ntsave && next_save <= t) {
    save(0.0, w0, isave);
    advance();
  }
  if (NE == 1 && isave >= 64) {
    sbase = isave;
    ts = sbase + lane < ntsave ? tsave[sbase + lane] : 0.0;
  }
  field(y, k[0]);
  ++nrhs;

  // initial step (Hairer-Norsett-Wanner II.4), scale atol + rtol |y0|
  double dt;
  {
    double s[2] = {0.0, 0.0};
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      const double ay2 = y[q].x * y[q].x + y[q].y * y[q].y;
      const double sc = atol + rtol * sqrt(ay2);
      s[0] += weight(q) * ay2 / (sc * sc);
      s[1] += weight(q) * ((double)k[0][q].x * k[0][q].x + (double)k[0][q].y * k[0][q].y) / (sc * sc);
    }
    block_sums<NTH>(s, red, par);
    const double d0 = sqrt(s[0] * inv_nn), d1 = sqrt(s[1] * inv_nn);
    const double h0 = (d0 < 1e-5 || d1 < 1e-5) ? 1e-6 : 0.01 * d0 / d1;
#pragma unroll
    for (int q = 0; q < NE; ++q) y1[q] = make_double2(y[q].x + h0 * k[0][q].x, y[q].y + h0 * k[0][q].y);
    field(y1, k[1]);
    ++nrhs;
    double s2[1] = {0.0};
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      const double sc = atol + rtol * sqrt(y[q].x * y[q].x + y[q].y * y[q].y);
      const double dr = (double)k[1][q].x - k[0][q].x, di = (double)k[1][q].y - k[0][q].y;
      s2[0] += weight(q) * (dr * dr + di * di) / (sc * sc);
    }
    block_sums<NTH>(s2, red, par);
    const double d2 = sqrt(s2[0] * inv_nn) / h0;
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
    if (pwc && locate()) {
      __syncthreads();  // no wave still reads the previous tables
      build(seg);
    }
    if (need_k0) {
      field(y, k[0]);
      ++nrhs;
      need_k0 = false;
    }
    // clip the step to the end time or the next breakpoint strictly after t
    double h = dt, target = t_end;
    bool target_jump = false;
    if (pwc && seg + 1 < nseg && next_break < t_end) {
      target = next_break;
      target_jump = true;
    }
    bool made_jump = false;
    double t_new = t + h;
    if (snaps_to(t, h, target)) {
      h = target - t;
      t_new = target;
      made_jump = target_jump;
    }
    h = uniform<(NE > 1)>(h);
    t_new = uniform<(NE > 1)>(t_new);
    if (!(h > 0.0) || !(h > 1e-14 * fmax(1.0, fabs(t)))) {
      status = DQH_NONFINITE;
      break;
    }
    // stages 1..5 evaluate the field on the increment Delta_s = h sum_j a_sj k_j alone
    // (the generator is constant over the step): k[1..5] hold g_s = f(Delta_s), k_s =
    // k_0 + g_s, and every combination folds k_0 into the weight of k[0]. Stage 6 is a
    // full evaluation at y1 (the next k_0).
#pragma unroll
    for (int s = 1; s < 7; ++s) {
      CTab *w = weights<TAB>();
      if constexpr (NE > 1) pin_stages(s);
      const double a0 = w->C[s];  // row sum of A: the weight of k_0 with the increments folded in
#pragma unroll
      for (int q = 0; q < NE; ++q) {
        double re = a0 * (double)k[0][q].x, im = a0 * (double)k[0][q].y;
#pragma unroll
        for (int j = 1; j < s; ++j) {
          if (rk.A[s][j] != 0.0) {  // compile-time
            re += w->A[s][j] * (double)k[j][q].x;
            im += w->A[s][j] * (double)k[j][q].y;
          }
        }
        y1[q] = s < 6 ? make_double2(h * re, h * im) : make_double2(y[q].x + h * re, y[q].y + h * im);
        if constexpr (NE > 2) __builtin_amdgcn_sched_barrier(0);
      }
      field(y1, k[s]);
    }
    nrhs += 6;
    // error norm in FP64; y1 is the candidate of stage 6
    double ss[1] = {0.0};
    CTab *we = weights<TAB>();
    if constexpr (NE > 1) pin_stages(7);
    double e0 = 0.0;
#pragma unroll
    for (int j = 0; j < 6; ++j) e0 += we->E[j];
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      double er = e0 * (double)k[0][q].x, em = e0 * (double)k[0][q].y;
#pragma unroll
      for (int j = 1; j < 7; ++j) {
        if (rk.E[j] != 0.0) {
          er += we->E[j] * (double)k[j][q].x;
          em += we->E[j] * (double)k[j][q].y;
        }
      }
      er *= h;
      em *= h;
      const double sc = atol + rtol * sqrt(fmax(y[q].x * y[q].x + y[q].y * y[q].y,
                                                y1[q].x * y1[q].x + y1[q].y * y1[q].y));
      ss[0] += weight(q) * (er * er + em * em) / (sc * sc);
      if constexpr (NE > 2) __builtin_amdgcn_sched_barrier(0);
    }
    block_sums<NTH>(ss, red, par);
    const double norm = sqrt(ss[0] * inv_nn);
    const bool finite = isfinite(norm);
    const bool keep = finite && norm < 1.0;
    double factor;
    if (!finite)
      factor = p.factormin;
    else if (norm == 0.0)
      factor = p.factormax;
    else
      factor = p.safety * ctrl_pow(norm, -0.2);
    factor = fmin(fmax(factor, keep ? 1.0 : p.factormin), p.factormax);
    ++nsteps;
    if (keep) {
      if (tid == 0 && nacc < p.step_log_cap) gp<double>(p.step_log)[nacc] = t_new;
      ++nacc;
      if constexpr (NE == 1) {
        // the dense-output weights of all saves that are due at once, one save per lane
        // (several elements per thread have no registers for them)
        for (int m = due(t_new); m > 0; m = due(t_new)) {
          CTab *wr = weights<TAB>();
          const double th = (ts - t) / h;
          double wl[7];
#pragma unroll
          for (int j = 0; j < 7; ++j)
            wl[j] = th * (wr->R[j][0] + th * (wr->R[j][1] + th * (wr->R[j][2] + th * wr->R[j][3])));
          fold_k0(wl);
          for (; m > 0; --m, ++isave) {
            double w[7];
#pragma unroll
            for (int j = 0; j < 7; ++j) w[j] = lane_of(wl[j], isave - sbase);
            save(h, w, isave);
          }
          if (isave == sbase + 64) {
            sbase = isave;
            ts = sbase + lane < ntsave ? tsave[sbase + lane] : 0.0;
          }
        }
      } else {
        while (isave < ntsave && next_save <= t_new) {
          const double th = (next_save - t) / h;
          CTab *wr = weights<TAB>();
          double w[7];
#pragma unroll
          for (int j = 0; j < 7; ++j)
            w[j] = th * (wr->R[j][0] + th * (wr->R[j][1] + th * (wr->R[j][2] + th * wr->R[j][3])));
          fold_k0(w);
#pragma unroll
          for (int j = 0; j < 7; ++j) w[j] = uniform<(NE > 1)>(w[j]);
          save(h, w, isave);
          advance();
        }
      }
#pragma unroll
      for (int q = 0; q < NE; ++q) {
        k[0][q] = k[6][q];
        y[q] = y1[q];
      }
      t = uniform<(NE > 1)>(t_new);
      need_k0 = made_jump;
    } else {
      ++nrej;
    }
    dt = uniform<(NE > 1)>(factor * h);
  }
  for (; isave < ntsave; ++isave) save(0.0, w0, isave);
  float2 *fin = gp<float2>(p.final_state);
  float2 *st = gp<float2>(p.states);
#pragma unroll
  for (int q = 0; q < NE; ++q) {
    int i, j;
    if (at(q, i, j)) {
      const float2 v = make_float2((float)y[q].x, (float)y[q].y), vc = make_float2(v.x, -v.y);
      fin[(size_t)i * n + j] = v;
      if (i != j) fin[(size_t)j * n + i] = vc;
      if (!save_states) {
        st[(size_t)i * n + j] = v;
        if (i != j) st[(size_t)j * n + i] = vc;
      }
    }
  }
  if (tid == 0) {
    stats[0] = nsteps;
    stats[1] = nacc;
    stats[2] = nrej;
    stats[3] = status;
    stats[4] = nrhs;
  }
}

// The same solve with the coefficients read from LDS tables at every evaluation (one copy
// of the stage input, two barriers per stage): for 64 < n < 128, for more than kMaxShift
// shifts, and for modulated terms, whose tables are rebuilt at every stage time. The terms
// are an outer loop, so that each one keeps NE independent reads in flight. KM: the stages
// and the state are in global memory (work: 7 NU float2, y: NU double2, in owner order; L2
// serves them), for n > 90, where they do not fit the registers.
// Bound by the LDS reads, three 8-byte ones per term and element. 48 two-mode problems of
// n = 81 (10 parts, about 150 steps): 61.2 -> 2.12 ms against the dense body; 32 problems
// of n = 127 with one jump diagonal, 8 steps: 12.7 -> 1.28 ms (memory form).
template <int NTH, int NE, bool KM, int TAB>
__global__ __launch_bounds__(NTH) void k_tsit5_diag_tab(const dqh_me_inst *__restrict__ insts, Pattern pat) {
  extern __shared__ __align__(16) char smem[];
  const dqh_me_inst &p = insts[blockIdx.x];
  constexpr RKTab rk = kRKTabs[TAB];
  constexpr int QC = NE < 2 ? NE : 2;
  const int n = (int)p.n, np = (int)p.np, nE = (int)p.nE, ntsave = (int)p.ntsave, nseg = (int)p.nseg;
  const int LD = row_stride(n), NLD = n * LD, tid = (int)threadIdx.x;
  const int npwc = (int)p.npwc, nmod = (int)p.nmod;
  const bool pwc = npwc > 0, smooth = nmod > 0;
  double2 *dcur = reinterpret_cast<double2 *>(smem);
  double *red = reinterpret_cast<double *>(dcur + n);
  float2 *ys = reinterpret_cast<float2 *>(red + 4 * (NTH / 64));
  float2 *Gt = ys + NLD + 1;
  float2 *Lt = Gt + pat.nH * n;
  int64_t *stats = gp<int64_t>(p.stats);
  const int NU = n * (n + 1) / 2;
  if (n >= 128 || NU > NTH * NE || nmod > DQH_MAX_MOD || (pwc && nseg < 2) || (smooth && p.mod_nint < 1) ||
      (KM && !p.work) || (p.flags & (DQH_FLAG_GLOBAL | DQH_FLAG_LMOD | DQH_FLAG_DOPRI8 | DQH_FLAG_EULER)) ||
      ((p.flags & DQH_FLAG_DOPRI5) != 0) != (TAB == 1)) {
    if (tid == 0) stats[3] = DQH_UNSUPPORTED;
    return;
  }
  const double *tsave = gp<const double>(p.tsave);
  const double *ptimes = gp<const double>(p.pwc_times);
  const double rtol = p.rtol, atol = p.atol, t_end = p.t1;
  const double inv_nn = uniform<(NE > 1)>(1.0 / ((double)n * n));
  const bool save_states = (p.flags & DQH_FLAG_SAVE_STATES) != 0;

  // owned elements, packed i | j << 8 (i <= j; -1 past the end)
  int ij[NE];
#pragma unroll
  for (int q = 0; q < NE; ++q) {
    int rem = tid + NTH * q, i = 0;
    ij[q] = -1;
    if (rem < NU) {
      while (rem >= n - i) {
        rem -= n - i;
        ++i;
      }
      ij[q] = i | ((i + rem) << 8);
    }
  }
  // row and column of element q (0, 0 past the end), formed where they are used
  auto at = [&](int q, int &i, int &j) {
    int x = ij[q];
    asm volatile("" : "+v"(x));
    x = max(x, 0);
    i = x & 255;
    j = x >> 8;
  };
  for (int e = tid; e <= NLD; e += NTH) ys[e] = make_float2(0.f, 0.f);
  for (int e = tid; e < pat.nLrow * n; e += NTH) {
    const int r = e / n, i = e - r * n;
    Lt[e] = gp<const float2>(p.Dops)[(size_t)r * np + i];
  }
  // Gt, dcur <- the constant generator + the PWC terms of segment seg + f_j(tau) O_j
  auto tables = [&](int seg, double tau) {
    const float2 *G0 = gp<const float2>(p.Hnh);
    const double2 *d0g = gp<const double2>(p.hdiag);
    const float2 *Hp = gp<const float2>(p.Hpwc), *Hm = gp<const float2>(p.Hmod);
    const double *vals = gp<const double>(p.pwc_vals);
    const int nv = nseg - 1, rows = pat.nH + 1;
    const bool inside = pwc && seg >= 0 && seg < nv;
    double2 fm[DQH_MAX_MOD];
#pragma unroll
    for (int j = 0; j < DQH_MAX_MOD; ++j) fm[j] = make_double2(0.0, 0.0);
    if (smooth) {
      const int64_t nint = p.mod_nint;
      int64_t m = (int64_t)floor((tau - p.mod_t0) / p.mod_dt);
      m = m < 0 ? 0 : (m >= nint ? nint - 1 : m);
      const double x = tau - (p.mod_t0 + (double)m * p.mod_dt);
#pragma unroll
      for (int j = 0; j < DQH_MAX_MOD; ++j) {
        if (j < nmod) {
          const double2 *c = gp<const double2>(p.mod_coef) + ((size_t)j * nint + m) * 4;
          double re = c[0].x, im = c[0].y;
#pragma unroll
          for (int d = 1; d < 4; ++d) {
            re = re * x + c[d].x;
            im = im * x + c[d].y;
          }
          fm[j] = make_double2(re, im);
        }
      }
    }
    for (int e = tid; e < rows * n; e += NTH) {
      const int r = e / n, i = e - r * n;
      const size_t w = (size_t)r * np + i, stride = (size_t)rows * np;
      double re, im;
      if (r < pat.nH) {
        const float2 o = G0[w];
        re = o.x;
        im = o.y;
      } else {
        re = d0g[i].x;
        im = d0g[i].y;
      }
      if (inside) {
        for (int j = 0; j < npwc; ++j) {
          const double vr = vals[2 * (j * nv + seg)], vi = vals[2 * (j * nv + seg) + 1];
          const float2 o = Hp[j * stride + w];
          re += vr * o.x - vi * o.y;
          im += vr * o.y + vi * o.x;
        }
      }
#pragma unroll
      for (int j = 0; j < DQH_MAX_MOD; ++j) {
        if (j < nmod) {
          const float2 o = Hm[j * stride + w];
          re += fm[j].x * o.x - fm[j].y * o.y;
          im += fm[j].x * o.y + fm[j].y * o.x;
        }
      }
      if (r < pat.nH)
        Gt[e] = make_float2((float)re, (float)im);
      else
        dcur[i] = make_double2(re, im);
    }
  };

  // state and stages: registers, or global memory in owner order (KM)
  double2 yr[KM ? 1 : NE], v[NE];
  float2 kr[KM ? 1 : 7][KM ? 1 : NE];
  double2 *const ym = gp<double2>(p.y) + (size_t)np * np;
  float2 *const km = gp<float2>(p.work);
  int k0 = 0, k6 = 6;  // KM: slots of stages 0 and 6, swapped on accepted steps
  // a uniform base per access and the thread as a 32-bit lane offset (the opaque zero keeps
  // the bases from being formed ahead and held)
  auto slot = [&](int j, int q) -> float2 * {
    int u = (j == 0 ? k0 : (j == 6 ? k6 : j)) * NU + NTH * q;
    asm volatile("" : "+s"(u));
    return km + u + (unsigned)tid;
  };
  auto own = [&](int q) { return tid + NTH * q < NU; };
  auto yget = [&](int q) -> double2 {
    if constexpr (KM)
      return own(q) ? (ym + NTH * q)[(unsigned)tid] : make_double2(0.0, 0.0);
    else
      return yr[q];
  };
  auto yset = [&](int q, double2 x) {
    if constexpr (KM) {
      if (own(q)) (ym + NTH * q)[(unsigned)tid] = x;
    } else {
      yr[q] = x;
    }
  };
  auto kget = [&](int j, int q) -> float2 {
    if constexpr (KM)
      return own(q) ? *slot(j, q) : make_float2(0.f, 0.f);
    else
      return kr[j][q];
  };
  auto kset = [&](int j, int q, float2 x) {
    if constexpr (KM) {
      if (own(q)) *slot(j, q) = x;
    } else {
      kr[j][q] = x;
    }
  };
  {
    const double2 *y0 = gp<const double2>(p.y);
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      int i, j;
      at(q, i, j);
      double2 x = own(q) ? y0[(size_t)i * np + j] : make_double2(0.0, 0.0);
      if (i == j) x.y = 0.0;
      yset(q, x);
      v[q] = make_double2(0.0, 0.0);
#pragma unroll
      for (int s = 0; s < 7; ++s) kset(s, q, make_float2(0.f, 0.f));
    }
  }

  // k_s = f(v), with the tables rebuilt at (seg, tau) when asked
  auto field = [&](int s, bool rebuild, int seg, double tau) {
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      int i, j;
      at(q, i, j);
      const float2 x = make_float2((float)v[q].x, (float)v[q].y);
      const bool on = own(q);
      ys[on ? j * LD + i : NLD] = make_float2(x.x, -x.y);
      ys[on ? i * LD + j : NLD] = x;
    }
    if (rebuild) tables(seg, tau);
    __syncthreads();
    // QC elements at a time: each term keeps their reads in flight
#pragma unroll
    for (int c = 0; c < NE; c += QC) {
      const int nq = NE - c < QC ? NE - c : QC;  // constant once unrolled
      float fr[QC], fi[QC];
      int i[QC], j[QC];
#pragma unroll
      for (int q = 0; q < nq; ++q) {
        fr[q] = fi[q] = 0.f;
        at(c + q, i[q], j[q]);
      }
#pragma unroll 2
      for (int x = 0; x < pat.nH; ++x) {
        const int o = pat.offH[x];
#pragma unroll
        for (int q = 0; q < nq; ++q) {
          const float2 cr = Gt[x * n + i[q]], cc = Gt[x * n + j[q]];
          const int e = i[q] * LD + j[q];
          const float2 a = ys[min(max(e + o * LD, 0), NLD)], b = ys[min(max(e + o, 0), NLD)];
          fr[q] = fmaf(cr.x, a.x, fmaf(-cr.y, a.y, fmaf(cc.x, b.x, fmaf(cc.y, b.y, fr[q]))));
          fi[q] = fmaf(cr.x, a.y, fmaf(cr.y, a.x, fmaf(cc.x, b.y, fmaf(-cc.y, b.x, fi[q]))));
        }
      }
#pragma unroll 2
      for (int x = 0; x < pat.npair; ++x) {
        const Part pr = pat.pair[x];
        const int sh = pat.pa[x] * LD + pat.pb[x];
#pragma unroll
        for (int q = 0; q < nq; ++q) {
          const float2 l = Lt[pr.x * n + i[q]], m = Lt[pr.y * n + j[q]];
          const float2 z = ys[min(max(i[q] * LD + j[q] + sh, 0), NLD)];
          const float cr = l.x * m.x + l.y * m.y, ci = l.y * m.x - l.x * m.y;
          fr[q] = fmaf(cr, z.x, fmaf(-ci, z.y, fr[q]));
          fi[q] = fmaf(cr, z.y, fmaf(ci, z.x, fi[q]));
        }
      }
#pragma unroll
      for (int q = 0; q < nq; ++q) {
        const double2 da = dcur[i[q]], db = dcur[j[q]];
        double gr = da.x + db.x, gi = da.y - db.y;
#pragma unroll 1
        for (int x = 0; x < pat.nzero; ++x) {  // products of the main diagonals, in FP64
          const float2 l = Lt[pat.zero[x].x * n + i[q]], m = Lt[pat.zero[x].y * n + j[q]];
          gr += (double)l.x * m.x + (double)l.y * m.y;
          gi += (double)l.y * m.x - (double)l.x * m.y;
        }
        const double2 u = v[c + q];
        const double re = (double)fr[q] + (gr * u.x - gi * u.y);
        const double im = (double)fi[q] + (gr * u.y + gi * u.x);
        kset(s, c + q, make_float2((float)re, i[q] == j[q] ? 0.f : (float)im));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();  // the next stage overwrites ys
  };

  int par = 0;
  // as in k_tsit5_diag: one element at a time, formed anew for every operator
  auto save = [&](double h, const double (&w)[7], int isave) {
    float2 *st = gp<float2>(p.states) + (size_t)isave * n * n;
    auto value = [&](int q) {
      const double2 y = yget(q);
      double re = 0.0, im = 0.0;
      if (h != 0.0) {
#pragma unroll
        for (int j = 0; j < 7; ++j) {
          float2 x = kget(j, q);
          asm volatile("" : "+v"(x.x), "+v"(x.y));
          re += w[j] * (double)x.x;
          im += w[j] * (double)x.y;
        }
      }
      return make_double2(y.x + h * re, y.y + h * im);
    };
    if (save_states) {
#pragma unroll
      for (int q = 0; q < NE; ++q) {
        const double2 v = value(q);
        int i, j;
        at(q, i, j);
        if (own(q)) {
          st[(size_t)i * n + j] = make_float2((float)v.x, (float)v.y);
          if (i != j) st[(size_t)j * n + i] = make_float2((float)v.x, (float)-v.y);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    const float2 *ET = gp<const float2>(p.EopsT);
    for (int e = 0; e < nE; ++e) {
      const float2 *E = ET + (size_t)e * np * np;
      double s[2] = {0.0, 0.0};
#pragma unroll
      for (int q = 0; q < NE; ++q) {
        const double2 v = value(q);
        if (own(q)) {
          int i, j;
          at(q, i, j);
          const float2 o = E[(size_t)i * np + j];
          s[0] += o.x * v.x - o.y * v.y;
          s[1] += o.x * v.y + o.y * v.x;
          if (i != j) {
            const float2 m = E[(size_t)j * np + i];
            s[0] += m.x * v.x + m.y * v.y;
            s[1] += m.y * v.x - m.x * v.y;
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      block_sums<NTH>(s, red, par);
      if (tid == 0) gp<float2>(p.expects)[(size_t)e * ntsave + isave] = make_float2((float)s[0], (float)s[1]);
    }
  };
  const double w0[7] = {0, 0, 0, 0, 0, 0, 0};
  auto weight = [&](int q) {
    int i, j;
    at(q, i, j);
    return !own(q) ? 0.0 : (i == j ? 1.0 : 2.0);
  };

  double t = p.t0;
  int isave = 0, status = 0;
  int64_t nsteps = 0, nacc = 0, nrej = 0, nrhs = 0;
  double next_save = ntsave > 0 ? tsave[0] : 0.0;
  auto advance = [&]() {
    ++isave;
    if (isave < ntsave) next_save = uniform<(NE > 1)>(tsave[isave]);
  };
  int seg = -1;
  double next_break = pwc ? ptimes[0] : 0.0;
  auto locate = [&]() {
    bool moved = false;
    while (seg + 1 < nseg && next_break <= t) {
      ++seg;
      moved = true;
      if (seg + 1 < nseg) next_break = ptimes[seg + 1];
    }
    return moved;
  };
  if (pwc) locate();
  __syncthreads();  // the tables and the zeroed copy
  while (isave < ntsave && next_save <= t) {
    save(0.0, w0, isave);
    advance();
  }
#pragma unroll
  for (int q = 0; q < NE; ++q) v[q] = yget(q);
  field(0, true, seg, t);
  ++nrhs;

  double dt;  // initial step, as in k_tsit5_diag
  {
    double s[2] = {0.0, 0.0};
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      const float2 kq = kget(0, q);
      const double ay2 = v[q].x * v[q].x + v[q].y * v[q].y;
      const double sc = atol + rtol * sqrt(ay2);
      s[0] += weight(q) * ay2 / (sc * sc);
      s[1] += weight(q) * ((double)kq.x * kq.x + (double)kq.y * kq.y) / (sc * sc);
    }
    block_sums<NTH>(s, red, par);
    const double d0 = sqrt(s[0] * inv_nn), d1 = sqrt(s[1] * inv_nn);
    const double h0 = (d0 < 1e-5 || d1 < 1e-5) ? 1e-6 : 0.01 * d0 / d1;
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      const float2 kq = kget(0, q);
      v[q] = make_double2(v[q].x + h0 * kq.x, v[q].y + h0 * kq.y);
    }
    field(1, smooth, seg, t + h0);
    ++nrhs;
    double s2[1] = {0.0};
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      const double2 y = yget(q);
      const float2 ka = kget(0, q), kb = kget(1, q);
      const double sc = atol + rtol * sqrt(y.x * y.x + y.y * y.y);
      const double dr = (double)kb.x - ka.x, di = (double)kb.y - ka.y;
      s2[0] += weight(q) * (dr * dr + di * di) / (sc * sc);
    }
    block_sums<NTH>(s2, red, par);
    const double d2 = sqrt(s2[0] * inv_nn) / h0;
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
    bool fresh = pwc && locate();  // the tables of the new segment, rebuilt with the next field
    if (need_k0) {
#pragma unroll
      for (int q = 0; q < NE; ++q) v[q] = yget(q);
      field(0, fresh || smooth, seg, t);
      fresh = false;
      ++nrhs;
      need_k0 = false;
    }
    double h = dt, target = t_end;
    bool target_jump = false;
    if (pwc && seg + 1 < nseg && next_break < t_end) {
      target = next_break;
      target_jump = true;
    }
    bool made_jump = false;
    double t_new = t + h;
    if (snaps_to(t, h, target)) {
      h = target - t;
      t_new = target;
      made_jump = target_jump;
    }
    h = uniform<(NE > 1)>(h);
    t_new = uniform<(NE > 1)>(t_new);
    if (!(h > 0.0) || !(h > 1e-14 * fmax(1.0, fabs(t)))) {
      status = DQH_NONFINITE;
      break;
    }
    // the increment form of k_tsit5_diag for constant generators (stages 1..5 on the
    // increment alone); modulated ones evaluate every stage at the full input
#pragma unroll
    for (int s = 1; s < 7; ++s) {
      CTab *w = weights<TAB>();
      const double a0 = smooth ? w->A[s][0] : w->C[s];
      if constexpr (!KM && NE > 1) {  // as pin_stages in k_tsit5_diag
#pragma unroll
        for (int j = 0; j < s; ++j)
#pragma unroll
          for (int q = 0; q < NE; ++q) asm volatile("" : "+v"(kr[j][q].x), "+v"(kr[j][q].y));
      }
#pragma unroll
      for (int q = 0; q < NE; ++q) {
        if constexpr (KM || NE > 2) __builtin_amdgcn_sched_barrier(0);
        const float2 ka = kget(0, q);
        double re = a0 * (double)ka.x, im = a0 * (double)ka.y;
#pragma unroll
        for (int j = 1; j < s; ++j) {
          if (rk.A[s][j] != 0.0) {
            const float2 kq = kget(j, q);
            re += w->A[s][j] * (double)kq.x;
            im += w->A[s][j] * (double)kq.y;
          }
        }
        double2 y = make_double2(0.0, 0.0);
        if (smooth || s == 6) y = yget(q);
        v[q] = make_double2(y.x + h * re, y.y + h * im);
      }
      field(s, smooth || fresh, seg, t + w->C[s] * h);
      fresh = false;
    }
    nrhs += 6;
    CTab *we = weights<TAB>();
    double ss[1] = {0.0};
    double e0 = we->E[0];
    if (!smooth) {
#pragma unroll
      for (int j = 1; j < 6; ++j) e0 += we->E[j];
    }
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      const float2 ka = kget(0, q);
      const double2 y = yget(q);
      double er = e0 * (double)ka.x, em = e0 * (double)ka.y;
#pragma unroll
      for (int j = 1; j < 7; ++j) {
        if (rk.E[j] != 0.0) {
          const float2 kq = kget(j, q);
          er += we->E[j] * (double)kq.x;
          em += we->E[j] * (double)kq.y;
        }
      }
      er *= h;
      em *= h;
      const double sc = atol + rtol * sqrt(fmax(y.x * y.x + y.y * y.y, v[q].x * v[q].x + v[q].y * v[q].y));
      ss[0] += weight(q) * (er * er + em * em) / (sc * sc);
      if constexpr (KM || NE > 2) __builtin_amdgcn_sched_barrier(0);
    }
    block_sums<NTH>(ss, red, par);
    const double norm = sqrt(ss[0] * inv_nn);
    const bool finite = isfinite(norm);
    const bool keep = finite && norm < 1.0;
    double factor;
    if (!finite)
      factor = p.factormin;
    else if (norm == 0.0)
      factor = p.factormax;
    else
      factor = p.safety * ctrl_pow(norm, -0.2);
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
        if (!smooth) fold_k0(w);
#pragma unroll
        for (int j = 0; j < 7; ++j) w[j] = uniform<(NE > 1)>(w[j]);
        save(h, w, isave);
        advance();
      }
#pragma unroll
      for (int q = 0; q < NE; ++q) {
        if constexpr (!KM) kr[0][q] = kr[6][q];
        yset(q, v[q]);
      }
      const int sw = k0;
      k0 = k6;
      k6 = sw;
      t = t_new;
      need_k0 = made_jump;
    } else {
      ++nrej;
    }
    dt = uniform<(NE > 1)>(factor * h);
  }
  while (isave < ntsave) {
    save(0.0, w0, isave);
    advance();
  }
  float2 *fin = gp<float2>(p.final_state);
  float2 *st = gp<float2>(p.states);
#pragma unroll
  for (int q = 0; q < NE; ++q) {
    if (own(q)) {
      int i, j;
      at(q, i, j);
      const double2 y = yget(q);
      const float2 x = make_float2((float)y.x, (float)y.y), xc = make_float2(x.x, -x.y);
      fin[(size_t)i * n + j] = x;
      if (i != j) fin[(size_t)j * n + i] = xc;
      if (!save_states) {
        st[(size_t)i * n + j] = x;
        if (i != j) st[(size_t)j * n + i] = xc;
      }
    }
  }
  if (tid == 0) {
    stats[0] = nsteps;
    stats[1] = nacc;
    stats[2] = nrej;
    stats[3] = status;
    stats[4] = nrhs;
  }
}

// Shifts of the operators' stencil and the parts of their coefficients, sorted by shift
// (so that an operator set and its zero-extended superset add up in the same order).
// nterm is kMaxShift + 1 when there are more shifts than the register form holds. False
// when the parts exceed kMaxPart.
bool make_pattern(const dqh_dia_ops &ops, int n, Pattern &pt) {
  std::memset(&pt, 0, sizeof(pt));
  std::vector<std::pair<std::pair<int, int>, Part>> parts;
  pt.nH = ops.noff[0];
  for (int x = 0; x < ops.noff[0]; ++x) {
    const int o = ops.off[0][x];
    if (o == 0) return false;  // the main diagonal goes in hdiag
    pt.offH[x] = o;
    parts.push_back({{o, 0}, Part{0, (uint8_t)x, 0, 0}});
    parts.push_back({{0, o}, Part{1, (uint8_t)x, 0, 0}});
  }
  int row = 0;
  for (int s = 1; s < ops.nops; ++s) {
    for (int u = 0; u < ops.noff[s]; ++u)
      for (int v = 0; v < ops.noff[s]; ++v) {
        const int a = ops.off[s][u], b = ops.off[s][v];
        const Part part{2, (uint8_t)(row + u), (uint8_t)(row + v), 0};
        if (a == 0 && b == 0) {
          if (pt.nzero >= kMaxPart) return false;
          pt.zero[pt.nzero++] = part;
        } else {
          if (pt.npair >= kMaxPart) return false;
          pt.pa[pt.npair] = (int16_t)a;
          pt.pb[pt.npair] = (int16_t)b;
          pt.pair[pt.npair++] = part;
          parts.push_back({{a, b}, part});
        }
      }
    row += ops.noff[s];
  }
  pt.nLrow = row;
  if ((int)parts.size() > kMaxPart) return false;
  std::stable_sort(parts.begin(), parts.end(), [](const auto &l, const auto &r) { return l.first < r.first; });
  for (size_t i = 0; i < parts.size(); ++i) {
    if (i == 0 || parts[i].first != parts[i - 1].first) {
      if (pt.nterm >= kMaxShift) {
        pt.nterm = kMaxShift + 1;
        return true;
      }
      pt.a[pt.nterm] = parts[i].first.first;
      pt.b[pt.nterm] = parts[i].first.second;
      pt.first[pt.nterm++] = (int32_t)i;
    }
    pt.part[i] = parts[i].second;
  }
  for (int t = pt.nterm; t <= kMaxShift; ++t) pt.first[t] = (int32_t)parts.size();
  for (int t = 0; t < pt.nterm; ++t) pt.guard = std::max(pt.guard, std::abs(pt.a[t] * row_stride(n) + pt.b[t]));
  return true;
}

template <int NTH, int NE, int T, int TAB>
int launch(const dqh_me_inst *d, int64_t ninst, int n, const Pattern &pt, hipStream_t st) {
  const size_t lds = lds_bytes<NTH>(n, pt.nH, pt.nLrow, pt.guard);
  const void *fn = reinterpret_cast<const void *>(&k_tsit5_diag<NTH, NE, T, TAB>);
  hipError_t err = hipSuccess;
  if (lds > 65536) err = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (err == hipSuccess) {
    hipLaunchKernelGGL((k_tsit5_diag<NTH, NE, T, TAB>), dim3((unsigned)ninst), dim3(NTH), lds, st, d, pt);
    err = hipGetLastError();
  }
  return err == hipSuccess ? DQH_OK : fail(DQH_HIP_ERROR, std::string("dqh_mesolve_tsit5_diag: ") + hipGetErrorString(err));
}

template <int T, int TAB>
int launch_size(const dqh_me_inst *d, int64_t ninst, int n, const Pattern &pt, hipStream_t st) {
  const int nu = n * (n + 1) / 2;
  // One element per thread up to nine waves. The class above 192 elements is wide: at n = 20
  // to 22 four waves would do, at n = 23 to 27 six (a driven oscillator, one instance 71 us,
  // 54 with 256 threads and 62 with 384; 1000 instances 322 us, 131 and 265).
  if (nu <= 64) return launch<64, 1, T, TAB>(d, ninst, n, pt, st);
  if (nu <= 192) return launch<192, 1, T, TAB>(d, ninst, n, pt, st);
  if (nu <= 576) return launch<576, 1, T, TAB>(d, ninst, n, pt, st);
  if (nu <= 1152) return launch<576, 2, T, TAB>(d, ninst, n, pt, st);
  return launch<704, 3, T, TAB>(d, ninst, n, pt, st);
}

template <int NTH, int NE, bool KM, int TAB>
int launch_tab(const dqh_me_inst *d, int64_t ninst, int n, const Pattern &pt, hipStream_t st) {
  const size_t lds = (size_t)(n * row_stride(n) + 1 + (pt.nH + pt.nLrow) * n) * sizeof(float2) +
                     (size_t)n * sizeof(double2) + (size_t)(4 * (NTH / 64)) * sizeof(double);
  const void *fn = reinterpret_cast<const void *>(&k_tsit5_diag_tab<NTH, NE, KM, TAB>);
  hipError_t err = hipSuccess;
  if (lds > 160 * 1024) return fail(DQH_BAD_SHAPE, "dqh_mesolve_tsit5_diag: the operators' diagonals exceed the LDS");
  if (lds > 65536) err = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (err == hipSuccess) {
    hipLaunchKernelGGL((k_tsit5_diag_tab<NTH, NE, KM, TAB>), dim3((unsigned)ninst), dim3(NTH), lds, st, d, pt);
    err = hipGetLastError();
  }
  return err == hipSuccess ? DQH_OK : fail(DQH_HIP_ERROR, std::string("dqh_mesolve_tsit5_diag: ") + hipGetErrorString(err));
}

template <int TAB>
int launch_tab_size(const dqh_me_inst *d, int64_t ninst, int n, const Pattern &pt, hipStream_t st) {
  const int nu = n * (n + 1) / 2;
  if (nu <= 576) return launch_tab<576, 1, false, TAB>(d, ninst, n, pt, st);
  if (nu <= 2048) return launch_tab<1024, 2, false, TAB>(d, ninst, n, pt, st);
  // 704 threads (11 waves) have 168 registers each, which hold the stages of 4 elements and
  // nearly those of 5; 1024 have 128 (48 two-mode solves: n = 72 2.98 ms with 1024 threads,
  // 1.61 with 704; n = 81 2.93 and 2.12). In memory, the fewest elements per thread that cover
  // the triangle (n = 100: 8.1 ms with 8, 4.5 with 5).
  if (nu <= 2816) return launch_tab<704, 4, false, TAB>(d, ninst, n, pt, st);
  if (nu <= 3520) return launch_tab<704, 5, false, TAB>(d, ninst, n, pt, st);
  if (nu <= 4096) return launch_tab<1024, 4, false, TAB>(d, ninst, n, pt, st);
  if (nu <= 5120) return launch_tab<1024, 5, true, TAB>(d, ninst, n, pt, st);
  if (nu <= 6144) return launch_tab<1024, 6, true, TAB>(d, ninst, n, pt, st);
  return launch_tab<1024, 8, true, TAB>(d, ninst, n, pt, st);
}

}  // namespace diag
}  // namespace dqh

using namespace dqh;

extern "C" int dqh_mesolve_tsit5_diag(const dqh_me_inst *d_insts, int64_t ninst, int64_t n, const dqh_dia_ops *ops,
                                      int64_t flags, int64_t modulated, void *stream) {
  if (!d_insts || !ops || ninst <= 0 || ninst > (1 << 30))
    return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_diag: bad arguments");
  if (n <= 0 || n >= 128) return fail(DQH_BAD_SHAPE, "dqh_mesolve_tsit5_diag: 1 <= n < 128");
  if (ops->nops < 1 || ops->nops > DQH_DIA_MAXOPS)
    return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_diag: 1 <= nops <= 8 (the generator, then the jump operators)");
  for (int s = 0; s < ops->nops; ++s) {
    if (ops->noff[s] < 0 || ops->noff[s] > DQH_DIA_MAXOFF)
      return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_diag: bad number of diagonals");
    for (int u = 0; u < ops->noff[s]; ++u)
      if (ops->off[s][u] <= -n || ops->off[s][u] >= n)
        return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_diag: offset outside (-n, n)");
  }
  diag::Pattern pt;
  if (!diag::make_pattern(*ops, (int)n, pt))
    return fail(DQH_BAD_SHAPE, "dqh_mesolve_tsit5_diag: at most 48 parts and no main diagonal in operator 0");
  hipStream_t st = (hipStream_t)stream;
  const bool dopri5 = (flags & DQH_FLAG_DOPRI5) != 0;
  // the register form for what fits its registers and LDS (the guards of far shifts) and is
  // constant over a step; the table form for the rest
  if (n > 64 || pt.nterm > diag::kMaxShift || modulated ||
      diag::lds_bytes<704>((int)n, pt.nH, pt.nLrow, pt.guard) > 150 * 1024)
    return dopri5 ? diag::launch_tab_size<1>(d_insts, ninst, (int)n, pt, st)
                  : diag::launch_tab_size<0>(d_insts, ninst, (int)n, pt, st);
  if (pt.nterm <= 6)
    return dopri5 ? diag::launch_size<6, 1>(d_insts, ninst, (int)n, pt, st)
                  : diag::launch_size<6, 0>(d_insts, ninst, (int)n, pt, st);
  return dopri5 ? diag::launch_size<12, 1>(d_insts, ninst, (int)n, pt, st)
                : diag::launch_size<12, 0>(d_insts, ninst, (int)n, pt, st);
}
