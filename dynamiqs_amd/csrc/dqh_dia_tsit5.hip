// Adaptive Tsit5 / Dopri5 for sparse-DIA master equations (gfx950).
//
// The large-n counterpart of the persistent dense kernel: a state of n = 1024
// does not fit one workgroup, so every stage is one grid-wide launch over all
// instances and the step controller lives on the device. Every launch is bound by HBM
// (or, for small batches, by the latency of one launch), so the design counts bytes:
//   * a Hermitian rho0 stays Hermitian, so only the upper triangle is swept (64-column
//     strips of 4 NE rows). Stencil reads may cross the diagonal by at most `spread`
//     elements; the writers keep that band below the diagonal up to date. A rho0 that is
//     not Hermitian (checked on the device) takes the same kernels over the full matrix;
//   * stage 1 forms its input y + h a_10 k_0 where the stencil reads it, so that no pass
//     over the matrix has to follow the choice of h;
//   * stage 5 writes the candidate y1 in FP64 (a second state buffer) and stage 6 reads
//     its stencil input from it, so accepting a step moves nothing: the buffers swap roles;
//   * accept / reject, saves and the next dt are formed at the start of the next step's
//     stage 1, by every workgroup from the same partial sums in the same order (identical
//     decisions everywhere, no atomics).
// Bytes per element and step: 40 + 56 + 64 + 72 + 88 + 88 = 408, of half the elements,
// against 496 of all of them with full-matrix sweeps and a commit pass. The stages are
// evaluated on the rounded states y + Delta_s as before: on the increments alone (344 bytes,
// about 1 ms less below) the error estimate loses the FP32 noise that holds the steps down in the
// full-matrix form, and the solutions moved by up to 8e-3 of the largest elements' scale.
// The order of rounding within a field is that of the full-matrix form too (stencil below).
// Measured (rtol 1e-6, atol 1e-8, two coupled modes with 8 shifts): four solves of n = 1024,
// 36 steps, 21.7 -> 7.4 ms, stages at 3.8 to 5.3 TB/s (a copy reaches 4.7); one of
// n = 323, 29 steps, 2.4 -> 1.2 ms, bound by the latency of a launch (about 5 us).
// Time-dependent Hamiltonians take a separate controller launch before the first stage,
// because their diagonals are rebuilt in between.
//
// Control blocks are double-buffered by step parity (a step reads the other block and
// writes block `cur`), so a fixed sequence of launches is valid for any step and is
// captured once as a hipGraph of graph_steps steps and replayed. Instances keep their own
// t, dt, counters and save cursor; an instance that is done turns every later launch into
// an early return. The host loop reads a completion count after each replay; max_steps
// bounds the number of replays. Semantics follow diffrax_integrator.py:59-81, 101-147
// (Tsit5 + PID controller + SaveAt dense output) as the dense kernel implements them.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>

#include "dqh.h"
#include "dqh_common.h"
#include "dqh_dia_tile.h"
#include "dqh_dia_tri.h"
#include "dqh_expect.h"
#include "dqh_tsit5_tableau.h"

namespace dqh {
namespace diats {

using namespace tri;

struct Ctrl {
  double t, dt;
  int64_t nsteps, nacc, nrej, status, isave, rot;  // rot: slot of k_0 in the 7 stage buffers, and the flags below
};
static_assert(sizeof(Ctrl) == 64, "control block is 64 bytes");

// Ctrl::rot: slot of k_0 (bits 0-2), and
constexpr int64_t kJump = 8;    // the last accepted step ended on a PWC breakpoint: k_0 is evaluated anew
constexpr int64_t kFresh = 16;  // no attempt to commit yet
constexpr int64_t kSel = 32;    // the state is in the second FP64 buffer

// A shift of a jump operator: f[i][j] += r[i + p] z, z = go z_before + X[i + p][j + q] conj(c[j + q]).
// The column offsets of a row offset share its factor: go = 1 from the second on, and r is a
// vector of zeros but for the last.
struct Term {
  const float2 *r, *c;
  int32_t p, q;
  float go;
  int32_t pad;
};
static_assert(sizeof(Term) == 32, "terms are read as 32-byte scalars");
constexpr int kMaxTerm = (DQH_DIA_MAXOPS - 1) * DQH_DIA_MAXOFF * DQH_DIA_MAXOFF;
constexpr int kHead = 4;  // terms in the kernel arguments: one round trip less than from the list

struct V {
  int64_t n, n_true, ninst, nsave, max_steps, npart, flags;
  int32_t herm, spread, npair, nterm, nb, total;  // nb: 64-element blocks per side; total: tiles per instance
  int32_t presum;  // the control blocks are formed by k_ctl
  int32_t off[DQH_DIA_MAXOFF];  // offsets of the generator (operator 0): npair of them
  Term head[kHead];             // the first of the nterm terms
  double rtol, atol, safety, fmin_, fmax_, t0, t1, inv_nn;
  float2 *k;      // [7][ninst][n][n]
  float2 *ys;     // [2][ninst][n][n]
  double2 *y2;    // [ninst][n][n]: second FP64 state
  Term *terms;    // [nterm]
  float2 *zeros;  // [n]
  double *part;   // [ninst][2][npart]
  Ctrl *ctrl;     // [2][ninst]
  int64_t *flag;  // completion count; before the first step: rho0 is not Hermitian
  double2 *y;     // [ninst][n][n]
  const double *tsave;
  float2 *states;
  int64_t *stats;
  // time-dependent Hamiltonian terms (npwc + nmod > 0): hcur[inst] holds the
  // diagonals of Hnh at the current stage time on the noff0 offsets of operator 0
  int64_t npwc, nseg, nmod, noff0, mod_nint;
  double mod_t0, mod_dt;
  const double *ptimes;
  const double *pvals;
  const double2 *mcoef;
  const float2 *H0;
  const float2 *Hterms;
  float2 *hcur;
};

__device__ __forceinline__ bool is_done(const Ctrl &c, double t1) { return c.status != 0 || !(c.t < t1); }

// searchsorted(ptimes, t, 'right') - 1: the PWC segment of t (-1 before the first breakpoint)
__device__ __forceinline__ int seg_of(const V &v, double t) {
  int lo = 0, hi = (int)v.nseg;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (v.ptimes[mid] <= t)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo - 1;
}
// the end time, or the first breakpoint strictly after t when it comes before it
__device__ __forceinline__ double target_of(const V &v, double t) {
  if (v.npwc > 0) {
    const int m = seg_of(v, t) + 1;
    if (m < v.nseg && v.ptimes[m] < v.t1) return v.ptimes[m];
  }
  return v.t1;
}
// step of the attempt described by c: the proposed dt, or exactly the rest of the
// interval when it would end within the snapping tolerance of t1
__device__ __forceinline__ double step_h(const V &v, const Ctrl &c) {
  const double tg = target_of(v, c.t);
  return snaps_to(c.t, c.dt, tg) ? tg - c.t : c.dt;
}
__device__ __forceinline__ double step_end(const V &v, const Ctrl &c) {
  const double tg = target_of(v, c.t);
  return snaps_to(c.t, c.dt, tg) ? tg : c.t + c.dt;
}
// the attempt ends on a breakpoint before t1
__device__ __forceinline__ bool ends_on_jump(const V &v, const Ctrl &c) {
  const double tg = target_of(v, c.t);
  return tg < v.t1 && snaps_to(c.t, c.dt, tg);
}

__device__ __forceinline__ float2 *kslot(const V &v, int j, int64_t rot, size_t inst) {
  const size_t nn = (size_t)v.n * v.n;
  return v.k + ((size_t)((j + (int)(rot & 7)) % 7) * v.ninst + inst) * nn;
}
__device__ __forceinline__ float2 *ysbuf(const V &v, int which, size_t inst) {
  const size_t nn = (size_t)v.n * v.n;
  return v.ys + ((size_t)which * v.ninst + inst) * nn;
}
// the FP64 state (other = 0) or the buffer of the candidate (other = 1)
__device__ __forceinline__ double2 *ybuf(const V &v, int64_t rot, int other, size_t inst) {
  const size_t nn = (size_t)v.n * v.n;
  return (((rot & kSel) != 0) != (other != 0) ? v.y2 : v.y) + inst * nn;
}
__device__ __forceinline__ double *partial(const V &v, size_t inst, int which) {
  return v.part + (inst * 2 + which) * v.npart;
}

// FP64 sum over a workgroup of 256; every thread returns the same value.
__device__ __forceinline__ double block_sum(double x, double *sh) {
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = x;
  __syncthreads();
  return (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// Sum of m partials of an instance, the same order in every workgroup.
__device__ __forceinline__ double reduce_partials(const double *p, int64_t m, double *sh) {
  double s = 0.0;
  for (int64_t b = threadIdx.x; b < m; b += 256) s += p[b];
  return block_sum(s, sh);
}

__device__ __forceinline__ double sq(double2 v) { return v.x * v.x + v.y * v.y; }
__device__ __forceinline__ double2 add(double2 a, double w, float2 x) {
  return make_double2(a.x + w * (double)x.x, a.y + w * (double)x.y);
}
__device__ __forceinline__ float2 f32(double2 a) { return make_float2((float)a.x, (float)a.y); }

// stencil inputs: an FP32 matrix, an FP64 one, or y + s k
struct InF {
  const float2 *b;
  __device__ __forceinline__ float2 operator()(size_t e) const { return b[e]; }
};
struct InY {
  const double2 *y;
  __device__ __forceinline__ float2 operator()(size_t e) const { return f32(y[e]); }
};
struct InYK {
  const double2 *y;
  const float2 *k;
  double s;
  __device__ __forceinline__ float2 operator()(size_t e) const { return f32(add(y[e], s, k[e])); }
};

typedef const __attribute__((address_space(4))) Term CTerm;
typedef int Int8 __attribute__((ext_vector_type(8)));

// A control block that no workgroup of the launch writes, through the scalar cache
__device__ __forceinline__ Ctrl read_ctrl(const Ctrl *p) {
  const __attribute__((address_space(4))) Ctrl *c = (const __attribute__((address_space(4))) Ctrl *)p;
  return Ctrl{c->t, c->dt, c->nsteps, c->nacc, c->nrej, c->status, c->isave, c->rot};
}

typedef const __attribute__((address_space(4))) float CFloat;
typedef const __attribute__((address_space(1))) float GFloat;

// f(X) at rows i0 .. i0 + NE - 1 of column j (columns past the matrix read column
// n_true - 1 and are dropped by the caller). The row factors are alike in a wave,
// out-of-range neighbours have a zero factor.
// Order of rounding: every product of complex numbers is rounded before it is added, and
// X conj(c) is summed over a jump operator's column offsets before the row factor. The error
// estimate of the first steps lies in the FP32 noise of f, so the step sequence follows the
// rounding, and the components at the stability limit follow the steps: with the products
// chained into the sum by fused multiply-adds the states of n = 1024 differed from those of
// the full-matrix form by up to 2.5e-2 of their rms (12 batches of four), now by up to 3.7e-3
// (40 batches; the full-matrix form sums the lower triangle in another order).
// The loads of a chunk are in flight together: with one row per thread those of up to 4
// offsets of the generator and 4 terms (n = 323: a solve 1.2 ms, 1.4 with terms of one kind
// in chunks of 8 that share code), with four rows about 16 of the matrix. One row per thread
// reads its row factors like the column's, because a scalar load is waited for in its block.
template <int NE, bool TD, class In>
__device__ __forceinline__ void stencil(const V &v, size_t inst, const In &X, int i0, int j, float2 (&f)[NE]) {
  const int n = (int)v.n, lim = (int)v.n_true, np = v.npair, nt = v.nterm;
  const float2 *D = TD ? v.hcur + inst * (size_t)v.noff0 * v.n : v.H0;
  float2 z[NE];
#pragma unroll
  for (int m = 0; m < NE; ++m) f[m] = z[m] = make_float2(0.f, 0.f);
  auto clamp = [&](int a) { return min(max(a, 0), lim - 1); };
  auto outside = [&](int a) { return (unsigned)a >= (unsigned)lim; };
  auto column = [&](const float2 *d, int qc) {
    GFloat *cp = (GFloat *)d;
    return make_float2(cp[2 * qc], cp[2 * qc + 1]);
  };
  auto rows = [&](const float2 *d, int p, float2 (&r)[NE]) {
    CFloat *rp = (CFloat *)d;
#pragma unroll
    for (int m = 0; m < NE; ++m) {
      int a = clamp(i0 + m + p);
      if constexpr (NE == 1) {
        asm volatile("" : "+v"(a));
        r[m] = column(d, a);
      } else {
        r[m] = make_float2(rp[2 * a], rp[2 * a + 1]);
      }
    }
  };
  // an offset p of the generator: G[i][i + p] X[i + p][j], then X[i][j + p] conj(G[j][j + p])
  struct Pair {
    int p;
    float2 c, r[NE], x[NE], w[NE];
  };
  auto load_pair = [&](Pair &o, int u, int p) {
    const float2 *d = D + (size_t)u * n;
    o.p = p;
    const int qc = clamp(j + o.p);
    o.c = column(d, qc);
    rows(d, o.p, o.r);
#pragma unroll
    for (int m = 0; m < NE; ++m) {
      o.x[m] = X((size_t)clamp(i0 + m + o.p) * n + j);
      o.w[m] = X((size_t)min(i0 + m, lim - 1) * n + qc);
    }
  };
  auto add_pair = [&](Pair &o) {
    if (outside(j + o.p)) o.c = make_float2(0.f, 0.f);
#pragma unroll
    for (int m = 0; m < NE; ++m) {
      if (outside(i0 + m + o.p)) o.r[m] = make_float2(0.f, 0.f);
      f[m].x += fmaf(o.r[m].x, o.x[m].x, -(o.r[m].y * o.x[m].y));
      f[m].y += fmaf(o.r[m].x, o.x[m].y, o.r[m].y * o.x[m].x);
      f[m].x += fmaf(o.w[m].x, o.c.x, o.w[m].y * o.c.y);
      f[m].y += fmaf(o.w[m].y, o.c.x, -(o.w[m].x * o.c.y));
    }
  };
  struct Jump {
    int p, q;
    float go;
    float2 c, r[NE], x[NE];
  };
  auto load_jump = [&](Jump &o, const auto &t) {
    o.p = t.p;
    o.q = t.q;
    o.go = t.go;
    const int qc = clamp(j + o.q);
    o.c = column(t.c, qc);
    rows(t.r, o.p, o.r);
#pragma unroll
    for (int m = 0; m < NE; ++m) o.x[m] = X((size_t)clamp(i0 + m + o.p) * n + qc);
  };
  auto add_jump = [&](Jump &o) {
    if (outside(j + o.q)) o.c = make_float2(0.f, 0.f);
#pragma unroll
    for (int m = 0; m < NE; ++m) {
      if (outside(i0 + m + o.p)) o.r[m] = make_float2(0.f, 0.f);
      z[m].x = fmaf(z[m].x, o.go, fmaf(o.x[m].x, o.c.x, o.x[m].y * o.c.y));
      z[m].y = fmaf(z[m].y, o.go, fmaf(o.x[m].y, o.c.x, -(o.x[m].x * o.c.y)));
      f[m].x += fmaf(o.r[m].x, z[m].x, -(o.r[m].y * z[m].y));
      f[m].y += fmaf(o.r[m].y, z[m].x, o.r[m].x * z[m].y);
    }
  };
  // offsets in chunks of PF, the last PL or fewer together with the first SL terms, the
  // other terms in chunks of SF
  constexpr int PF = NE > 1 ? 2 : 4, PL = NE > 1 ? 1 : 4, SL = NE > 1 ? 2 : kHead, SF = 4;
  int u = 0;
  for (; np - u > PL; u += PF) {
    Pair o[PF];
#pragma unroll
    for (int x = 0; x < PF; ++x) load_pair(o[x], u + x, v.off[u + x]);
#pragma unroll
    for (int x = 0; x < PF; ++x) add_pair(o[x]);
  }
  {
    Pair o[PL];
    Jump s[SL];
    int off[PL];
    Int8 head[SL];
#pragma unroll
    for (int x = 0; x < PL; ++x) off[x] = v.off[min(u + x, DQH_DIA_MAXOFF - 1)];
#pragma unroll
    for (int x = 0; x < SL; ++x) __builtin_memcpy(&head[x], &v.head[x], sizeof(Term));
    // these arrive together: in the blocks below each would be waited for by itself
#pragma unroll
    for (int x = 0; x < PL; ++x) asm volatile("" : "+s"(off[x]));
#pragma unroll
    for (int x = 0; x < SL; ++x) asm volatile("" : "+s"(head[x]));
#pragma unroll
    for (int x = 0; x < PL; ++x)
      if (u + x < np) load_pair(o[x], u + x, off[x]);
#pragma unroll
    for (int x = 0; x < SL; ++x) {
      Term t;
      __builtin_memcpy(&t, &head[x], sizeof(Term));
      if (x < nt) load_jump(s[x], t);
    }
#pragma unroll
    for (int x = 0; x < PL; ++x)
      if (u + x < np) add_pair(o[x]);
#pragma unroll
    for (int x = 0; x < SL; ++x)
      if (x < nt) add_jump(s[x]);
  }
  CTerm *terms = (CTerm *)v.terms;
  int t = SL;
  for (; t + SF <= nt; t += SF) {
    Jump s[SF];
#pragma unroll
    for (int x = 0; x < SF; ++x) load_jump(s[x], terms[t + x]);
#pragma unroll
    for (int x = 0; x < SF; ++x) add_jump(s[x]);
  }
  for (; t < nt; ++t) {
    Jump s;
    load_jump(s, terms[t]);
    add_jump(s);
  }
  if (v.herm) {
#pragma unroll
    for (int m = 0; m < NE; ++m)
      if (i0 + m == j) f[m].y = 0.f;
  }
}

// ------------------------------------------------------------------ one step
// The outcome of the attempt of control block c, whose error partials sum to esum (norm
// squared times n^2): accept or reject and the next dt, as the next attempt's block.
__device__ __forceinline__ Ctrl outcome(const V &v, const Ctrl &c, double esum) {
  const double h = step_h(v, c);
  const double norm = sqrt(esum * v.inv_nn);
  const bool finite = isfinite(norm);
  const bool keep = finite && norm < 1.0;
  double factor;
  if (!finite)
    factor = v.fmin_;
  else if (norm == 0.0)
    factor = v.fmax_;
  else
    factor = v.safety * pow(norm, -0.2);
  factor = fmin(fmax(factor, keep ? 1.0 : v.fmin_), v.fmax_);
  Ctrl o = c;
  o.nsteps += 1;
  if (keep) {
    o.nacc += 1;
    o.t = step_end(v, c);
    // FSAL: k_6 of this step is k_0 of the next; the candidate becomes the state
    o.rot = (((c.rot & 7) + 6) % 7) | (ends_on_jump(v, c) ? kJump : 0) | ((c.rot & kSel) ^ kSel);
    while (o.isave < v.nsave && v.tsave[o.isave] <= o.t) ++o.isave;
  } else {
    o.nrej += 1;
    o.rot = c.rot & ~kJump;
  }
  o.dt = factor * h;
  if (o.t < v.t1) {
    if (o.nsteps >= v.max_steps) {
      o.status = DQH_MAX_STEPS;
    } else {
      const double hn = step_h(v, o);
      if (!(hn > 0.0) || !(hn > 1e-14 * fmax(1.0, fabs(o.t)))) o.status = DQH_NONFINITE;
    }
  }
  return o;
}

__device__ __forceinline__ Ctrl next_ctrl(const V &v, const Ctrl &c, size_t inst, double *sh) {
  if (is_done(c, v.t1) || (c.rot & kFresh)) {
    Ctrl o = c;
    o.rot &= ~kFresh;
    return o;
  }
  return outcome(v, c, reduce_partials(partial(v, inst, 0), v.total, sh));
}

// The control block of the next attempt (block cur, from block 1 - cur), formed by every
// workgroup of the instance alike and stored by workgroup 0, or read where k_ctl has
// formed it; and the saves of the step that block 1 - cur describes.
template <int NE, bool TD>
__device__ __forceinline__ Ctrl commit(const V &v, int cur, size_t inst, int id, int i0, int j, double *sh) {
  const RKTab &rk = rk_tab(v.flags);
  const Ctrl c = read_ctrl(v.ctrl + (size_t)(1 - cur) * v.ninst + inst);
  Ctrl *nx = v.ctrl + (size_t)cur * v.ninst + inst;
  Ctrl o;
  if (v.presum) {
    o = read_ctrl(nx);
  } else {
    o = next_ctrl(v, c, inst, sh);
    if (id == 0 && threadIdx.x == 0) *nx = o;
  }
  const int64_t is_end = o.isave;
  const double h = step_h(v, c);
  if (is_end > c.isave) {
    const int64_t ntn = v.n_true * v.n_true;
    const double2 *y = ybuf(v, c.rot, 0, inst);
#pragma unroll
    for (int m = 0; m < NE; ++m) {
      const int i = i0 + m;
      if (!owned(v, i, j)) continue;
      const size_t e = (size_t)i * v.n + j;
      float2 kk[7];
#pragma unroll
      for (int q = 0; q < 7; ++q) kk[q] = kslot(v, q, c.rot, inst)[e];
      const double2 yv = y[e];
      for (int64_t is = c.isave; is < is_end; ++is) {
        const double th = (v.tsave[is] - c.t) / h;
        double w[7];
#pragma unroll
        for (int q = 0; q < 7; ++q)
          w[q] = th * (rk.R[q][0] + th * (rk.R[q][1] + th * (rk.R[q][2] + th * rk.R[q][3])));
        double2 s = yv;
#pragma unroll
        for (int q = 0; q < 7; ++q) s = add(s, h * w[q], kk[q]);
        float2 *st = v.states + (inst * v.nsave + is) * ntn;
        float2 x = f32(s);
        st[(size_t)i * v.n_true + j] = x;
        if (v.herm && i != j) {
          x.y = -x.y;
          st[(size_t)j * v.n_true + i] = x;
        }
      }
    }
  }
  return o;
}

// Stage S: k_S and the input of stage S + 1, or the error partials (S = 6). S = 0 (TD only):
// k_0 = f(y) after a step that ended on a breakpoint.
template <int S, int NE, bool TD>
__global__ __launch_bounds__(256) void k_stage(V v, int cur) {
  const RKTab &rk = rk_tab(v.flags);
  __shared__ double sh[4];
  const size_t inst = blockIdx.y;
  int id, i0, j;
  if (!tile<NE>(v, id, i0, j)) return;
  Ctrl c;
  if constexpr (S == 1 && !TD)
    c = commit<NE, TD>(v, cur, inst, id, i0, j, sh);
  else
    c = read_ctrl(v.ctrl + (size_t)cur * v.ninst + inst);
  if (is_done(c, v.t1)) return;
  if (S == 0 && !(c.rot & kJump)) return;
  const double h = step_h(v, c);
  double acc = 0.0;
  // a wave without elements (past the matrix, below the diagonal) only joins the sum
  const int jw = j - ((int)threadIdx.x & 63);
  if (i0 >= 0 && i0 < (int)v.n_true && jw < (int)v.n_true && (!v.herm || jw + 63 >= i0)) {
    const int jc = min(j, (int)v.n_true - 1);
    // this element's own operands: in flight while the stencil runs, except for the many
    // of stages 5 and 6 with several rows, whose registers would halve the waves per SIMD
    constexpr int NK = S == 6 ? 6 : S;
    constexpr bool kAfter = NE > 1 && S >= 5;
    float2 kq[NK > 0 ? NK : 1][NE];
    double2 yv[NE], y1[NE];
    auto own = [&]() {
#pragma unroll
      for (int m = 0; m < NE; ++m) {
        const size_t e = (size_t)min(i0 + m, (int)v.n_true - 1) * v.n + jc;
#pragma unroll
        for (int q = 0; q < NK; ++q) kq[q][m] = kslot(v, q, c.rot, inst)[e];
        if (S >= 1) yv[m] = ybuf(v, c.rot, 0, inst)[e];
        if (S == 6) y1[m] = ybuf(v, c.rot, 1, inst)[e];
      }
    };
    if (!kAfter) own();
    float2 f[NE];
    if constexpr (S == 0)
      stencil<NE, TD>(v, inst, InY{ybuf(v, c.rot, 0, inst)}, i0, jc, f);
    else if constexpr (S == 6)
      stencil<NE, TD>(v, inst, InY{ybuf(v, c.rot, 1, inst)}, i0, jc, f);
    else if constexpr (S == 1)
      stencil<NE, TD>(v, inst, InYK{ybuf(v, c.rot, 0, inst), kslot(v, 0, c.rot, inst), h * rk.A[1][0]}, i0, jc, f);
    else
      stencil<NE, TD>(v, inst, InF{ysbuf(v, S & 1, inst)}, i0, jc, f);
    if (kAfter) {
      // the loads stay behind the stencil
      asm volatile("" ::: "memory");
      own();
    }
#pragma unroll
    for (int m = 0; m < NE; ++m) {
      const int i = i0 + m;
      if (!owned(v, i, j)) continue;
      const size_t e = (size_t)i * v.n + j;
      float2 *ks = kslot(v, S, c.rot, inst);
      if constexpr (S == 0 || S == 6)
        put(v, ks, i, j, f[m]);
      else
        ks[e] = f[m];
      if constexpr (S >= 1 && S <= 5) {
        double2 d = yv[m];
        if (S < 5) d = add(d, h * rk.A[S + 1][S], f[m]);
#pragma unroll
        for (int q = 0; q < S; ++q) d = add(d, h * rk.A[S + 1][q], kq[q][m]);
        if (S == 5) d = add(d, h * rk.A[S + 1][S], f[m]);  // the candidate
        if constexpr (S == 5)
          put(v, ybuf(v, c.rot, 1, inst), i, j, d);
        else
          put(v, ysbuf(v, (S + 1) & 1, inst), i, j, f32(d));
      }
      if constexpr (S == 6) {
        double2 er = make_double2(0.0, 0.0);
#pragma unroll
        for (int q = 0; q < 6; ++q) er = add(er, rk.E[q], kq[q][m]);
        er = add(er, rk.E[6], f[m]);
        er.x *= h;
        er.y *= h;
        const double sc = v.atol + v.rtol * sqrt(fmax(sq(yv[m]), sq(y1[m])));
        acc += (v.herm && i != j ? 2.0 : 1.0) * sq(er) / (sc * sc);
      }
    }
  }
  if constexpr (S == 6) {
    const double tot = block_sum(acc, sh);
    if (threadIdx.x == 0) partial(v, inst, 0)[id] = tot;
  }
}

// the controller alone (time-dependent generators: the diagonals are rebuilt between it
// and the first stage)
template <int NE>
__global__ __launch_bounds__(256) void k_commit(V v, int cur) {
  __shared__ double sh[4];
  int id, i0, j;
  if (!tile<NE>(v, id, i0, j)) return;
  (void)commit<NE, true>(v, cur, blockIdx.y, id, i0, j, sh);
}

// the control blocks alone, for grids in which every workgroup forming them costs more
// than one more launch
__global__ __launch_bounds__(256) void k_ctl(V v, int cur) {
  __shared__ double sh[4];
  const size_t inst = blockIdx.x;
  const Ctrl o = next_ctrl(v, v.ctrl[(size_t)(1 - cur) * v.ninst + inst], inst, sh);
  if (threadIdx.x == 0) v.ctrl[(size_t)cur * v.ninst + inst] = o;
}

// number of instances that are done, after an even number of steps (parity 0)
__global__ __launch_bounds__(256) void k_count(V v) {
  __shared__ double sh[4];
  double cnt = 0.0;
  for (int64_t b = threadIdx.x; b < v.ninst; b += 256) cnt += is_done(v.ctrl[v.ninst + b], v.t1) ? 1.0 : 0.0;
  const double tot = block_sum(cnt, sh);
  if (threadIdx.x == 0) *v.flag = (int64_t)(tot + 0.5);
}

// ------------------------------------------------------------- initial step
// The jump operators' terms, the first `most` of them written to list; returns how many there are.
__host__ __device__ inline int list_terms(const dqh_dia_ops &ops, int64_t n, const float2 *zeros, Term *list, int most) {
  int m = 0;
  for (int s = 1; s < ops.nops; ++s) {
    const float2 *A = (const float2 *)ops.diags[s];
    for (int u = 0; u < ops.noff[s]; ++u)
      for (int w = 0; w < ops.noff[s]; ++w, ++m)
        if (m < most)
          list[m] = Term{w + 1 < ops.noff[s] ? zeros : A + (size_t)u * n, A + (size_t)w * n, ops.off[s][u], ops.off[s][w],
                         w > 0 ? 1.f : 0.f, 0};
  }
  return m;
}

// The list of terms, the vector of zeros, and the flag that k_init sets.
__global__ __launch_bounds__(256) void k_setup(V v, dqh_dia_ops ops) {
  for (int64_t e = threadIdx.x; e < v.n; e += 256) v.zeros[e] = make_float2(0.f, 0.f);
  if (threadIdx.x != 0) return;
  *v.flag = 0;
  list_terms(ops, v.n, v.zeros, v.terms, kMaxTerm);
}

// Control block and the saves at tsave <= t0; sets the flag where rho0 is not Hermitian.
__global__ __launch_bounds__(256) void k_init(V v) {
  const size_t inst = blockIdx.y;
  int64_t is0 = 0;
  while (is0 < v.nsave && v.tsave[is0] <= v.t0) ++is0;
  const int64_t n = v.n;
  const size_t nn = (size_t)n * n;
  int i, j;
  if (diat::row_elem(n, i, j) && i < v.n_true && j < v.n_true) {
    const double2 *y = v.y + inst * nn;
    const double2 yv = y[(int64_t)i * n + j];
    const float2 f = f32(yv);
    const int64_t ntn = v.n_true * v.n_true;
    for (int64_t is = 0; is < is0; ++is) v.states[(inst * v.nsave + is) * ntn + (size_t)i * v.n_true + j] = f;
    if (j >= i) {
      if (!hermitian_at(y, n, i, j)) *v.flag = 1;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    Ctrl c;
    c.t = v.t0;
    c.dt = 0.0;
    c.nsteps = c.nacc = c.nrej = 0;
    c.status = v.max_steps <= 0 && v.t0 < v.t1 ? DQH_MAX_STEPS : 0;
    c.isave = is0;
    c.rot = 0;
    v.ctrl[inst] = c;
    v.ctrl[v.ninst + inst] = c;
  }
}

// pass 0: k_0 = f(y0), partials |y0|^2 / sc^2 and |k_0|^2 / sc^2;
// pass 1: partials |f(y0 + h0 k_0) - k_0|^2 / sc^2 (sc = atol + rtol |y0|), h0 in control
// block 1.
// Hairer-Norsett-Wanner II.4 starting step as the dense kernel computes it.
template <int NE, bool TD>
__global__ __launch_bounds__(256) void k_init_rhs(V v, int pass) {
  __shared__ double sh[4];
  const size_t inst = blockIdx.y;
  int id, i0, j;
  if (!tile<NE>(v, id, i0, j)) return;
  if (is_done(v.ctrl[inst], v.t1)) return;
  const double2 *y = ybuf(v, 0, 0, inst);
  float2 *k0 = kslot(v, 0, 0, inst);
  double a0 = 0.0, a1 = 0.0;
  if (i0 >= 0 && i0 < (int)v.n_true) {
    const int jc = min(j, (int)v.n_true - 1);
    const double h0 = pass == 0 ? 0.0 : v.ctrl[v.ninst + inst].dt;
    float2 f[NE];
    if (pass == 0)
      stencil<NE, TD>(v, inst, InY{y}, i0, jc, f);
    else
      stencil<NE, TD>(v, inst, InYK{y, k0, h0}, i0, jc, f);
#pragma unroll
    for (int m = 0; m < NE; ++m) {
      const int i = i0 + m;
      if (!owned(v, i, j)) continue;
      const size_t e = (size_t)i * v.n + j;
      const double2 yv = y[e];
      const double sc = v.atol + v.rtol * sqrt(sq(yv)), w = v.herm && i != j ? 2.0 : 1.0;
      if (pass == 0) {
        put(v, k0, i, j, f[m]);
        a0 += w * sq(yv) / (sc * sc);
        a1 += w * sq(make_double2(f[m].x, f[m].y)) / (sc * sc);
      } else {
        const float2 kq = k0[e];
        a0 += w * sq(make_double2((double)f[m].x - kq.x, (double)f[m].y - kq.y)) / (sc * sc);
      }
    }
  }
  const double t0s = block_sum(a0, sh);
  const double t1s = block_sum(a1, sh);
  if (threadIdx.x == 0) {
    partial(v, inst, 0)[id] = t0s;
    if (pass == 0) partial(v, inst, 1)[id] = t1s;
  }
}

// h0 from d0, d1, parked in control block 1; d1 moves to slot 0 of its partials
__global__ __launch_bounds__(256) void k_init_h0(V v) {
  __shared__ double sh[4];
  const size_t inst = blockIdx.x;
  const Ctrl c = v.ctrl[inst];
  if (is_done(c, v.t1)) return;
  const double d0 = sqrt(reduce_partials(partial(v, inst, 0), v.total, sh) * v.inv_nn);
  const double d1 = sqrt(reduce_partials(partial(v, inst, 1), v.total, sh) * v.inv_nn);
  if (threadIdx.x == 0) {
    partial(v, inst, 1)[0] = d1;
    Ctrl o = c;
    o.dt = (d0 < 1e-5 || d1 < 1e-5) ? 1e-6 : 0.01 * d0 / d1;
    v.ctrl[v.ninst + inst] = o;
  }
}

// dt0 = min(100 h0, (0.01 / max(d1, d2))^kInitExp): control block 1, which the first step reads
__global__ __launch_bounds__(256) void k_init_dt(V v) {
  __shared__ double sh[4];
  const size_t inst = blockIdx.x;
  const Ctrl c = v.ctrl[v.ninst + inst];
  if (is_done(c, v.t1)) return;
  const double h0 = c.dt;
  const double d1 = partial(v, inst, 1)[0];
  const double d2 = sqrt(reduce_partials(partial(v, inst, 0), v.total, sh) * v.inv_nn) / h0;
  const double md = fmax(d1, d2);
  const double h1 = md <= 1e-15 ? fmax(1e-6, h0 * 1e-3) : pow(0.01 / md, kInitExp);
  Ctrl o = c;
  o.dt = fmin(100.0 * h0, h1);
  o.rot |= kFresh;
  const double hn = step_h(v, o);
  if (!(hn > 0.0) || !(hn > 1e-14 * fmax(1.0, fabs(o.t)))) o.status = DQH_NONFINITE;
  if (threadIdx.x == 0) v.ctrl[v.ninst + inst] = o;
}

// f_j(tau) of modulated table j (Horner on the interval that contains tau)
__device__ __forceinline__ double2 mod_at(const V &v, int j, double tau) {
  int64_t i = (int64_t)floor((tau - v.mod_t0) / v.mod_dt);
  i = i < 0 ? 0 : (i >= v.mod_nint ? v.mod_nint - 1 : i);
  const double x = tau - (v.mod_t0 + (double)i * v.mod_dt);
  const double2 *q = v.mcoef + ((size_t)j * v.mod_nint + i) * 4;
  double re = q[0].x, im = q[0].y;
#pragma unroll
  for (int m = 1; m < 4; ++m) {
    re = re * x + q[m].x;
    im = im * x + q[m].y;
  }
  return make_double2(re, im);
}

// hcur <- diagonals of Hnh(tau) = H0 + sum_j c_j Hterms_j per instance, PWC values
// on the segment of the step start. mode 0..6: stage mode of the attempt in control
// block cur (0: the k_0 refresh after a breakpoint, only then); 7: t0 (k_0 of the
// initial step); 8: t0 + h0 (the initial step's probe, h0 parked in block 1).
// grid (ceil(noff0 n / 256), ninst)
__global__ __launch_bounds__(256) void k_hupd(V v, int cur, int mode) {
  const RKTab &rk = rk_tab(v.flags);
  const size_t inst = blockIdx.y;
  double tseg, tau;
  if (mode <= 6) {
    const Ctrl c = v.ctrl[(size_t)cur * v.ninst + inst];
    if (is_done(c, v.t1) || (mode == 0 && !(c.rot & kJump))) return;
    tseg = c.t;
    tau = c.t + rk.C[mode] * step_h(v, c);
  } else {
    const Ctrl c = v.ctrl[(mode == 7 ? 0 : v.ninst) + inst];
    if (is_done(c, v.t1)) return;
    tseg = c.t;
    tau = mode == 7 ? c.t : c.t + c.dt;
  }
  const size_t m = (size_t)v.noff0 * v.n;
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= m) return;
  const int nv = (int)v.nseg - 1;
  const int seg = v.npwc > 0 ? seg_of(v, tseg) : -1;
  const float2 h0 = v.H0[e];
  double re = h0.x, im = h0.y;
  if (seg >= 0 && seg < nv)
    for (int j = 0; j < (int)v.npwc; ++j) {
      const double cr = v.pvals[2 * ((size_t)j * nv + seg)], ci = v.pvals[2 * ((size_t)j * nv + seg) + 1];
      const float2 o = v.Hterms[(size_t)j * m + e];
      re += cr * o.x - ci * o.y;
      im += cr * o.y + ci * o.x;
    }
  for (int j = 0; j < (int)v.nmod; ++j) {
    const double2 f = mod_at(v, j, tau);
    const float2 o = v.Hterms[(size_t)(v.npwc + j) * m + e];
    re += f.x * o.x - f.y * o.y;
    im += f.x * o.y + f.y * o.x;
  }
  v.hcur[inst * m + e] = make_float2((float)re, (float)im);
}

// saves not reached (an instance that stopped early keeps its last state), the final state
// on both triangles in v.y, and stats
__global__ __launch_bounds__(256) void k_finish(V v) {
  const size_t inst = blockIdx.y;
  const Ctrl c = v.ctrl[v.ninst + inst];
  const int64_t n = v.n;
  const size_t nn = (size_t)n * n;
  int i, j;
  if (diat::row_elem(n, i, j) && owned(v, i, j)) {
    const int64_t ntn = v.n_true * v.n_true;
    const size_t e = (size_t)i * n + j, em = (size_t)j * n + i;
    const bool mirror = v.herm && i != j;
    double2 *y = v.y + inst * nn;
    const double2 yv = ybuf(v, c.rot, 0, inst)[e], yc = make_double2(yv.x, -yv.y);
    if (c.rot & kSel) y[e] = yv;
    if (mirror) y[em] = yc;
    for (int64_t is = c.isave; is < v.nsave; ++is) {
      float2 *st = v.states + (inst * v.nsave + is) * ntn;
      st[(size_t)i * v.n_true + j] = f32(yv);
      if (mirror) st[(size_t)j * v.n_true + i] = f32(yc);
    }
  }
  if (blockIdx.x == 0 && threadIdx.x < 8) {
    int64_t *st = v.stats + inst * 8;
    const int64_t vals[8] = {c.nsteps, c.nacc, c.nrej, c.status, 2 + 6 * c.nsteps, 0, 0, 0};
    st[threadIdx.x] = vals[threadIdx.x];
  }
}

struct Layout {
  size_t k, ys, y2, terms, zeros, part, ctrl, flag, total;
  int64_t npart;
};

inline size_t align256(size_t x) { return (x + 255) / 256 * 256; }

inline Layout layout(int64_t n, int64_t ninst) {
  const size_t nn = (size_t)n * n;
  const int nb = (int)((n + 63) / 64);
  Layout L;
  L.npart = std::max(tiles_of(nb, false, 1), tiles_of(nb, true, 1));  // tiles of the smallest kind
  L.k = 0;
  L.ys = L.k + align256(7 * (size_t)ninst * nn * sizeof(float2));
  L.y2 = L.ys + align256(2 * (size_t)ninst * nn * sizeof(float2));
  L.terms = L.y2 + align256((size_t)ninst * nn * sizeof(double2));
  L.zeros = L.terms + align256(kMaxTerm * sizeof(Term));
  L.part = L.zeros + align256((size_t)n * sizeof(float2));
  L.ctrl = L.part + align256((size_t)ninst * 2 * L.npart * sizeof(double));
  L.flag = L.ctrl + align256(2 * (size_t)ninst * sizeof(Ctrl));
  L.total = L.flag + 256;
  return L;
}

}  // namespace diats
}  // namespace dqh

using namespace dqh;

extern "C" int64_t dqh_sizeof_dia_tsit5(void) { return (int64_t)sizeof(dqh_dia_tsit5); }

extern "C" int64_t dqh_dia_tsit5_work_bytes(int64_t n, int64_t ninst) {
  if (n <= 0 || ninst <= 0) return -1;
  return (int64_t)diats::layout(n, ninst).total;
}

namespace {

// grid of k_hupd: the noff0 x n diagonal elements per instance
inline dim3 hupd_grid(const diats::V &v) {
  return dim3((unsigned)(((size_t)v.noff0 * v.n + 255) / 256), (unsigned)v.ninst);
}
inline dim3 tile_grid(const diats::V &v) { return dim3((unsigned)((v.total + 7) / 8 * 8), (unsigned)v.ninst); }

template <int S, int NE, bool TD>
void launch_stages(const diats::V &v, int cur, hipStream_t s) {
  if (TD) hipLaunchKernelGGL(diats::k_hupd, hupd_grid(v), dim3(256), 0, s, v, cur, S);
  hipLaunchKernelGGL((diats::k_stage<S, NE, TD>), tile_grid(v), dim3(256), 0, s, v, cur);
  if constexpr (S > 0 && S < 6) launch_stages<S + 1, NE, TD>(v, cur, s);
}

template <int NE, bool TD>
void launch_step(const diats::V &v, int cur, hipStream_t s) {
  if (v.presum) hipLaunchKernelGGL(diats::k_ctl, dim3((unsigned)v.ninst), dim3(256), 0, s, v, cur);
  if constexpr (TD) {
    hipLaunchKernelGGL(diats::k_commit<NE>, tile_grid(v), dim3(256), 0, s, v, cur);
    // k_0 anew after a breakpoint (instances that did not land on one return at once)
    if (v.npwc > 0) launch_stages<0, NE, TD>(v, cur, s);
  }
  launch_stages<1, NE, TD>(v, cur, s);
}

struct Steps {  // the captured steps and what captured them
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  hipStream_t cs = nullptr;
  ~Steps() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    if (cs) (void)hipStreamDestroy(cs);
  }
  // G steps + the completion count
  template <int NE, bool TD>
  hipError_t capture(const diats::V &v, int64_t G) {
    hipError_t err = hipStreamCreateWithFlags(&cs, hipStreamNonBlocking);
    if (err == hipSuccess) err = hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal);
    if (err != hipSuccess) return err;
    for (int64_t g = 0; g < G; ++g) launch_step<NE, TD>(v, (int)(g & 1), cs);
    hipLaunchKernelGGL(diats::k_count, dim3(1), dim3(256), 0, cs, v);
    err = hipStreamEndCapture(cs, &graph);
    if (err == hipSuccess) err = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    return err;
  }
};

struct Events {
  hipEvent_t ev[2] = {nullptr, nullptr};
  ~Events() {
    for (int q = 0; q < 2; ++q)
      if (ev[q]) (void)hipEventDestroy(ev[q]);
  }
};

// tiles for a sweep over the upper triangle or the full matrix
template <int NE>
void set_tiles(diats::V &v, bool herm) {
  v.herm = herm;
  v.nb = (int)((v.n_true + 63) / 64);
  v.total = diats::tiles_of(v.nb, herm, NE);
  // Forming the control block delays a workgroup of stage 1 by about 5 us: hidden while
  // they all run at once, less than the launch of k_ctl; paid per round of workgroups in
  // larger grids (four solves of n = 1024: 30 us -> 4 + 27 with
  // the saves).
  v.presum = (int64_t)v.total * v.ninst > 1024;
}

template <int NE, bool TD>
int drive(const dqh_dia_tsit5 &p, diats::V v, hipStream_t st) {
  const dim3 gflat = diat::row_grid(p.n, p.ninst);
  // Steps per replay: at most 4, because the replay in flight when the count shows the end
  // and the rest of the last one are launches without work (n = 323, 29
  // steps: 1.30 ms a solve with 4, 1.40 with 16; four solves of n = 1024: 7.66 and 8.15)
  const int64_t G = p.graph_steps > 0 ? std::min<int64_t>(p.graph_steps, 4) : 2;
  volatile int64_t *hf = reinterpret_cast<volatile int64_t *>(p.host_flags);
  hf[0] = hf[1] = -1;
  Events E;
  hipError_t err = hipSuccess;
  for (int q = 0; q < 2 && err == hipSuccess; ++q) err = hipEventCreateWithFlags(&E.ev[q], hipEventDisableTiming);
  if (err != hipSuccess) return fail(DQH_HIP_ERROR, std::string("dqh_mesolve_tsit5_dia event: ") + hipGetErrorString(err));
  hipLaunchKernelGGL(diats::k_setup, dim3(1), dim3(256), 0, st, v, p.ops);
  hipLaunchKernelGGL(diats::k_init, gflat, dim3(256), 0, st, v);
  err = hipGetLastError();
  if (err == hipSuccess)
    err = hipMemcpyAsync(const_cast<int64_t *>(hf), v.flag, sizeof(int64_t), hipMemcpyDeviceToHost, st);
  if (err == hipSuccess) err = hipEventRecord(E.ev[0], st);
  // the steps are captured while the device looks at rho0: for the upper triangle, and
  // once more for the full matrix where that proves necessary
  set_tiles<NE>(v, true);
  Steps steps, full;
  Steps *use = &steps;
  if (err == hipSuccess && p.graph_steps > 0) err = steps.template capture<NE, TD>(v, G);
  if (err == hipSuccess) err = hipEventSynchronize(E.ev[0]);
  if (err == hipSuccess && hf[0] != 0) {
    set_tiles<NE>(v, false);
    use = &full;
    if (p.graph_steps > 0) err = full.template capture<NE, TD>(v, G);
  }
  if (err != hipSuccess) return fail(DQH_HIP_ERROR, std::string("dqh_mesolve_tsit5_dia graph: ") + hipGetErrorString(err));
  hf[0] = -1;
  const dim3 gt = tile_grid(v), gi((unsigned)v.ninst);
  if (TD) hipLaunchKernelGGL(diats::k_hupd, hupd_grid(v), dim3(256), 0, st, v, 0, 7);
  hipLaunchKernelGGL((diats::k_init_rhs<NE, TD>), gt, dim3(256), 0, st, v, 0);
  hipLaunchKernelGGL(diats::k_init_h0, gi, dim3(256), 0, st, v);
  if (TD) hipLaunchKernelGGL(diats::k_hupd, hupd_grid(v), dim3(256), 0, st, v, 0, 8);
  hipLaunchKernelGGL((diats::k_init_rhs<NE, TD>), gt, dim3(256), 0, st, v, 1);
  hipLaunchKernelGGL(diats::k_init_dt, gi, dim3(256), 0, st, v);
  err = hipGetLastError();
  if (err != hipSuccess) return fail(DQH_HIP_ERROR, std::string("dqh_mesolve_tsit5_dia init: ") + hipGetErrorString(err));
  // every instance stops within max_steps attempts, and the step after the last one
  // commits it, so this many replays always suffice
  const int64_t max_iters = p.max_steps / G + 4;
  bool finished = false;
  for (int64_t it = 0; it < max_iters && err == hipSuccess; ++it) {
    if (use->exec) {
      err = hipGraphLaunch(use->exec, st);
    } else {
      for (int64_t g = 0; g < G; ++g) launch_step<NE, TD>(v, (int)(g & 1), st);
      hipLaunchKernelGGL(diats::k_count, dim3(1), dim3(256), 0, st, v);
      err = hipGetLastError();
    }
    if (err == hipSuccess)
      err = hipMemcpyAsync(const_cast<int64_t *>(hf + (it & 1)), v.flag, sizeof(int64_t), hipMemcpyDeviceToHost, st);
    if (err == hipSuccess) err = hipEventRecord(E.ev[it & 1], st);
    if (err == hipSuccess && it > 0) {
      err = hipEventSynchronize(E.ev[(it - 1) & 1]);
      if (err == hipSuccess && hf[(it - 1) & 1] >= v.ninst) {
        finished = true;
        break;
      }
    }
  }
  if (err == hipSuccess && !finished) {
    // the last replay may have finished the batch
    err = hipStreamSynchronize(st);
    int64_t last = -1;
    if (err == hipSuccess) err = hipMemcpy(&last, v.flag, sizeof(int64_t), hipMemcpyDeviceToHost);
    finished = err == hipSuccess && last >= v.ninst;
  }
  if (err != hipSuccess) return fail(DQH_HIP_ERROR, std::string("dqh_mesolve_tsit5_dia: ") + hipGetErrorString(err));
  hipLaunchKernelGGL(diats::k_finish, gflat, dim3(256), 0, st, v);
  if (p.nE > 0)
    launch_expect(p.n_true, p.nsave, p.ninst, p.nE, p.states, p.EopsT, p.expects, v.k,
                  9 * (size_t)v.n * v.n * v.ninst * sizeof(float2), st);
  err = hipGetLastError();
  if (err != hipSuccess) return fail(DQH_HIP_ERROR, std::string("dqh_mesolve_tsit5_dia: ") + hipGetErrorString(err));
  if (!finished) return fail(DQH_HIP_ERROR, "dqh_mesolve_tsit5_dia: instances still running after max_steps steps");
  return DQH_OK;
}

}  // namespace

extern "C" int dqh_mesolve_tsit5_dia(const dqh_dia_tsit5 *pb, void *stream) {
  if (!pb) return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_dia: null problem");
  const dqh_dia_tsit5 &p = *pb;
  if (p.n <= 0 || p.ninst <= 0 || p.n_true <= 0 || p.n_true > p.n || p.n > (1 << 16) || p.nsave < 1)
    return fail(DQH_BAD_SHAPE, "dqh_mesolve_tsit5_dia: need 0 < n_true <= n <= 65536, ninst >= 1, nsave >= 1");
  if (!p.y || !p.work || !p.tsave || !p.states || !p.stats || !p.host_flags)
    return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_dia: null buffer");
  if (p.nE < 0 || (p.nE > 0 && (!p.EopsT || !p.expects)))
    return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_dia: nE > 0 needs EopsT and expects");
  if (p.graph_steps < 0 || (p.graph_steps & 1))
    return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_dia: graph_steps must be 0 or a positive even number");
  if (!(p.t1 >= p.t0) || !(p.rtol >= 0) || !(p.atol >= 0) || !(p.rtol + p.atol > 0))
    return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_dia: need t1 >= t0 and positive tolerances");
  if (p.ops.nops < 1 || p.ops.nops > DQH_DIA_MAXOPS)
    return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_dia: 1 <= nops <= 8 (Hnh, then the jump operators)");
  for (int k = 0; k < p.ops.nops; ++k) {
    if (p.ops.noff[k] < 1 || p.ops.noff[k] > DQH_DIA_MAXOFF || !p.ops.diags[k])
      return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_dia: bad number of diagonals or null diagonals");
    for (int u = 0; u < p.ops.noff[k]; ++u)
      if (p.ops.off[k][u] <= -p.n || p.ops.off[k][u] >= p.n)
        return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_dia: offset outside (-n, n)");
  }
  if (p.variant == DQH_SWEEP_SPLIT)
    return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_dia: the split sweep applies to the Rouchon1 Kraus map only");
  if (p.npwc < 0 || p.nmod < 0 || p.npwc + p.nmod > 64)
    return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_dia: 0 <= npwc, nmod and npwc + nmod <= 64");
  if (p.npwc + p.nmod > 0 && (!p.Hterms || !p.hcur))
    return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_dia: time-dependent terms need Hterms and hcur");
  if (p.npwc > 0 && (p.nseg < 2 || !p.pwc_times || !p.pwc_vals))
    return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_dia: PWC terms need nseg >= 2 breakpoints and their values");
  if (p.nmod > 0 && (!p.mod_coef || p.mod_nint < 1 || !(p.mod_dt > 0)))
    return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_dia: modulated terms need their tables");
  const int halo = diat::resolve_halo(p.variant, p.n, diat::max_abs_offset(p.ops));
  if (halo < 0)
    return fail(DQH_BAD_ARG, "dqh_mesolve_tsit5_dia: the tiled sweep needs n % 64 == 0 and every |offset| <= its halo");
  const diats::Layout L = diats::layout(p.n, p.ninst);
  char *w = reinterpret_cast<char *>(p.work);
  diats::V v;
  v.n = p.n;
  v.n_true = p.n_true;
  v.ninst = p.ninst;
  v.nsave = p.nsave;
  v.max_steps = p.max_steps;
  v.flags = p.flags;
  v.rtol = p.rtol;
  v.atol = p.atol;
  v.safety = p.safety;
  v.fmin_ = p.factormin;
  v.fmax_ = p.factormax;
  v.t0 = p.t0;
  v.t1 = p.t1;
  v.inv_nn = 1.0 / ((double)p.n_true * (double)p.n_true);
  v.k = reinterpret_cast<float2 *>(w + L.k);
  v.ys = reinterpret_cast<float2 *>(w + L.ys);
  v.y2 = reinterpret_cast<double2 *>(w + L.y2);
  v.terms = reinterpret_cast<diats::Term *>(w + L.terms);
  v.zeros = reinterpret_cast<float2 *>(w + L.zeros);
  v.npart = L.npart;
  v.part = reinterpret_cast<double *>(w + L.part);
  v.ctrl = reinterpret_cast<diats::Ctrl *>(w + L.ctrl);
  v.flag = reinterpret_cast<int64_t *>(w + L.flag);
  v.y = reinterpret_cast<double2 *>(p.y);
  v.tsave = reinterpret_cast<const double *>(p.tsave);
  v.states = reinterpret_cast<float2 *>(p.states);
  v.stats = reinterpret_cast<int64_t *>(p.stats);
  const bool td = p.npwc + p.nmod > 0;
  v.npwc = td ? p.npwc : 0;
  v.nseg = p.npwc > 0 ? p.nseg : 0;
  v.nmod = td ? p.nmod : 0;
  v.noff0 = p.ops.noff[0];
  v.mod_nint = p.mod_nint;
  v.mod_t0 = p.mod_t0;
  v.mod_dt = p.mod_dt;
  v.ptimes = reinterpret_cast<const double *>(p.pwc_times);
  v.pvals = reinterpret_cast<const double *>(p.pwc_vals);
  v.mcoef = reinterpret_cast<const double2 *>(p.mod_coef);
  v.H0 = reinterpret_cast<const float2 *>(p.ops.diags[0]);
  v.Hterms = td ? reinterpret_cast<const float2 *>(p.Hterms) : nullptr;
  v.hcur = td ? reinterpret_cast<float2 *>(p.hcur) : nullptr;
  v.npair = p.ops.noff[0];
  for (int u = 0; u < DQH_DIA_MAXOFF; ++u) v.off[u] = u < v.npair ? p.ops.off[0][u] : 0;
  for (int x = 0; x < diats::kHead; ++x) v.head[x] = diats::Term{};
  v.nterm = diats::list_terms(p.ops, p.n, v.zeros, v.head, diats::kHead);
  v.spread = 0;  // largest p - q of a shift (p, q)
  for (int u = 0; u < p.ops.noff[0]; ++u) v.spread = std::max(v.spread, std::abs(p.ops.off[0][u]));
  for (int k = 1; k < p.ops.nops; ++k)
    for (int u = 0; u < p.ops.noff[k]; ++u)
      for (int w = 0; w < p.ops.noff[k]; ++w) v.spread = std::max(v.spread, p.ops.off[k][u] - p.ops.off[k][w]);
  v.herm = v.nb = v.total = v.presum = 0;
  hipStream_t st = (hipStream_t)stream;
  // four rows per thread share the column factors and keep more loads in flight; the upper
  // triangle of 2^21 elements, 2^20, leaves them four waves per SIMD. Below, one row per
  // thread spreads the work over more CUs.
  const bool large = (double)p.n_true * (double)p.n_true * (double)p.ninst >= (double)(1 << 21);
  if (td) return large ? drive<4, true>(p, v, st) : drive<1, true>(p, v, st);
  return large ? drive<4, false>(p, v, st) : drive<1, false>(p, v, st);
}
