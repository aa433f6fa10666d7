// Resident Jacobi-PCG on sliced ELL (see lfgpu_resident.hip): a workgroup owns
// a run of storage rows (in the locality order, so that what it reads of
// others is a compact neighbourhood), keeps their x, r and q in registers and
// their p in LDS, followed by the p of the outside rows that it reads.  The
// columns are stored once more as places in that LDS array (16 bits).  The
// matrix is streamed every iteration (10 B a slot in FP64, 6 in FP32) unless
// a thread has one to three rows: then their first 40, 16 or 8 slots stay in
// registers and an iteration is the exchange, the team sum and the gathers.
// Time per iteration, sweeps against this, FP64: P1 on 300 x 260 unstructured
// squares 20.8 -> 4.1 us, 600^2 30.3 -> 6.7, 900^2 45 -> 17; P3 on 37 x 29
// 19.6 -> 3.5, 200^2 35.9 -> 10.6, 384^2 84 -> 43 (226 MB of matrix, 28 us of
// it at 8 TB/s); FP32 matrix, P3 384^2: 64 -> 36.
#include <hip/hip_bf16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "lfgpu_reduce.h"
#include "lfgpu_resident.h"
#include "lfgpu_resident_device.h"

using namespace lfgpu;
using namespace lfgpu::res;

namespace {

// One workgroup's share: the `slices` slices listed at slist[first..], which
// lie in the storage rows [r0, r1) (and are all of them where the kernel
// takes no list), LDS places 0.. for their rows and from 64 * slices on for
// the `outside` rows listed at ext[at..].
struct EllPart {
  int32_t r0, r1, slices, first, outside;
  int64_t at;
};
// One problem of a batch.
struct EllJob {
  int32_t index, team;
  uint64_t sums_at;
};

struct EllArgs {
  int32_t n;  // storage rows
  const int32_t *__restrict__ slice_off;
  const uint16_t *__restrict__ lcol;
  const double *__restrict__ val;
  const float *__restrict__ val32;
  const double *__restrict__ rowsum;
  const float *__restrict__ rowsum32;
  const double *__restrict__ dinv;
  const float *__restrict__ dinv32;
  const __hip_bfloat16 *__restrict__ dinv16;
  const int32_t *__restrict__ perm;  // storage row -> row of x, b; -1: none; may be null
  const EllPart *__restrict__ parts;
  const int32_t *__restrict__ slist;
  const int32_t *__restrict__ ext;
  const uint8_t *__restrict__ needed;
  const double *__restrict__ b;
  double *x;
  double *xlo;  // storage order
  word_t *words;  // [2][planes(rpt)][n]
  word_t *part, *total;
  ResidentAbort *abort;
  uint32_t tag0;
  double tol2;
  int maxit;
  double delta2;
  int max_interval;
  ResidentState *st;
  // batches
  const EllJob *__restrict__ jobs;
  const int2 *__restrict__ job_slots;  // slot (= part) -> job, rank in its team
  int nslots;
  int *ticket, *running, *arrived;
};

// the precision modes: FP64; FP32 vectors; FP64 vectors with the FP32 matrix
template <int MODE>
struct Mode;
template <>
struct Mode<LFGPU_PCG_FP64> {
  typedef double VT;
  typedef double MT;
};
template <>
struct Mode<LFGPU_PCG_MIXED> {
  typedef float VT;
  typedef float MT;
};
template <>
struct Mode<LFGPU_PCG_MIXED_MATRIX> {
  typedef double VT;
  typedef float MT;
};

// acc + the sum over a row's slots k.. of w of v_k (p_{c_k} - pi) from LDS; vp
// and cp point at the row's first slot, a row's slots are 64 apart.  Eight
// slots' loads are issued before the first use, and the up to seven last ones'
// of an FP64 matrix (four and then one after the other: P1 on 900 x 900
// unstructured squares takes 21.3 us an iteration instead of 17.1, P3 on
// 200 x 200 11.4 instead of 10.6; with FP32 values 64 P3 problems of 8 to 64
// cells take 26.2 ms that way and 30.3 this way).
template <class MT>
__device__ __forceinline__ double ell_lds_row(const MT *__restrict__ vp,
                                              const uint16_t *__restrict__ cp, int32_t k,
                                              int32_t w, const double *lp, double pi,
                                              double acc) {
  for (; k + 8 <= w; k += 8) {
    MT v[8];
    uint16_t c[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      c[u] = cp[64 * (k + u)];
      v[u] = vp[64 * (k + u)];
    }
    double y[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) y[u] = lp[c[u]];
#pragma unroll
    for (int u = 0; u < 8; ++u) acc = __builtin_fma((double)v[u], y[u] - pi, acc);
  }
  if constexpr (sizeof(MT) < 8) {
    if (k + 4 <= w) {
      MT v[4];
      uint16_t c[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        c[u] = cp[64 * (k + u)];
        v[u] = vp[64 * (k + u)];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) acc = __builtin_fma((double)v[u], lp[c[u]] - pi, acc);
      k += 4;
    }
    for (; k < w; ++k) acc = __builtin_fma((double)vp[64 * k], lp[cp[64 * k]] - pi, acc);
    return acc;
  }
  const int32_t left = __builtin_amdgcn_readfirstlane(w - k);
  if (left > 0) {
    MT v[7];
    uint16_t c[7];
#pragma unroll
    for (int u = 0; u < 7; ++u) {
      c[u] = 0;
      v[u] = (MT)0;
      if (u < left) {
        c[u] = cp[64 * (k + u)];
        v[u] = vp[64 * (k + u)];
      }
    }
#pragma unroll
    for (int u = 0; u < 7; ++u)
      if (u < left) acc = __builtin_fma((double)v[u], lp[c[u]] - pi, acc);
  }
  return acc;
}

// Up to this many rows a thread a part is small: its slices come from a list,
// the first held_slots() slots of every row stay in registers, and the outside
// rows' r, q, D^-1 and p are kept here and updated by their owners'
// operations, so that what travels is q, during the team sum (as GHOST in
// lfgpu_resident.hip).  Above, LDS and registers do not hold that, and the
// exchange of p is a tenth of an iteration.
constexpr int kSmallRows = 3;
constexpr int held_slots(int rpt) {
  return rpt == 1 ? 40 : rpt == 2 ? 16 : rpt <= kSmallRows ? 8 : 0;
}
// words per row and parity: two of p or q, and two of r (small parts)
constexpr int planes(int rpt) { return rpt <= kSmallRows ? 4 : 2; }

// RPT: rows per thread: thread t = 64 wave + lane owns the local rows
// 64 (wave + 8 j) + lane, so a wavefront works on whole slices.  DREG: D^-1
// and row sums in registers (else read every iteration).
template <int MODE, int RPT, bool DREG>
__device__ __forceinline__ bool ell_solve(const EllArgs &a, int32_t slot, int rank, int team,
                                          double *lp, SumLds &sh) {
  typedef typename Mode<MODE>::VT VT;
  typedef typename Mode<MODE>::MT MT;
  constexpr bool kMixed = MODE != LFGPU_PCG_FP64;
  constexpr bool kSmall = RPT <= kSmallRows;
  constexpr int kHeld = held_slots(RPT);
  const int t = threadIdx.x;
  Team tm{rank, team, a.part, a.total, a.abort, a.tag0};
  uint32_t tag = a.tag0;
  if (t == 0) sh.bad = 0;
  const EllPart &part = a.parts[slot];
  const int32_t slices = part.slices, place = 64 * slices, next = part.outside;
  const int32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int32_t s0 = (part.r0 >> 6) + wave;
  // small parts: the outside rows' r, q, D^-1 and storage rows
  VT *const gr = reinterpret_cast<VT *>(lp + place + next), *const gq = gr + next,
     *const gd = gq + next;
  int32_t *const gsrc = reinterpret_cast<int32_t *>(gd + next);
  const int32_t *const ext = a.ext + part.at;
  // the wavefront's slice number j, and its thread's storage row there
  int32_t list[kSmall ? RPT : 1];
  if constexpr (kSmall)
#pragma unroll
    for (int j = 0; j < RPT; ++j)
      list[j] = wave + j * kWaves < slices ? a.slist[part.first + wave + j * kWaves] : 0;
  auto slice = [&](int j) { return kSmall ? list[kSmall ? j : 0] : s0 + j * kWaves; };
  auto row = [&](int j) { return 64 * slice(j) + (t & 63); };

  auto dinv_of = [&](int32_t g) -> VT {
    if constexpr (MODE == LFGPU_PCG_FP64) return a.dinv[g];
    else if constexpr (MODE == LFGPU_PCG_MIXED) return __bfloat162float(a.dinv16[g]);
    else return a.dinv32[g];
  };
  auto rowsum_of = [&](int32_t g) -> double {
    if constexpr (kMixed) return (double)a.rowsum32[g];
    else return a.rowsum[g];
  };
  auto at = [&](int32_t g) { return a.perm ? a.perm[g] : g; };
  // Publishes storage row g's value (VT or, for reliable updates, double) in
  // a plane's words, and hands the outside rows' e = 0.. to fn(e, value),
  // four in flight for each of the threads from `from` on.
  auto publish = [&](int32_t g, auto v, int plane) {
    word_t *w = a.words + ((size_t)(tag & 1u) * planes(RPT) + plane) * a.n + g;
    if constexpr (sizeof(v) == 8) {
      put(w, low_word(v, tag));
      put(w + a.n, high_word(v, tag));
    } else {
      put(w, ((word_t)__float_as_uint(v) << 32) | tag);
    }
  };
  auto fetch = [&](auto like, int plane, int from, auto &&fn) {
    typedef decltype(like) FT;
    constexpr bool kTwo = sizeof(like) == 8;
    if (t < from) return;
    const word_t *w = a.words + ((size_t)(tag & 1u) * planes(RPT) + plane) * a.n;
    const int32_t step = kThreads - from;
    for (int32_t e0 = t - from; e0 < next; e0 += 4 * step) {
      int32_t src[4];
      word_t lo[4], hi[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int32_t e = min(e0 + u * step, next - 1);
        src[u] = kSmall ? gsrc[e] : ext[e];
      }
      bool ok;
      Wait wait(a.abort);
      do {
        ok = true;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          lo[u] = get(&w[src[u]]);
          if constexpr (kTwo) hi[u] = get(&w[a.n + src[u]]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          ok = ok && tagged(lo[u], tag);
          if constexpr (kTwo) ok = ok && tagged(hi[u], tag);
        }
      } while (!ok && wait.more());
      if (!ok) sh.bad = 1;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (e0 + u * step < next) {
          FT v;
          if constexpr (kTwo) v = from_words(lo[u], hi[u]);
          else v = __uint_as_float((uint32_t)(lo[u] >> 32));
          fn(e0 + u * step, v);
        }
    }
  };
  auto to_lds = [&](int32_t e, auto v) { lp[place + e] = (double)v; };

  // (places past the last row are read and have to be finite)
  for (int32_t i = t; i < place; i += kThreads) lp[i] = 0.0;
  if constexpr (kSmall)
    for (int32_t e = t; e < next; e += kThreads) {
      const int32_t g = ext[e];
      gsrc[e] = g;
      gd[e] = dinv_of(g);
      gr[e] = gq[e] = (VT)0;
      lp[place + e] = 0.0;
    }

  // x: the solution (FP64) or the mixed modes' increment
  VT x[RPT], r[RPT], q[RPT], di[DREG ? RPT : 1];
  double rs[DREG ? RPT : 1];
  // the held slots: values (0 past the row's end) and LDS places, two a word
  MT hv[kSmall ? RPT : 1][kSmall ? kHeld : 1];
  uint32_t hc[kSmall ? RPT : 1][kSmall ? kHeld / 2 : 1];
  uint32_t live = 0, needed = 0;
#pragma unroll
  for (int j = 0; j < RPT; ++j) {
    const int32_t g = row(j), i = t + j * kThreads;
    x[j] = r[j] = q[j] = (VT)0;
    if constexpr (DREG) {
      rs[j] = 0.0;
      di[j] = (VT)0;
    }
    if (i < place && g < a.n && at(g) >= 0) {
      live |= 1u << j;
      if (a.needed[g]) needed |= 1u << j;
      if constexpr (DREG) {
        rs[j] = rowsum_of(g);
        di[j] = dinv_of(g);
      }
      if constexpr (kMixed) a.xlo[g] = 0.0;
    }
    if constexpr (kSmall) {
      const bool in = wave + j * kWaves < slices;
      const int32_t o = in ? a.slice_off[slice(j)] : 0;
      const int32_t w = in ? (a.slice_off[slice(j) + 1] - o) >> 6 : 0;
      const MT *vp;
      if constexpr (kMixed) vp = a.val32;
      else vp = a.val;
#pragma unroll
      for (int k = 0; k < kHeld; ++k) {
        const int32_t l = o + 64 * k + (t & 63);
        hv[j][k] = k < w ? vp[l] : (MT)0;
        const uint32_t c = k < w ? (uint32_t)a.lcol[l] : (uint32_t)(in ? i : 0);
        if (k % 2) hc[j][k / 2] |= c << 16;
        else hc[j][k / 2] = c;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }

  // fn(j, local row, row sum of the slots' terms, p_i) for this thread's rows
  auto rows = [&](const auto *val, auto &&fn) {
    const int32_t ti = opaque(t);
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      if (wave + j * kWaves < slices) {
        const int32_t s = slice(j), i = ti + j * kThreads;
        const int32_t o = a.slice_off[s], w = (a.slice_off[s + 1] - o) >> 6;
        const double pi = lp[i];
        const int32_t l = o + (ti & 63);
        fn(j, 64 * s + (ti & 63), ell_lds_row(val + l, a.lcol + l, 0, w, lp, pi, 0.0), pi);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // the same with the held slots, eight gathers in flight
  auto held_rows = [&](const MT *val, auto &&fn) {
    const int32_t ti = opaque(t);
#pragma unroll
    for (int j = 0; j < (kSmall ? RPT : 0); ++j) {
      if (wave + j * kWaves < slices) {
        const int32_t s = slice(j), i = ti + j * kThreads;
        const int32_t o = a.slice_off[s], w = (a.slice_off[s + 1] - o) >> 6;
        const double pi = lp[i];
        double acc = 0.0;
#pragma unroll
        for (int k = 0; k < kHeld; k += 8)
          if (k < w) {
            double y[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
              const uint32_t c = hc[j][(k + u) / 2];
              y[u] = lp[u % 2 ? c >> 16 : c & 0xffffu];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
              acc = __builtin_fma((double)hv[j][k + u], y[u] - pi, acc);
          }
        const int32_t l = o + (ti & 63);
        if (w > kHeld) acc = ell_lds_row(val + l, a.lcol + l, kHeld, w, lp, pi, acc);
        fn(j, 64 * s + (ti & 63), acc, pi);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  bool first = true, ok = true;
  int itp = 0, last_refine = 0, refinements = 0, converged = 0;
  double rr = 0.0, rz = 0.0, bb = 0.0, thr = 0.0, rr_ref = 0.0, rr_out = 0.0;
  for (;;) {
    double s[5] = {0.0, 0.0, 0.0, rr, rz};
    bool refine = first;
    if (!first) {
      if constexpr (kSmall) ++tag;
      else fetch((VT)0, 0, 0, to_lds);
      __syncthreads();
      auto product = [&](int j, int32_t g, double acc, double pi) {
        const double ri = DREG ? rs[DREG ? j : 0] : rowsum_of(min(g, a.n - 1));
        const VT dv = DREG ? di[DREG ? j : 0] : dinv_of(min(g, a.n - 1));
        VT qi = (VT)__builtin_fma(ri, pi, acc);
        qi = (live >> j) & 1 ? qi : (VT)0;
        q[j] = qi;
        if constexpr (kSmall)
          if ((needed >> j) & 1) publish(g, qi, 0);
        const double qd = (double)qi, dq = (double)(dv * qi);
        s[0] = __builtin_fma(pi, qd, s[0]);
        s[1] = __builtin_fma(dq, (double)r[j], s[1]);
        s[2] = __builtin_fma(dq, qd, s[2]);
        pin(q[j]), pin(s[0]), pin(s[1]), pin(s[2]);
      };
      const MT *val;
      if constexpr (kMixed) val = a.val32;
      else val = a.val;
      if constexpr (kSmall) held_rows(val, product);
      else rows(val, product);
      ok = team_sum(tm, sh, s, [&] {
        if constexpr (kSmall)
          fetch((VT)0, 0, sums_threads(tm), [&](int32_t e, VT v) { gq[e] = v; });
      });
      if (!ok) break;
      if constexpr (kMixed) {
        // (a step between two reliable updates, so that the loop ends)
        refine = itp > last_refine && (s[3] < thr || s[3] < a.delta2 * rr_ref ||
                                       itp - last_refine >= a.max_interval || itp >= a.maxit);
      } else {
        rr_out = s[3];
        if (s[3] < thr) {
          converged = 1;
          itp = max(itp - 1, 0);
          break;
        }
        if (itp >= a.maxit) break;
      }
    }
    if (!refine) {
      itp += 1;
      const double rho = s[4], alpha = rho / s[0];
      const double rho_next = rho - 2.0 * alpha * s[1] + alpha * alpha * s[2];
      const VT fa = (VT)alpha, fb = (VT)(rho_next / rho);
      // z and the next p of a row
      auto step = [&](VT dv, VT qi, VT pi, VT &ri, VT &z) {
        if constexpr (MODE == LFGPU_PCG_FP64) {
          ri = __builtin_fma(-fa, qi, ri);
          z = dv * ri;
          return __builtin_fma(fb, pi, z);
        } else {
          ri = ri - fa * qi;
          z = dv * ri;
          return z + fb * pi;
        }
      };
      rr = rz = 0.0;
      if constexpr (!kSmall) ++tag;
      const int32_t ti = opaque(t);
#pragma unroll
      for (int j = 0; j < RPT; ++j) {
        const int32_t i = ti + j * kThreads;
        if ((live >> j) & 1) {
          const int32_t g = 64 * slice(j) + (ti & 63);
          const VT dv = DREG ? di[DREG ? j : 0] : dinv_of(g);
          const VT pi = (VT)lp[i];
          VT z;
          if constexpr (MODE == LFGPU_PCG_FP64) x[j] = __builtin_fma(fa, pi, x[j]);
          else x[j] = x[j] + fa * pi;
          const VT p = step(dv, q[j], pi, r[j], z);
          const double rd = (double)r[j];
          rr = __builtin_fma(rd, rd, rr);
          rz = __builtin_fma(rd, (double)z, rz);
          lp[i] = (double)p;
          if constexpr (!kSmall)
            if ((needed >> j) & 1) publish(g, p, 0);
        }
        pin(r[j]), pin(x[j]), pin(rr), pin(rz);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (kSmall)
        for (int32_t e = ti; e < next; e += kThreads) {
          VT z, rn = gr[e];
          lp[place + e] = (double)step(gd[e], gq[e], (VT)lp[place + e], rn, z);
          gr[e] = rn;
        }
      continue;
    }
    // the first residual b - A x, or a reliable update's b - A x - A (xa + xlo)
    double r64[RPT];
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      const int32_t i = t + j * kThreads;
      r64[j] = (live >> j) & 1 ? a.b[at(row(j))] : 0.0;
      if (!first && ((live >> j) & 1)) q[j] = (VT)lp[i];  // p
      __builtin_amdgcn_sched_barrier(0);
    }
    if (first) {
#pragma unroll
      for (int j = 0; j < RPT; ++j) bb = __builtin_fma(r64[j], r64[j], bb);
    }
    for (int turn = 0; turn < (first ? 1 : 2); ++turn) {
      if (turn == 0) {
        __syncthreads();  // the last readers of LDS are done
      } else {
        // nor does a workgroup overwrite words that another still waits for
        // (who reads whom need not be symmetric where the pattern is not)
        double none[1] = {0.0};
        ok = team_sum(tm, sh, none, [] {});
        if (!ok) break;
      }
      ++tag;
      const int32_t ti = opaque(t);
#pragma unroll
      for (int j = 0; j < RPT; ++j) {
        const int32_t i = ti + j * kThreads;
        if ((live >> j) & 1) {
          const int32_t g = 64 * slice(j) + (ti & 63);
          const double y = turn == 0 ? a.x[at(g)] : (double)x[j] + a.xlo[g];
          if (!kMixed) x[j] = (VT)y;
          lp[i] = y;
          if ((needed >> j) & 1) publish(g, y, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      fetch(0.0, 0, 0, to_lds);
      __syncthreads();
      rows(a.val, [&](int j, int32_t g, double acc, double yi) {
        if ((live >> j) & 1) r64[j] -= __builtin_fma(a.rowsum[g], yi, acc);
        pin(r64[j]);
      });
    }
    if (!ok) break;
    double u[2] = {0.0, bb};
#pragma unroll
    for (int j = 0; j < RPT; ++j) u[0] = __builtin_fma(r64[j], r64[j], u[0]);
    ok = team_sum(tm, sh, u, [] {});
    if (!ok) break;
    rr_out = u[0];
    bool stop;
    if (first) {
      bb = u[1];
      thr = a.tol2 * bb;
      thr = thr > 2.2250738585072014e-308 ? thr : 2.2250738585072014e-308;
      converged = bb == 0.0 || u[0] < thr ? 1 : 0;
      stop = converged || a.maxit <= 0;
    } else {
      refinements += 1;
      last_refine = itp;
      converged = u[0] < thr ? 1 : 0;
      stop = converged || itp >= a.maxit;
#pragma unroll
      for (int j = 0; j < RPT; ++j) {
        if ((live >> j) & 1) {
          const int32_t g = at(row(j));
          const double hi = a.x[g], dx = (double)x[j];
          const double sm = hi + dx, bp = sm - hi;
          const double err = (hi - (sm - bp)) + (dx - bp);
          a.x[g] = sm;
          a.xlo[row(j)] += err;
        }
        x[j] = (VT)0;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    rr_ref = u[0];
    if (stop) break;
    // r = r64, p += M (r64 - r); the first p is M r64
    rr = rz = 0.0;
    ++tag;
    const int32_t ti = opaque(t);
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      const int32_t i = ti + j * kThreads;
      if ((live >> j) & 1) {
        const VT rn = (VT)r64[j];
        const int32_t g = 64 * slice(j) + (ti & 63);
        const VT m = DREG ? di[DREG ? j : 0] : dinv_of(g);
        const VT z = m * rn;
        const VT p = first ? z : q[j] + m * (rn - r[j]);
        r[j] = rn;
        lp[i] = (double)p;
        if ((needed >> j) & 1) {
          publish(g, p, 0);
          if constexpr (kSmall) publish(g, rn, 2);
        }
        // (the first rho, as the sweeps take it: with the FP64 D^-1 and residual)
        const double rd = first ? r64[j] : (double)rn;
        const double zd = first ? a.dinv[g] * rd : (double)z;
        rr = __builtin_fma(rd, rd, rr);
        rz = __builtin_fma(rd, zd, rz);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (kSmall) {
      fetch((VT)0, 0, 0, to_lds);
      fetch((VT)0, 2, 0, [&](int32_t e, VT v) { gr[e] = v; });
    }
    first = false;
  }
  if (ok) {
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      if ((live >> j) & 1) {
        const int32_t g = at(row(j));
        if (bb == 0.0) a.x[g] = 0.0;
        else if (kMixed) a.x[g] = a.x[g] + a.xlo[row(j)];
        else if (!first) a.x[g] = (double)x[j];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (rank == 0 && t == 0) {
    a.st->rr = rr_out;
    a.st->bb = bb;
    a.st->iter = itp;
    a.st->converged = converged;
    a.st->refinements = refinements;
    a.st->aborted = ok ? 0 : 1;
  }
  return ok;
}

template <int MODE, int RPT, bool DREG>
__global__ __launch_bounds__(kThreads) void k_res_ell(EllArgs a) {
  extern __shared__ double dyn[];
  __shared__ SumLds sh;
  (void)ell_solve<MODE, RPT, DREG>(a, blockIdx.x, blockIdx.x, gridDim.x, dyn, sh);
}

// A batch: the workgroups take slots from a counter, in order (batch_loop in
// lfgpu_resident.hip says why that ends).
template <int MODE, int RPT>
__global__ __launch_bounds__(kThreads) void k_res_ell_batch(EllArgs base) {
  extern __shared__ double dyn[];
  __shared__ SumLds sh;
  __shared__ int slot, up;
  if (threadIdx.x == 0) atomicAdd(base.running, 1);
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) slot = atomicAdd(base.ticket, 1);
    __syncthreads();
    const int k = __builtin_amdgcn_readfirstlane(slot);
    if (k >= base.nslots) return;
    const int2 jr = base.job_slots[k];
    if (!team_assembles(base.arrived + jr.x, base.jobs[jr.x].team, base.running, base.abort, up))
      return;
    const EllJob &jb = base.jobs[jr.x];
    EllArgs a = base;
    a.part += jb.sums_at;
    a.total = a.part + part_words(jb.team);
    a.st += jb.index;
    if (!ell_solve<MODE, RPT, true>(a, k, jr.y, jb.team, dyn, sh)) return;
  }
}

// ---------------------------------------------------------------------------
// the split, built once per pattern
// ---------------------------------------------------------------------------
// One workgroup per part: a bitmap of the outside columns over the window
// that 16-bit offsets reach, the number of them before each of its words, which
// gives a column's place behind the own rows, and every slot's place.  home:
// every slice's part and number in it.  parts[g].outside = number of outside
// rows; a part with more than `room` places writes nothing else.  A wavefront
// takes a slice; those of a long row all of them together, four columns of a
// lane in flight (one thread a row, its slots and a binary search for each of
// them one after the other, took 70 ms for a matrix with one row of 20000).
constexpr int kSplitThreads = 512;
constexpr int kSplitWaves = kSplitThreads / 64;
constexpr int32_t kLongSlice = 64;
__global__ __launch_bounds__(kSplitThreads) void k_ell_split(
    int32_t n, const int32_t *slice_off, const int16_t *dcol, const int32_t *slist,
    const int2 *home, int32_t room, EllPart *parts, int32_t *ext, uint16_t *lcol,
    uint8_t *needed) {
  extern __shared__ uint32_t map[];
  __shared__ int32_t sums[kSplitThreads];
  const int t = threadIdx.x, me = blockIdx.x, lane = t & 63, wave = t >> 6;
  EllPart &part = parts[me];
  const int32_t r0 = part.r0, slices = part.slices, rows = 64 * slices;
  slist += part.first;
  int32_t *list = ext + part.at;
  const int32_t words = (part.r1 - r0 + 65567) / 32;
  uint32_t *const ahead = map + words;  // outside columns before a word
  for (int32_t k = t; k < words; k += kSplitThreads) map[k] = 0;
  __syncthreads();
  // fn(slot, column, its slice's part and number) for the part's slots of rows
  // below n, and pad(slot) for the others
  auto slots = [&](auto &&fn, auto &&pad) {
    for (int longs = 0; longs < 2; ++longs)
      for (int32_t i = longs ? 0 : wave; i < slices; i += longs ? 1 : kSplitWaves) {
        const int32_t s = slist[i], r = 64 * s + lane;
        const int32_t o = slice_off[s], w = (slice_off[s + 1] - o) >> 6;
        if ((w > kLongSlice) != (longs != 0)) continue;
        const int32_t step = longs ? kSplitWaves : 1;
        for (int32_t k0 = longs ? wave : 0; k0 < w; k0 += 4 * step) {
          int32_t c[4];
          int2 h[4];
#pragma unroll
          for (int u = 0; u < 4; ++u)
            c[u] = r + dcol[o + 64 * min(k0 + u * step, w - 1) + lane];
#pragma unroll
          for (int u = 0; u < 4; ++u) h[u] = home[r < n ? c[u] >> 6 : 0];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int32_t k = k0 + u * step;
            if (k >= w) continue;
            if (r < n) fn(o + 64 * k + lane, c[u], h[u]);
            else pad(o + 64 * k + lane);
          }
        }
      }
  };
  slots([&](int32_t, int32_t c, int2 h) {
    if (h.x != me) {
      const int32_t b = c - r0 + 32768;
      atomicOr(&map[b >> 5], 1u << (b & 31));
    }
  }, [](int32_t) {});
  __syncthreads();
  // thread t's run of words and the number of outside rows before it
  const int32_t per = (words + kSplitThreads - 1) / kSplitThreads;
  const int32_t k0 = min(t * per, words), k1 = min(k0 + per, words);
  int32_t mine = 0;
  for (int32_t k = k0; k < k1; ++k) mine += __popc(map[k]);
  sums[t] = mine;
  __syncthreads();
  int32_t before = 0, all = 0;
  for (int q = 0; q < kSplitThreads; ++q) {
    if (q < t) before += sums[q];
    all += sums[q];
  }
  if (t == 0) part.outside = all;
  if (all > room - rows) return;
  int32_t e = before;
  for (int32_t k = k0; k < k1; ++k) {
    ahead[k] = e;
    for (uint32_t m = map[k]; m; m &= m - 1) {
      const int32_t c = r0 - 32768 + 32 * k + (__ffs(m) - 1);
      list[e++] = c;
      needed[c] = 1;
    }
  }
  __syncthreads();
  slots([&](int32_t at, int32_t c, int2 h) {
    int32_t place = 64 * h.y + (c & 63);
    if (h.x != me) {
      const int32_t b = c - r0 + 32768;
      place = rows + ahead[b >> 5] + __popc(map[b >> 5] & ((1u << (b & 31)) - 1u));
    }
    lcol[at] = (uint16_t)place;
  }, [&](int32_t at) { lcol[at] = 0; });  // (lanes past the last row)
}

struct EllVariant {
  int rpt;
  const void *fn[3];
};
#define LFG_ELL(R, D)                                                             \
  {R, {reinterpret_cast<const void *>(&k_res_ell<LFGPU_PCG_FP64, R, D>),          \
       reinterpret_cast<const void *>(&k_res_ell<LFGPU_PCG_MIXED, R, D>),         \
       reinterpret_cast<const void *>(&k_res_ell<LFGPU_PCG_MIXED_MATRIX, R, D>)}}
// (Registers spilled, by mode: 26, 14 and 56 with 11 rows a thread, 36, 34 and 50
// with 15, 135, 138 and 114 with 19; the streamed matrix hides most of it: P3 on
// 384 x 384, 11 rows, takes 42.5 us an iteration, 28 of them the matrix.)
const std::vector<EllVariant> kEllVariants = {LFG_ELL(1, true),  LFG_ELL(2, true),
                                              LFG_ELL(3, true),  LFG_ELL(5, true),
                                              LFG_ELL(8, true),  LFG_ELL(11, true),
                                              LFG_ELL(15, false), LFG_ELL(19, false)};
#undef LFG_ELL

const void *const kEllBatch[2][3] = {
    {reinterpret_cast<const void *>(&k_res_ell_batch<LFGPU_PCG_FP64, 2>),
     reinterpret_cast<const void *>(&k_res_ell_batch<LFGPU_PCG_MIXED, 2>),
     reinterpret_cast<const void *>(&k_res_ell_batch<LFGPU_PCG_MIXED_MATRIX, 2>)},
    {reinterpret_cast<const void *>(&k_res_ell_batch<LFGPU_PCG_FP64, 8>),
     reinterpret_cast<const void *>(&k_res_ell_batch<LFGPU_PCG_MIXED, 8>),
     reinterpret_cast<const void *>(&k_res_ell_batch<LFGPU_PCG_MIXED_MATRIX, 8>)}};

}  // namespace

namespace lfgpu {
struct ResidentEllPlan {
  int rpt = 0, nparts = 0;  // rpt 0: does not fit
  size_t lds = 0;           // most bytes of a workgroup
  EllPart *parts = nullptr;
  int32_t *slist = nullptr;   // the parts' slices
  int32_t *ext = nullptr;     // the outside rows of every part, ascending
  uint16_t *lcol = nullptr;   // per slot: the column's place in the workgroup's LDS
  uint8_t *needed = nullptr;  // per row: some other workgroup reads it
  // batches
  EllJob *jobs = nullptr;
  int2 *slots = nullptr;
  word_t *sums = nullptr;
  size_t sums_words = 0;
  ResidentControl *control = nullptr;
  int njobs = 0;
};

static void release(ResidentEllPlan *p) {
  dfree(p->parts);
  dfree(p->slist);
  dfree(p->ext);
  dfree(p->lcol);
  dfree(p->needed);
  dfree(p->jobs);
  dfree(p->slots);
  dfree(p->sums);
  dfree(p->control);
  *p = ResidentEllPlan{};
}

void resident_ell_free(ResidentEllPlan *p) {
  if (!p) return;
  release(p);
  delete p;
}
bool resident_ell_fits(const ResidentEllPlan *p) { return p && p->rpt > 0; }
}  // namespace lfgpu

namespace {

// The parts of a split, their slices one after the other, and each part's
// problem's number of slices, which bounds the outside rows that it can have
// (most of a batch's small problems have one part, and none).
struct Split {
  std::vector<EllPart> parts;
  std::vector<int32_t> slist, of;
  void add(const std::vector<int32_t> &slices, int32_t n) {
    EllPart q{};
    q.r0 = 64 * slices.front();
    q.r1 = std::min(64 * (slices.back() + 1), n);
    q.slices = (int32_t)slices.size();
    q.first = (int32_t)slist.size();
    slist.insert(slist.end(), slices.begin(), slices.end());
    parts.push_back(q);
  }
  // the parts added since the last call make up a problem of n slices
  void problem(int32_t n) { of.resize(parts.size(), n); }
};

// Splits the slices [s0, s1) into runs of `each` slices.  (Runs of equally
// many slots on all 256 CUs: P3 on 384 x 384 takes 44.8 instead of 42.5 us an
// iteration, its parts read more outside rows.)
void split_runs(Split &out, int32_t s0, int32_t s1, int each, int32_t n) {
  std::vector<int32_t> part;
  for (int32_t s = s0; s < s1; s += each) {
    part.clear();
    for (int32_t k = s; k < std::min(s + each, s1); ++k) part.push_back(k);
    out.add(part, n);
  }
}

// The locality order sorts its windows' rows by length: on a third-order
// mesh, the cells', the edges' and then the vertices' rows.  Runs of a few
// slices are of one kind, so that some parts have four times the slots of
// others and read rows all over the window (37 x 29 cells: 600 outside rows in
// a part of edges, 3200 in one of vertices).  Where the windows hold several
// parts, every part gets its share of every length in the window.  Returns
// false if the windows are too small for that, or too many parts result.
bool split_windows(Split &out, const std::vector<int32_t> &off, int32_t s0, int32_t s1, int cap,
                   int most, int32_t n) {
  auto width = [&](int32_t s) { return off[s + 1] - off[s]; };
  std::vector<int32_t> starts{s0};  // of the runs of ascending lengths
  for (int32_t s = s0 + 1; s < s1; ++s)
    if (width(s) < width(s - 1)) starts.push_back(s);
  starts.push_back(s1);
  if (2 * (int64_t)(s1 - s0) < 3 * (int64_t)cap * (int64_t)(starts.size() - 1)) return false;
  const size_t had = out.parts.size(), had_slices = out.slist.size();
  auto fail = [&] {
    out.parts.resize(had);
    out.slist.resize(had_slices);
    return false;
  };
  for (size_t k = 0; k + 1 < starts.size(); ++k) {
    const int32_t u = starts[k], v = starts[k + 1];
    if (v - u > 1024) return fail();  // (the outside rows' bitmap covers a window)
    const int fewest = (v - u + cap - 1) / cap;
    bool done = false;
    for (int m = fewest; m <= fewest + fewest / 8 + 1 && !done; ++m) {
      // slice number k of a length's L goes to the part in which (k + phase) / L
      // of the window lies; the phase spreads lengths of few slices
      std::vector<std::vector<int32_t>> deal(m);
      double phase = 0.5;
      for (int32_t a = u; a < v;) {
        int32_t b = a + 1;
        while (b < v && width(b) == width(a)) ++b;
        for (int32_t s = a; s < b; ++s)
          deal[std::min(m - 1, (int)((s - a + phase) / (b - a) * m))].push_back(s);
        phase = std::fmod(phase + 0.6180339887498949, 1.0);
        a = b;
      }
      // what a part has above its cap goes to the next one with room
      std::vector<int32_t> over;
      for (auto &d : deal)
        for (; (int)d.size() > cap; d.pop_back()) over.push_back(d.back());
      for (auto &d : deal)
        for (; (int)d.size() < cap && !over.empty(); over.pop_back()) d.push_back(over.back());
      if (!over.empty()) continue;
      for (auto &d : deal) {
        if (d.empty()) continue;
        std::sort(d.begin(), d.end());
        out.add(d, n);
      }
      done = true;
    }
    if (!done) return fail();
    if ((int64_t)(out.parts.size() - had) > most) return fail();
  }
  return true;
}

// places that 16 bits and the LDS of a workgroup hold
constexpr int32_t kRoom =
    (int32_t)(kLdsDynamic / sizeof(double) < 65536 ? kLdsDynamic / sizeof(double) : 65536);

// Whether a row couples to more rows than a workgroup has places for.
bool row_too_long(const std::vector<int32_t> &off) {
  for (size_t s = 0; s + 1 < off.size(); ++s)
    if ((off[s + 1] - off[s]) / 64 >= kRoom) return true;
  return false;
}

// LDS of a part
size_t lds_bytes(const EllPart &q, int rpt) {
  const size_t places = 64 * (size_t)q.slices + q.outside;
  return (places + (rpt <= kSmallRows ? 3 * (size_t)q.outside : 0)) * 8 +
         (rpt <= kSmallRows ? 4 * (size_t)q.outside : 0);
}

// Builds the places of a split; *fits tells whether every part fits the LDS.
int ell_split(hipStream_t s, ResidentEllPlan *p, const ResidentEll &A, Split &split, int rpt,
              bool *fits) {
  const int32_t room = kRoom;
  *fits = false;
  int64_t at = 0;
  int32_t span = 0;
  std::vector<int2> home((size_t)(A.n + 63) / 64, int2{-1, 0});
  for (size_t g = 0; g < split.parts.size(); ++g) {
    EllPart &q = split.parts[g];
    if (64 * q.slices >= room) return LFGPU_OK;
    q.at = at;
    at += std::min(room - 64 * q.slices, 64 * (split.of[g] - q.slices));
    span = std::max(span, q.r1 - q.r0);
    for (int32_t k = 0; k < q.slices; ++k)
      home[split.slist[(size_t)q.first + k]] = int2{(int)g, k};
  }
  if (!p->lcol) {
    LFG_TRY(dalloc(&p->lcol, (size_t)std::max<int64_t>(A.slots, 1), "resident ELL places"));
    LFG_TRY(dalloc(&p->needed, (size_t)A.n, "resident ELL flags"));
  }
  dfree(p->ext);
  dfree(p->parts);
  dfree(p->slist);
  p->ext = nullptr;
  p->parts = nullptr;
  p->slist = nullptr;
  LFG_TRY(dalloc(&p->ext, (size_t)at, "resident ELL outside rows"));
  LFG_TRY(dalloc(&p->parts, split.parts.size(), "resident ELL parts"));
  LFG_TRY(dalloc(&p->slist, split.slist.size(), "resident ELL slices"));
  int2 *dhome = nullptr;
  LFG_TRY(dalloc(&dhome, home.size(), "resident ELL slices"));
  hipError_t e = hipMemcpyAsync(dhome, home.data(), home.size() * sizeof(int2),
                                hipMemcpyHostToDevice, s);
  if (e == hipSuccess)
    e = hipMemcpyAsync(p->parts, split.parts.data(), split.parts.size() * sizeof(EllPart),
                       hipMemcpyHostToDevice, s);
  if (e == hipSuccess)
    e = hipMemcpyAsync(p->slist, split.slist.data(), split.slist.size() * 4,
                       hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipMemsetAsync(p->needed, 0, (size_t)A.n, s);
  if (e == hipSuccess) {
    const size_t map = (size_t)(span + 65567) / 32 * 8;
    hipLaunchKernelGGL(k_ell_split, dim3((unsigned)split.parts.size()), dim3(kSplitThreads), map,
                       s, A.n, A.slice_off, A.dcol, p->slist, dhome, room, p->parts, p->ext,
                       p->lcol, p->needed);
    e = hipGetLastError();
  }
  if (e == hipSuccess)
    e = hipMemcpyAsync(split.parts.data(), p->parts, split.parts.size() * sizeof(EllPart),
                       hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  dfree(dhome);
  if (e != hipSuccess) return hip_fail(e, "resident ELL split");
  p->lds = 0;
  for (const EllPart &q : split.parts) {
    if (q.outside > room - 64 * q.slices || lds_bytes(q, rpt) > kLdsDynamic) return LFGPU_OK;
    p->lds = std::max(p->lds, lds_bytes(q, rpt));
  }
  p->nparts = (int)split.parts.size();
  *fits = true;
  return LFGPU_OK;
}

// the slices' offsets
int slice_offsets(hipStream_t s, const ResidentEll &A, std::vector<int32_t> &off) {
  off.resize((size_t)(A.n + 63) / 64 + 1);
  LFG_HIP(hipMemcpyAsync(off.data(), A.slice_off, off.size() * 4, hipMemcpyDeviceToHost, s));
  LFG_HIP(hipStreamSynchronize(s));
  return LFGPU_OK;
}

void fill_args(EllArgs &a, const ResidentEllPlan *plan, const ResidentEll &A,
               const lfgpu_pcg_opts &opts, const double *b, double *x) {
  a.n = A.n;
  a.slice_off = A.slice_off;
  a.lcol = plan->lcol;
  a.val = A.val;
  a.val32 = A.val32;
  a.rowsum = A.rowsum;
  a.rowsum32 = A.rowsum32;
  a.dinv = A.dinv;
  a.dinv32 = A.dinv32;
  a.dinv16 = static_cast<const __hip_bfloat16 *>(A.dinv16);
  a.perm = A.perm;
  a.parts = plan->parts;
  a.slist = plan->slist;
  a.ext = plan->ext;
  a.needed = plan->needed;
  a.b = b;
  a.x = x;
  a.xlo = A.xlo;
  a.tol2 = opts.rtol * opts.rtol;
  a.maxit = opts.maxit;
  a.delta2 = opts.refine_delta > 0.0 ? opts.refine_delta * opts.refine_delta : 0.09;
  a.max_interval = opts.refine_max_interval > 0 ? opts.refine_max_interval : 2147483647;
}

// tags of a solve: one exchange and one sum an iteration, four for a
// reliable update (at most one an iteration), and a few at the start
uint64_t ell_tags(const lfgpu_pcg_opts &opts) {
  return (uint64_t)opts.maxit * (opts.mode == LFGPU_PCG_FP64 ? 1 : 5) + 16;
}

}  // namespace

namespace lfgpu {

int resident_pcg_ell(lfgpu_ctx *ctx, ResidentBufs *bufs, ResidentEllPlan **pplan,
                     const ResidentEll &A, const lfgpu_pcg_opts &opts, const double *b, double *x,
                     ResidentOutcome *out, bool *taken) {
  *taken = false;
  if (A.n <= 0 || !A.dcol) return LFGPU_OK;
  hipStream_t s = ctx->stream;
  const int cus = std::min(ctx->cus, kMaxTeam);
  if (!*pplan) {
    ResidentEllPlan *p = *pplan = new ResidentEllPlan();
    std::vector<int32_t> off;
    LFG_TRY(slice_offsets(s, A, off));
    const int32_t slices = (int32_t)off.size() - 1;
    for (const EllVariant &v : kEllVariants) {
      const int cap = v.rpt * kWaves, want = (slices + cap - 1) / cap;
      if (want > cus || row_too_long(off)) continue;
      Split split;
      if (v.rpt > kSmallRows || !split_windows(split, off, 0, slices, cap, cus, A.n))
        split_runs(split, 0, slices, (slices + want - 1) / want, A.n);
      split.problem(slices);
      bool fits = false;
      LFG_TRY(ell_split(s, p, A, split, v.rpt, &fits));
      if (!fits) continue;
      p->rpt = v.rpt;
      break;
    }
    if (p->rpt == 0) release(p);  // (it only says that the matrix does not fit)
  }
  const ResidentEllPlan *plan = *pplan;
  if (plan->rpt == 0) return LFGPU_OK;
  const EllVariant *v = nullptr;
  for (const EllVariant &k : kEllVariants)
    if (k.rpt == plan->rpt) v = &k;
  EllArgs a{};
  LFG_TRY(resident_prepare(ctx, bufs, (size_t)2 * planes(plan->rpt) * A.n, ell_tags(opts),
                           &a.tag0));
  fill_args(a, plan, A, opts, b, x);
  a.words = bufs->halo;
  a.part = bufs->sums;
  a.total = bufs->sums + kPartWords;
  a.abort = &bufs->outcome->team;
  a.st = &bufs->outcome->solve;
  return resident_launch(s, bufs, v->fn[opts.mode], plan->nparts, &a, plan->lds, out, taken);
}

// The two batch kernels: rows a thread, and what an iteration takes (us, and us
// a slot of a workgroup's rows).
struct EllBatchKind {
  int rpt;
  double fixed, slot;
};
constexpr EllBatchKind kEllBatchKinds[2] = {{2, 2.5, 0.00015}, {8, 6.0, 0.0003}};

// Teams of a batch for one of the kernels.
struct EllTeams {
  std::vector<int32_t> take;   // slices a workgroup, by problem
  std::vector<size_t> order;   // longest problems first
  int64_t workgroups = 0;
  double span = 0.0;           // when the last problem ends
};

// Team sizes as for the lattice problems (resident_tiles_plan); false if a
// problem's team would not fit the chip.
bool ell_teams(const std::vector<ResidentProblem> &probs, const EllBatchKind &kind,
               double slots_per_slice, int cus, EllTeams &out) {
  const size_t np = probs.size();
  const int cap = kind.rpt * kWaves;
  const double slice_us = kind.slot * slots_per_slice;
  auto iterations = [&](const ResidentProblem &q) { return std::sqrt((double)q.n); };
  out.take.resize(np);
  auto team_of = [&](size_t k) {
    return ((probs[k].n + 63) / 64 + out.take[k] - 1) / out.take[k];
  };
  auto total = [&](double tau) {
    int64_t sum = 0;
    for (size_t k = 0; k < np; ++k) {
      const double c = tau > 0.0 ? (tau / iterations(probs[k]) - kind.fixed) / slice_us : cap;
      const int32_t want = (int32_t)std::min<double>(cap, std::max(c, 1.0));
      // evenly over the team, at most kMaxTeam members
      const int32_t n = (probs[k].n + 63) / 64, team = std::min((n + want - 1) / want, cus);
      out.take[k] = (n + team - 1) / team;
      if (out.take[k] > cap) return (int64_t)-1;
      sum += team_of(k);
    }
    return sum;
  };
  out.workgroups = total(0.0);
  if (out.workgroups < 0) return false;
  if (out.workgroups <= cus) {
    double lo = 0.0, hi = 0.0;
    for (const ResidentProblem &q : probs)
      hi = std::max(hi, iterations(q) * (kind.fixed + slice_us * cap));
    for (int step = 0; step < 12; ++step) {
      const double mid = 0.5 * (lo + hi);
      const int64_t n = total(mid);
      if (n >= 0 && n <= cus) hi = mid;
      else lo = mid;
    }
    out.workgroups = total(hi);
  }
  auto cost = [&](size_t k) {
    return iterations(probs[k]) * (kind.fixed + slice_us * out.take[k]);
  };
  out.order.resize(np);
  for (size_t k = 0; k < np; ++k) out.order[k] = k;
  std::stable_sort(out.order.begin(), out.order.end(),
                   [&](size_t i, size_t j) { return cost(i) > cost(j); });
  // the teams in order, each on the workgroups that are free first (ascending,
  // and the new ends go to their place: sorted anew for each of 20000 problems
  // of 8 x 8 unstructured squares, they took 24 ms)
  std::vector<double> until(cus, 0.0);
  out.span = 0.0;
  for (size_t k : out.order) {
    const int team = team_of(k);
    const double end = until[team - 1] + cost(k);
    const auto to = std::upper_bound(until.begin() + team, until.end(), end);
    std::fill(std::copy(until.begin() + team, to, until.begin()), to, end);
    out.span = std::max(out.span, end);
  }
  return true;
}

// The kernel whose teams end first by that model.  64 P3 problems of 8 to 64
// cells: two rows a thread, the matrix half in registers, in turns 18.5 ms;
// eight rows, nearly all problems at once with their matrices streamed, 24.5.
int resident_ell_batch_plan(lfgpu_ctx *ctx, const ResidentEll &A,
                            const std::vector<ResidentProblem> &probs, ResidentEllPlan **out) {
  ResidentEllPlan *p = *out = new ResidentEllPlan();
  hipStream_t s = ctx->stream;
  const int cus = std::min(ctx->cus, kMaxTeam);
  const size_t np = probs.size();
  if (np == 0 || !A.dcol) return LFGPU_OK;
  std::vector<int32_t> off;
  LFG_TRY(slice_offsets(s, A, off));
  if (row_too_long(off)) return LFGPU_OK;
  const double per_slice = 64.0 * (double)A.slots / std::max(A.n, 1);
  EllTeams teams[2];
  bool can[2];
  for (int k = 0; k < 2; ++k) can[k] = ell_teams(probs, kEllBatchKinds[k], per_slice, cus, teams[k]);
  const int better = can[0] && (!can[1] || teams[0].span <= teams[1].span) ? 0 : 1;
  std::vector<EllJob> jobs;
  std::vector<int2> slots;
  bool fits = false;
  // (the small kernel only if every part's LDS holds what it keeps of the
  // outside rows; with its share of the windows' lengths a part, or runs)
  for (int turn = 0; turn < 4 && !fits; ++turn) {
    const int kind = turn < 2 ? better : 1 - better;
    const bool windows = turn % 2 == 0;
    if (!can[kind] || (windows && kind == 1)) continue;
    const EllTeams &t = teams[kind];
    Split split;
    jobs.clear();
    slots.clear();
    p->sums_words = 0;
    for (size_t o = 0; o < np; ++o) {
      const ResidentProblem &q = probs[t.order[o]];
      const int32_t s0 = q.lo / 64, s1 = s0 + (q.n + 63) / 64, each = t.take[t.order[o]];
      const size_t had = split.parts.size();
      if (!windows || !split_windows(split, off, s0, s1, each, cus, A.n))
        split_runs(split, s0, s1, each, A.n);
      split.problem(s1 - s0);
      EllJob j{};
      j.index = q.index;
      j.team = (int32_t)(split.parts.size() - had);
      j.sums_at = p->sums_words;
      if (j.team > 1) p->sums_words += part_words(j.team) + kTotalWords;
      jobs.push_back(j);
      for (int r = 0; r < j.team; ++r) slots.push_back(int2{(int)o, r});
    }
    // (shares of windows may take more workgroups than planned)
    if (windows && t.workgroups <= cus && split.parts.size() > (size_t)cus) continue;
    p->rpt = 0;
    LFG_TRY(ell_split(s, p, A, split, kEllBatchKinds[kind].rpt, &fits));
    if (fits) p->rpt = kEllBatchKinds[kind].rpt;
  }
  if (!fits) return LFGPU_OK;
  LFG_TRY(dalloc(&p->jobs, np, "resident batch jobs"));
  LFG_TRY(dalloc(&p->slots, slots.size(), "resident batch slots"));
  LFG_TRY(dalloc(&p->sums, p->sums_words, "resident batch sums"));
  p->njobs = (int)np;
  LFG_TRY(ResidentControl::alloc(&p->control, np));
  LFG_HIP(hipMemcpyAsync(p->jobs, jobs.data(), np * sizeof(EllJob), hipMemcpyHostToDevice, s));
  LFG_HIP(hipMemcpyAsync(p->slots, slots.data(), slots.size() * sizeof(int2),
                         hipMemcpyHostToDevice, s));
  LFG_HIP(hipStreamSynchronize(s));
  return LFGPU_OK;
}

int resident_ell_batch_run(lfgpu_ctx *ctx, ResidentBufs *bufs, ResidentEllPlan *plan,
                           const ResidentEll &A, const lfgpu_pcg_opts &opts, const double *b,
                           double *x, ResidentState *st, ResidentAbort *ab, bool *taken) {
  *taken = false;
  hipStream_t s = ctx->stream;
  EllArgs a{};
  // (the problems' sums have their own words; they are cleared with the rest)
  const size_t words = (size_t)2 * planes(plan->rpt) * A.n;
  const bool fresh = resident_will_clear(bufs, words, ell_tags(opts));
  LFG_TRY(resident_prepare(ctx, bufs, words, ell_tags(opts), &a.tag0));
  if (fresh) LFG_TRY(resident_clear(s, plan->sums, plan->sums_words));
  LFG_TRY(resident_start_batch(ctx, plan->control, plan->njobs));
  fill_args(a, plan, A, opts, b, x);
  a.words = bufs->halo;
  a.part = plan->sums;
  a.abort = &plan->control->abort;
  a.st = st;
  a.jobs = plan->jobs;
  a.job_slots = plan->slots;
  a.nslots = plan->nparts;
  a.ticket = &plan->control->ticket;
  a.running = &plan->control->running;
  a.arrived = plan->control->arrived();
  LFG_TRY(resident_launch_team(s, kEllBatch[plan->rpt == 2 ? 0 : 1][opts.mode],
                               std::min(plan->nparts, std::min(ctx->cus, kMaxTeam)), &a,
                               plan->lds, taken));
  LFG_HIP(hipMemcpyAsync(ab, a.abort, sizeof(ResidentAbort), hipMemcpyDeviceToHost, s));
  return LFGPU_OK;
}

}  // namespace lfgpu
