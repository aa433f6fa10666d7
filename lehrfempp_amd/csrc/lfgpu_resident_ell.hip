// Resident Jacobi-PCG on sliced ELL (see lfgpu_resident.hip): a workgroup owns
// a run of storage rows (in the locality order, so that what it reads of
// others is a compact neighbourhood), keeps their x, r and q in registers and
// their p in LDS, followed by the p of the outside rows that it reads.  The
// columns are stored once more as places in that LDS array (16 bits).  The
// matrix is streamed every iteration (10 B a slot in FP64, 6 in FP32): what
// the row sweeps spend beside it (two reduction launches, the vectors' trips,
// the gathers' L2 misses) is gone.  Time per iteration, sweeps against this,
// FP64: P1 on 300 x 260 unstructured squares 20.8 -> 7.4 us, 600^2 30.3 ->
// 12.2; P3 on 37 x 29 19.6 -> 7.5, 200^2 35.9 -> 18.6, 384^2 86 -> 45 (226 MB
// of matrix); FP32 matrix, P3 384^2: 64 -> 38.
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

// One workgroup's share: storage rows [r0, r1), LDS places 0.. for them and
// from `rows` on for the `outside` rows listed at ext[at..].
struct EllPart {
  int32_t r0, r1, rows, outside;
  int64_t at;
};
// One problem of a batch.
struct EllJob {
  int32_t index, team;
  uint32_t sums_at;
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
  const int32_t *__restrict__ ext;
  const uint8_t *__restrict__ needed;
  const double *__restrict__ b;
  double *x;
  double *xlo;  // storage order
  word_t *words;  // [2][2][n]
  word_t *part, *total;
  int *abort;
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
  int *ticket;
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

// sum over a row's w slots of v_k (p_{c_k} - pi) from LDS; vp and cp point at
// the row's first slot, a row's slots are 64 apart.  Eight, then four slots'
// loads are issued before the first use.
template <class MT>
__device__ __forceinline__ double ell_lds_row(const MT *__restrict__ vp,
                                              const uint16_t *__restrict__ cp, int32_t w,
                                              const double *lp, double pi) {
  double acc = 0.0;
  int32_t k = 0;
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

// RPT: rows per thread: thread t = 64 wave + lane owns the local rows
// 64 (wave + 8 j) + lane, so a wavefront works on whole slices.  DREG: D^-1
// and row sums in registers (else read every iteration).
template <int MODE, int RPT, bool DREG>
__device__ __forceinline__ bool ell_solve(const EllArgs &a, int32_t slot, int rank, int team,
                                          double *lp, SumLds &sh) {
  typedef typename Mode<MODE>::VT VT;
  typedef typename Mode<MODE>::MT MT;
  constexpr bool kMixed = MODE != LFGPU_PCG_FP64;
  const int t = threadIdx.x;
  Team tm{rank, team, a.part, a.total, a.abort, a.tag0};
  uint32_t tag = a.tag0;
  if (t == 0) sh.bad = 0;
  const EllPart &part = a.parts[slot];
  const int32_t r0 = part.r0, mine = part.r1 - part.r0, place = part.rows;
  const int32_t next = part.outside;
  const int32_t *ext = a.ext + part.at;
  const int32_t s0 = (r0 >> 6) + __builtin_amdgcn_readfirstlane(t >> 6);
  const int32_t slices = (mine + 63) >> 6;

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
  // Publishes row r0 + i's value (VT or, for reliable updates, double) and
  // fetches the outside rows' into LDS, four in flight per thread.
  auto publish = [&](int32_t i, auto v) {
    word_t *w = a.words + (size_t)(tag & 1u) * 2 * a.n + r0 + i;
    if constexpr (sizeof(v) == 8) {
      put(w, low_word(v, tag));
      put(w + a.n, high_word(v, tag));
    } else {
      put(w, ((word_t)__float_as_uint(v) << 32) | tag);
    }
  };
  auto fetch = [&](auto like) {
    constexpr bool kTwo = sizeof(like) == 8;
    const word_t *w = a.words + (size_t)(tag & 1u) * 2 * a.n;
    for (int32_t e0 = t; e0 < next; e0 += 4 * kThreads) {
      int32_t src[4];
      word_t lo[4], hi[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) src[u] = ext[min(e0 + u * kThreads, next - 1)];
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
        if (e0 + u * kThreads < next) {
          if constexpr (kTwo) lp[place + e0 + u * kThreads] = from_words(lo[u], hi[u]);
          else lp[place + e0 + u * kThreads] = (double)__uint_as_float((uint32_t)(lo[u] >> 32));
        }
    }
  };

  // (places past the last row are read and have to be finite)
  for (int32_t i = t; i < place; i += kThreads) lp[i] = 0.0;

  // x: the solution (FP64) or the mixed modes' increment
  VT x[RPT], r[RPT], q[RPT], di[DREG ? RPT : 1];
  double rs[DREG ? RPT : 1];
  uint32_t live = 0, needed = 0;
#pragma unroll
  for (int j = 0; j < RPT; ++j) {
    const int32_t i = t + j * kThreads;
    x[j] = r[j] = q[j] = (VT)0;
    if constexpr (DREG) {
      rs[j] = 0.0;
      di[j] = (VT)0;
    }
    if (i < mine && at(r0 + i) >= 0) {
      live |= 1u << j;
      if (a.needed[r0 + i]) needed |= 1u << j;
      if constexpr (DREG) {
        rs[j] = rowsum_of(r0 + i);
        di[j] = dinv_of(r0 + i);
      }
      if constexpr (kMixed) a.xlo[r0 + i] = 0.0;
    }
    __builtin_amdgcn_sched_barrier(0);
  }

  // fn(j, local row, row sum of the slots' terms, p_i) for this thread's rows
  auto rows = [&](const auto *val, auto &&fn) {
    const int32_t ti = opaque(t);
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      const int32_t s = s0 + j * kWaves;
      if (s - (r0 >> 6) < slices) {
        const int32_t i = ti + j * kThreads;
        const int32_t o = a.slice_off[s], w = (a.slice_off[s + 1] - o) >> 6;
        const double pi = lp[i];
        const int32_t l = o + (ti & 63);
        fn(j, i, ell_lds_row(val + l, a.lcol + l, w, lp, pi), pi);
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
      fetch((VT)0);
      __syncthreads();
      auto product = [&](int j, int32_t i, double acc, double pi) {
        const double ri = DREG ? rs[DREG ? j : 0] : rowsum_of(r0 + min(i, mine - 1));
        const VT dv = DREG ? di[DREG ? j : 0] : dinv_of(r0 + min(i, mine - 1));
        VT qi = (VT)__builtin_fma(ri, pi, acc);
        qi = (live >> j) & 1 ? qi : (VT)0;
        q[j] = qi;
        const double qd = (double)qi, dq = (double)(dv * qi);
        s[0] = __builtin_fma(pi, qd, s[0]);
        s[1] = __builtin_fma(dq, (double)r[j], s[1]);
        s[2] = __builtin_fma(dq, qd, s[2]);
        pin(q[j]), pin(s[0]), pin(s[1]), pin(s[2]);
      };
      if constexpr (kMixed) rows(a.val32, product);
      else rows(a.val, product);
      ok = team_sum(tm, sh, s, [] {});
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
      rr = rz = 0.0;
      ++tag;
      const int32_t ti = opaque(t);
#pragma unroll
      for (int j = 0; j < RPT; ++j) {
        const int32_t i = ti + j * kThreads;
        if ((live >> j) & 1) {
          const VT dv = DREG ? di[DREG ? j : 0] : dinv_of(r0 + i);
          const VT pi = (VT)lp[i];
          VT z, p;
          if constexpr (MODE == LFGPU_PCG_FP64) {
            x[j] = __builtin_fma(fa, pi, x[j]);
            r[j] = __builtin_fma(-fa, q[j], r[j]);
            z = dv * r[j];
            p = __builtin_fma(fb, pi, z);
          } else {
            x[j] = x[j] + fa * pi;
            r[j] = r[j] - fa * q[j];
            z = dv * r[j];
            p = z + fb * pi;
          }
          const double rd = (double)r[j];
          rr = __builtin_fma(rd, rd, rr);
          rz = __builtin_fma(rd, (double)z, rz);
          lp[i] = (double)p;
          if ((needed >> j) & 1) publish(i, p);
        }
        pin(r[j]), pin(x[j]), pin(rr), pin(rz);
        __builtin_amdgcn_sched_barrier(0);
      }
      continue;
    }
    // the first residual b - A x, or a reliable update's b - A x - A xa - A xlo
    double r64[RPT];
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      const int32_t i = t + j * kThreads;
      r64[j] = (live >> j) & 1 ? a.b[at(r0 + i)] : 0.0;
      if (!first && ((live >> j) & 1)) q[j] = (VT)lp[i];  // p
      __builtin_amdgcn_sched_barrier(0);
    }
    if (first) {
#pragma unroll
      for (int j = 0; j < RPT; ++j) bb = __builtin_fma(r64[j], r64[j], bb);
    }
    for (int turn = 0; turn < (first ? 1 : 3); ++turn) {
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
          const double y = turn == 0 ? a.x[at(r0 + i)] : turn == 1 ? (double)x[j] : a.xlo[r0 + i];
          if (!kMixed) x[j] = (VT)y;
          lp[i] = y;
          if ((needed >> j) & 1) publish(i, y);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      fetch(0.0);
      __syncthreads();
      rows(a.val, [&](int j, int32_t i, double acc, double yi) {
        if ((live >> j) & 1) r64[j] -= __builtin_fma(a.rowsum[r0 + i], yi, acc);
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
        const int32_t i = t + j * kThreads;
        if ((live >> j) & 1) {
          const int32_t g = at(r0 + i);
          const double hi = a.x[g], dx = (double)x[j];
          const double sm = hi + dx, bp = sm - hi;
          const double err = (hi - (sm - bp)) + (dx - bp);
          a.x[g] = sm;
          a.xlo[r0 + i] += err;
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
        const VT m = DREG ? di[DREG ? j : 0] : dinv_of(r0 + i);
        const VT z = m * rn;
        const VT p = first ? z : q[j] + m * (rn - r[j]);
        r[j] = rn;
        lp[i] = (double)p;
        if ((needed >> j) & 1) publish(i, p);
        // (the first rho, as the sweeps take it: with the FP64 D^-1 and residual)
        const double rd = first ? r64[j] : (double)rn;
        const double zd = first ? a.dinv[r0 + i] * rd : (double)z;
        rr = __builtin_fma(rd, rd, rr);
        rz = __builtin_fma(rd, zd, rz);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    first = false;
  }
  if (ok) {
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      const int32_t i = t + j * kThreads;
      if ((live >> j) & 1) {
        const int32_t g = at(r0 + i);
        if (bb == 0.0) a.x[g] = 0.0;
        else if (kMixed) a.x[g] = a.x[g] + a.xlo[r0 + i];
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
  __shared__ int slot;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) slot = atomicAdd(base.ticket, 1);
    __syncthreads();
    const int k = __builtin_amdgcn_readfirstlane(slot);
    if (k >= base.nslots) return;
    const int2 jr = base.job_slots[k];
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
// that 16-bit offsets reach, its prefix sums as their places behind the own
// rows, and every slot's place.  parts[g].outside = number of outside rows; a
// part with more than `room` writes nothing else.
constexpr int kSplitThreads = 512;
__global__ __launch_bounds__(kSplitThreads) void k_ell_split(const int32_t *slice_off,
                                                             const int16_t *dcol, int32_t room,
                                                             EllPart *parts, int32_t *ext,
                                                             uint16_t *lcol, uint8_t *needed) {
  extern __shared__ uint32_t map[];
  __shared__ int32_t sums[kSplitThreads];
  const int t = threadIdx.x;
  EllPart &part = parts[blockIdx.x];
  const int32_t r0 = part.r0, r1 = part.r1, rows = part.rows;
  int32_t *list = ext + part.at;
  const int32_t words = (rows + 65536) / 32;
  for (int32_t k = t; k < words; k += kSplitThreads) map[k] = 0;
  __syncthreads();
  for (int32_t r = r0 + t; r < r1; r += kSplitThreads) {
    const int32_t s = r >> 6, o = slice_off[s] + (r & 63), w = (slice_off[s + 1] - slice_off[s]) >> 6;
    for (int32_t k = 0; k < w; ++k) {
      const int32_t c = r + dcol[o + 64 * k];
      if (c < r0 || c >= r1) {
        const int32_t b = c - r0 + 32768;
        atomicOr(&map[b >> 5], 1u << (b & 31));
      }
    }
  }
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
  for (int32_t k = k0; k < k1; ++k)
    for (uint32_t m = map[k]; m; m &= m - 1) {
      const int32_t c = r0 - 32768 + 32 * k + (__ffs(m) - 1);
      list[e++] = c;
      needed[c] = 1;
    }
  __syncthreads();
  const int32_t s1 = (r1 + 63) >> 6;
  for (int32_t r = r0 + t; r < s1 * 64; r += kSplitThreads) {
    const int32_t s = r >> 6, o = slice_off[s] + (r & 63), w = (slice_off[s + 1] - slice_off[s]) >> 6;
    for (int32_t k = 0; k < w; ++k) {
      int32_t at = 0;  // (lanes past the last row)
      if (r < r1) {
        const int32_t c = r + dcol[o + 64 * k];
        if (c >= r0 && c < r1) {
          at = c - r0;
        } else {
          // place of c among the outside rows: binary search in the list
          int32_t lo = 0, hi = all - 1;
          while (lo < hi) {
            const int32_t m = (lo + hi) >> 1;
            if (list[m] < c) lo = m + 1;
            else hi = m;
          }
          at = rows + lo;
        }
      }
      lcol[o + 64 * k] = (uint16_t)at;
    }
  }
}

struct EllVariant {
  int rpt;
  const void *fn[3];
};
#define LFG_ELL(R, D)                                                             \
  {R, {reinterpret_cast<const void *>(&k_res_ell<LFGPU_PCG_FP64, R, D>),          \
       reinterpret_cast<const void *>(&k_res_ell<LFGPU_PCG_MIXED, R, D>),         \
       reinterpret_cast<const void *>(&k_res_ell<LFGPU_PCG_MIXED_MATRIX, R, D>)}}
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
  int32_t most = 0;         // most places (own and outside rows) of a workgroup
  EllPart *parts = nullptr;
  int32_t *ext = nullptr;     // the outside rows of every part, ascending
  uint16_t *lcol = nullptr;   // per slot: the column's place in the workgroup's LDS
  uint8_t *needed = nullptr;  // per row: some other workgroup reads it
  // batches
  EllJob *jobs = nullptr;
  int2 *slots = nullptr;
  word_t *sums = nullptr;
  size_t sums_words = 0;
  int *ticket = nullptr;  // followed by the abort flag
};

void resident_ell_free(ResidentEllPlan *p) {
  if (!p) return;
  dfree(p->parts);
  dfree(p->ext);
  dfree(p->lcol);
  dfree(p->needed);
  dfree(p->jobs);
  dfree(p->slots);
  dfree(p->sums);
  dfree(p->ticket);
  delete p;
}
bool resident_ell_fits(const ResidentEllPlan *p) { return p && p->rpt > 0; }
}  // namespace lfgpu

namespace {

// Splits the storage into the given parts (r0, r1, rows filled in); *fits
// tells whether every part's places fit the LDS.
int ell_split(hipStream_t s, ResidentEllPlan *p, const ResidentEll &A, std::vector<EllPart> &parts,
              bool *fits) {
  const int32_t room = (int32_t)std::min<size_t>(kLdsDynamic / sizeof(double), 65536);
  *fits = false;
  int64_t at = 0;
  int32_t rows = 0;
  for (EllPart &q : parts) {
    if (q.rows >= room) return LFGPU_OK;
    q.at = at;
    at += room - q.rows;
    rows = std::max(rows, q.rows);
  }
  if (!p->lcol) {
    LFG_TRY(dalloc(&p->lcol, (size_t)std::max<int64_t>(A.slots, 1), "resident ELL places"));
    LFG_TRY(dalloc(&p->needed, (size_t)A.n, "resident ELL flags"));
  }
  dfree(p->ext);
  dfree(p->parts);
  p->ext = nullptr;
  p->parts = nullptr;
  LFG_TRY(dalloc(&p->ext, (size_t)at, "resident ELL outside rows"));
  LFG_TRY(dalloc(&p->parts, parts.size(), "resident ELL parts"));
  LFG_HIP(hipMemcpyAsync(p->parts, parts.data(), parts.size() * sizeof(EllPart),
                         hipMemcpyHostToDevice, s));
  LFG_HIP(hipMemsetAsync(p->needed, 0, (size_t)A.n, s));
  const size_t map = (size_t)(rows + 65536) / 32 * 4;
  hipLaunchKernelGGL(k_ell_split, dim3((unsigned)parts.size()), dim3(kSplitThreads), map, s,
                     A.slice_off, A.dcol, room, p->parts, p->ext, p->lcol, p->needed);
  LFG_HIP(hipGetLastError());
  LFG_HIP(hipMemcpyAsync(parts.data(), p->parts, parts.size() * sizeof(EllPart),
                         hipMemcpyDeviceToHost, s));
  LFG_HIP(hipStreamSynchronize(s));
  p->most = 0;
  for (const EllPart &q : parts) {
    if (q.outside > room - q.rows) return LFGPU_OK;
    p->most = std::max(p->most, q.rows + q.outside);
  }
  p->nparts = (int)parts.size();
  *fits = true;
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
                     ResidentState *st, bool *taken) {
  *taken = false;
  if (A.n <= 0 || !A.dcol) return LFGPU_OK;
  hipStream_t s = ctx->stream;
  const int cus = std::min(ctx->cus, kMaxTeam);
  if (!*pplan) {
    ResidentEllPlan *p = *pplan = new ResidentEllPlan();
    for (const EllVariant &v : kEllVariants) {
      const int64_t want = (A.n + (int64_t)v.rpt * kThreads - 1) / ((int64_t)v.rpt * kThreads);
      if (want > cus) continue;
      const int32_t rows = (int32_t)(((A.n + want - 1) / want + 63) / 64 * 64);
      std::vector<EllPart> parts((A.n + rows - 1) / rows);
      for (size_t g = 0; g < parts.size(); ++g)
        parts[g] = EllPart{(int32_t)g * rows, std::min((int32_t)(g + 1) * rows, A.n), rows, 0, 0};
      bool fits = false;
      LFG_TRY(ell_split(s, p, A, parts, &fits));
      if (!fits) continue;
      p->rpt = v.rpt;
      break;
    }
  }
  const ResidentEllPlan *plan = *pplan;
  if (plan->rpt == 0) return LFGPU_OK;
  const EllVariant *v = nullptr;
  for (const EllVariant &k : kEllVariants)
    if (k.rpt == plan->rpt) v = &k;
  EllArgs a{};
  LFG_TRY(resident_prepare(s, bufs, (size_t)4 * A.n, ell_tags(opts), &a.tag0));
  fill_args(a, plan, A, opts, b, x);
  a.words = bufs->halo;
  a.part = bufs->sums;
  a.total = bufs->sums + kPartWords;
  a.abort = bufs->abort;
  a.st = bufs->state;
  return resident_launch(s, bufs, v->fn[opts.mode], plan->nparts, &a,
                         (size_t)plan->most * sizeof(double), st, taken);
}

// Team sizes as for the lattice problems (resident_tiles_plan): an iteration
// takes about 6 us and 0.3 ns a slot of a workgroup's rows.
int resident_ell_batch_plan(lfgpu_ctx *ctx, const ResidentEll &A,
                            const std::vector<ResidentProblem> &probs, ResidentEllPlan **out) {
  ResidentEllPlan *p = *out = new ResidentEllPlan();
  hipStream_t s = ctx->stream;
  const int cus = std::min(ctx->cus, kMaxTeam);
  const size_t np = probs.size();
  if (np == 0 || !A.dcol) return LFGPU_OK;
  const int32_t cap = 8 * kThreads;
  const double row_us = 0.0003 * (double)A.slots / std::max(A.n, 1);
  auto iterations = [&](const ResidentProblem &q) { return std::sqrt((double)q.n); };
  std::vector<int32_t> rows(np);
  auto total = [&](double tau) {
    int64_t sum = 0;
    for (size_t k = 0; k < np; ++k) {
      const double c = tau > 0.0 ? (tau / iterations(probs[k]) - 6.0) / row_us : (double)cap;
      const int32_t want = (int32_t)std::min<double>((double)cap, std::max(c, 64.0));
      const int32_t n = (probs[k].n + 63) / 64 * 64;
      // evenly over the team, whole slices, at most kMaxTeam members
      const int32_t team = std::min((n + want - 1) / want, cus);
      rows[k] = ((n + team - 1) / team + 63) / 64 * 64;
      if (rows[k] > cap) return (int64_t)-1;
      sum += (n + rows[k] - 1) / rows[k];
    }
    return sum;
  };
  const int64_t all = total(0.0);
  if (all < 0) return LFGPU_OK;
  if (all <= cus) {
    double lo = 0.0, hi = 0.0;
    for (const ResidentProblem &q : probs)
      hi = std::max(hi, iterations(q) * (6.0 + row_us * cap));
    for (int step = 0; step < 12; ++step) {
      const double mid = 0.5 * (lo + hi);
      const int64_t n = total(mid);
      if (n >= 0 && n <= cus) hi = mid;
      else lo = mid;
    }
    (void)total(hi);
  }
  std::vector<size_t> order(np);
  for (size_t k = 0; k < np; ++k) order[k] = k;
  auto cost = [&](size_t k) { return iterations(probs[k]) * (6.0 + row_us * rows[k]); };
  std::stable_sort(order.begin(), order.end(),
                   [&](size_t i, size_t j) { return cost(i) > cost(j); });
  std::vector<EllJob> jobs(np);
  std::vector<EllPart> parts;
  std::vector<int2> slots;
  int32_t most = 0;
  for (size_t o = 0; o < np; ++o) {
    const ResidentProblem &q = probs[order[o]];
    const int32_t R = rows[order[o]], end = q.lo + (q.n + 63) / 64 * 64;
    EllJob &j = jobs[o];
    j.index = q.index;
    j.team = (end - q.lo + R - 1) / R;
    j.sums_at = (uint32_t)p->sums_words;
    p->sums_words += part_words(j.team) + kTotalWords;
    most = std::max(most, R);
    for (int r = 0; r < j.team; ++r) {
      parts.push_back(EllPart{q.lo + r * R, std::min(q.lo + (r + 1) * R, end), R, 0, 0});
      slots.push_back(int2{(int)o, r});
    }
  }
  bool fits = false;
  LFG_TRY(ell_split(s, p, A, parts, &fits));
  if (!fits) return LFGPU_OK;
  LFG_TRY(dalloc(&p->jobs, np, "resident batch jobs"));
  LFG_TRY(dalloc(&p->slots, slots.size(), "resident batch slots"));
  LFG_TRY(dalloc(&p->sums, p->sums_words, "resident batch sums"));
  LFG_TRY(dalloc(&p->ticket, 4, "resident batch counter"));
  LFG_HIP(hipMemcpyAsync(p->jobs, jobs.data(), np * sizeof(EllJob), hipMemcpyHostToDevice, s));
  LFG_HIP(hipMemcpyAsync(p->slots, slots.data(), slots.size() * sizeof(int2),
                         hipMemcpyHostToDevice, s));
  LFG_HIP(hipStreamSynchronize(s));
  p->rpt = most <= 2 * kThreads ? 2 : 8;
  return LFGPU_OK;
}

int resident_ell_batch_run(lfgpu_ctx *ctx, ResidentBufs *bufs, ResidentEllPlan *plan,
                           const ResidentEll &A, const lfgpu_pcg_opts &opts, const double *b,
                           double *x, ResidentState *st, bool *taken) {
  *taken = false;
  hipStream_t s = ctx->stream;
  EllArgs a{};
  // (the problems' sums have their own words; they are cleared with the rest)
  const bool fresh = resident_will_clear(bufs, (size_t)4 * A.n, ell_tags(opts));
  LFG_TRY(resident_prepare(s, bufs, (size_t)4 * A.n, ell_tags(opts), &a.tag0));
  if (fresh) LFG_TRY(resident_clear(s, plan->sums, plan->sums_words));
  // the counter and the abort flag
  LFG_TRY(resident_clear(s, reinterpret_cast<unsigned long long *>(plan->ticket), 2));
  fill_args(a, plan, A, opts, b, x);
  a.words = bufs->halo;
  a.part = plan->sums;
  a.abort = plan->ticket + 2;
  a.st = st;
  a.jobs = plan->jobs;
  a.job_slots = plan->slots;
  a.nslots = plan->nparts;
  a.ticket = plan->ticket;
  return resident_launch_team(s, kEllBatch[plan->rpt == 2 ? 0 : 1][opts.mode],
                              std::min(plan->nparts, std::min(ctx->cus, kMaxTeam)), &a,
                              (size_t)plan->most * sizeof(double), taken);
}

}  // namespace lfgpu
