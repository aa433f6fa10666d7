// Resident Jacobi-PCG: one cooperative launch runs a whole solve.
//
// The sweeps of lfgpu_solver.hip move every vector through memory twice an
// iteration (128 B a row in FP64) and pay two launches; below a million rows
// the launches alone bound them.  Here a team of up to 256 workgroups, one
// per CU, keeps x, r and q in registers and the search direction p in LDS
// (the chip holds 128 MB of registers and 40 MB of LDS).  Up to 9 rows a
// thread (1.18M rows on 256 CUs) the matrix stays in registers too and an
// iteration touches memory only for the boundary values and the team sums;
// above, the matrix is streamed once an iteration.  Time per iteration, P1,
// sweeps against this: 64^2 12.5 -> 3.2 us, 512^2 17.9 -> 5.3, 1024^2 32.0
// -> 10.0, 2048 x 256 21.3 -> 11.7, 1400^2 53.9 -> 21.6, 2048^2 101 -> 52.8.
//
// One iteration (the recurrences and the stopping test of the two-sweep
// solver, with one team sum instead of two):
//   q = A p; team sum of p.q, (q, D^-1 r), (q, D^-1 q) and of ||r||^2 and
//   (r, D^-1 r) left by the previous update; stop if ||r||^2 < thr;
//   alpha = rho / p.q, beta from rho' = rho - 2 alpha (q, D^-1 r) +
//   alpha^2 (q, D^-1 q); x += alpha p, r -= alpha q, p = D^-1 r + beta p,
//   the boundary values of p published as they are formed.
// The product that runs beside the stopping test of the last iteration is
// discarded, x is what the test was made on.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>

#include "lfgpu_reduce.h"
#include "lfgpu_resident.h"
#include "lfgpu_resident_device.h"

using namespace lfgpu;
using namespace lfgpu::res;

namespace {

constexpr int kMaxD = 6;

struct DiaArgs {
  int32_t n, rows;  // rows per workgroup
  int32_t halo;     // largest |offset|
  int32_t slots;    // published values per workgroup
  int32_t lds;      // doubles of LDS
  int ndiag;
  int32_t off[kMaxD];
  const double *__restrict__ val;
  const double *__restrict__ rowsum;
  const double *__restrict__ dinv;
  const double *__restrict__ b;
  double *__restrict__ x;
  word_t *halo_words;  // [2][team][2][slots]
  word_t *part, *total;
  int *abort;
  uint32_t tag0;
  double tol2;
  int maxit;
  ResidentState *st;
};

// A value of an array at a uniform base and a 32-bit byte offset per lane (one
// address register for all the arrays of a row).
__device__ __forceinline__ double load_at(const double *base, uint32_t bytes) {
  return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(base) + bytes);
}
// Hides a value from the optimiser, which else keeps every row's addresses
// and masks in registers across the iterations (several hundred of them).
__device__ __forceinline__ int32_t opaque(int32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}
__device__ __forceinline__ int32_t opaque_uniform(int32_t v) {
  asm volatile("" : "+s"(v));
  return v;
}
// Keeps a row's result where it is computed (the compiler else sinks whole
// rows past the next barrier and spills their operands).
__device__ __forceinline__ void pin(double &v) { asm volatile("" : "+v"(v)); }

// The workgroup's rows and its place in the team's halo exchange: local row
// i (0 <= i < rows) is global row r0 + i; its value sits at lp[halo + i], the
// `halo` rows before and after at lp[0..halo) and lp[halo + rows ..).
struct DiaRows {
  int32_t n, r0, rows, mine, halo, slots, rank, team;
  word_t *words;
  int *abort;
  uint32_t tag;

  __device__ __forceinline__ word_t *slot(int32_t owner) const {
    return words + ((size_t)(tag & 1u) * team + owner) * 2 * slots;
  }
  __device__ __forceinline__ int32_t mine_of(int32_t g) const { return min(rows, n - g * rows); }
  // fetches the lower (UP = false) or upper halo into dst[0..halo) with the
  // threads from `first` on; four values' words are in flight per thread
  // before the first is checked
  template <bool UP>
  __device__ __forceinline__ void fetch(double *dst, int first, int *bad) const {
    const int32_t owner = UP ? rank + 1 : rank - 1;
    if (owner < 0 || owner >= team) return;
    const int32_t have = UP ? min(halo, mine_of(owner)) : halo;
    const int32_t base = UP ? 0 : (rows <= 2 * halo ? rows - halo : halo);
    const int32_t step = kThreads - first;
    const word_t *w = slot(owner) + base;
    for (int32_t h0 = (int32_t)threadIdx.x - first; h0 < have; h0 += 4 * step) {
      word_t lo[4], hi[4];
      bool ok;
      Wait wait(abort);
      do {
        ok = true;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int32_t h = min(h0 + u * step, have - 1);
          lo[u] = get(&w[h]);
          hi[u] = get(&w[slots + h]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) ok = ok && tagged(lo[u], tag) && tagged(hi[u], tag);
      } while (!ok && wait.more());
      if (!ok) *bad = 1;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (h0 + u * step < have) dst[h0 + u * step] = from_words(lo[u], hi[u]);
    }
  }
};

// The rows that a workgroup publishes in one exchange: the first and the last
// `halo` (none without a team).
struct Publisher {
  int32_t below, from, shift, mine;
  uint32_t tag;
  word_t *lo, *hi;
  __device__ __forceinline__ explicit Publisher(const DiaRows &D)
      : below(D.team > 1 ? D.halo : 0),
        from(D.team > 1 ? D.rows - D.halo : 0x7fffffff),
        shift(max(D.rows - 2 * D.halo, 0)),
        mine(D.mine),
        tag(D.tag),
        lo(D.slot(D.rank)),
        hi(lo + D.slots) {}
  // local row i of a wavefront whose first row (uniform) is i0
  __device__ __forceinline__ void operator()(int32_t i0, int32_t i, double v) const {
    if (i0 >= below && i0 + 63 < from) return;
    if ((i < below || i >= from) && i < mine) {
      const uint32_t at = (uint32_t)(i < below ? i : i - shift);
      put(lo + at, low_word(v, tag));
      put(hi + at, high_word(v, tag));
    }
  }
};

constexpr int ND = 6;  // off-diagonals of a P1 matrix on a structured mesh

// How a variant keeps the neighbours' values of p and the matrix.
//   GHOST: the matrix stays in registers.  The neighbours' r, q, D^-1 and p
//     of the halo rows are kept here as well and updated by the same
//     operations as their owners', so that what travels is q: it is published
//     with the partial sums and arrives while the team sum runs, which takes
//     the exchange off the iteration's critical path.
//   HALO: the matrix stays in registers; p travels, published by the update
//     and waited for by the next product.
//   STREAM: p travels as in HALO; the matrix (its upper half: symmetric
//     values) is read from memory every iteration, the next row's loads in
//     flight while a row is worked on.  The upper halo takes the lower one's
//     place for the second half of the rows, which is what lets 16401 rows
//     with offsets of 2050 fit 160 KB.
enum { GHOST, HALO, STREAM };

// RPT: rows per thread (thread t of a workgroup owns its local rows t + 512 j).
// XR: the rows j < XR keep their x in a register, the others' is read and
// written in every update (as many as the registers hold without spills).
template <int KIND, int RPT, int XR>
__global__ __launch_bounds__(kThreads) void k_res_dia(DiaArgs a) {
  constexpr bool kStream = KIND == STREAM, kGhost = KIND == GHOST;
  constexpr int kHalf = (RPT + 1) / 2;  // STREAM: rows before the upper halo's turn
  extern __shared__ double lp[];
  __shared__ SumLds sh;
  const int t = threadIdx.x;
  const int32_t w0 = __builtin_amdgcn_readfirstlane(t & ~63);  // the wavefront's first row
  DiaRows D;
  D.n = a.n;
  D.rank = blockIdx.x;
  D.team = gridDim.x;
  D.rows = a.rows;
  D.r0 = D.rank * a.rows;
  D.mine = D.mine_of(D.rank);
  D.halo = a.halo;
  D.slots = a.slots;
  D.words = a.halo_words;
  D.abort = a.abort;
  D.tag = a.tag0;
  Team tm{D.rank, D.team, a.part, a.total, a.abort, a.tag0};
  if (t == 0) sh.bad = 0;
  const int32_t mine = D.mine, H = a.halo;
  for (int32_t i = t; i < a.lds; i += kThreads) lp[i] = 0.0;
  double *const up = lp + (kStream ? 0 : H + a.rows);  // the upper halo
  // GHOST: r, q and D^-1 of the halo rows
  double *const gr = lp + 2 * H + RPT * kThreads, *const gq = gr + 2 * H, *const gd = gq + 2 * H;

  double x[XR > 0 ? XR : 1], r[RPT], q[RPT];
  double v[kStream ? 1 : RPT][ND], rs[kStream ? 1 : RPT], di[kStream ? 1 : RPT];
  const double *rowsum = a.rowsum + D.r0, *dinv = a.dinv + D.r0;
  double *xg = a.x + D.r0;
  __syncthreads();
  // x0 and its boundary values
  ++D.tag;
  const Publisher pub0(D);
#pragma unroll
  for (int j = 0; j < RPT; ++j) {
    const int32_t i = t + j * kThreads;
    r[j] = q[j] = 0.0;
    if (j < XR) x[j] = 0.0;
    if constexpr (!kStream) {
      rs[j] = di[j] = 0.0;
#pragma unroll
      for (int d = 0; d < ND; ++d) v[j][d] = 0.0;
    }
    if (i < mine) {
      const double xi = xg[i];
      if (j < XR) x[j] = xi;
      lp[H + i] = xi;
      pub0(w0 + j * kThreads, i, xi);
      if constexpr (!kStream) {
        rs[j] = rowsum[i];
        di[j] = dinv[i];
#pragma unroll
        for (int d = 0; d < ND; ++d)
          if (d < a.ndiag) v[j][d] = a.val[(int64_t)d * a.n + D.r0 + i];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (kGhost) {
    for (int32_t h = t; h < 2 * H; h += kThreads) {
      const int32_t g = h < H ? D.r0 - H + h : D.r0 + D.rows + h - H;
      if (g >= 0 && g < a.n) gd[h] = a.dinv[g];
    }
  }

  // q_j = (A p)_i in difference form from LDS, handed to fn with p_i and
  // D^-1_i; the rows past the workgroup's end give q = 0
  auto sweep = [&](auto &&fn) {
    const int32_t ti = opaque(t);
    const double *lc = lp + H + ti;
    const double *bp[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) bp[d] = lc + a.off[d];
    if constexpr (!kStream) {
#pragma unroll
      for (int j = 0; j < RPT; ++j) {
        // every LDS read of the row before the first use
        const double pi = lc[j * kThreads];
        double c[ND], acc = 0.0;
#pragma unroll
        for (int d = 0; d < ND; ++d) c[d] = bp[d][j * kThreads];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int d = 0; d < ND; ++d) acc = __builtin_fma(v[j][d], c[d] - pi, acc);
        q[j] = __builtin_fma(rs[j], pi, acc);
        pin(q[j]);
        fn(j, pi, di[j]);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      // the next row of the stream: the diagonals (the lower ones as the
      // mirrored upper ones), row sum and D^-1
      double nv[ND], ns, nd;
      auto load_row = [&](int j) {
        const uint32_t at = (uint32_t)min(ti + j * kThreads, mine - 1) * 8u;
#pragma unroll
        for (int d = 0; d < ND; ++d) {
          const double *m = a.val + (int64_t)(d < ND / 2 ? ND - 1 - d : d) * a.n + D.r0;
          if (d < ND / 2) {
            m += a.off[d];
            // (only the first workgroup's first rows have no such neighbour)
            if (j < kHalf) {
              const int32_t from = -(D.r0 + a.off[d]) * 8;
              const double w = load_at(m, (uint32_t)max((int32_t)at, from));
              nv[d] = (int32_t)at >= from ? w : 0.0;
            } else {
              nv[d] = load_at(m, at);
            }
          } else {
            nv[d] = load_at(m, at);
          }
        }
        ns = load_at(rowsum, at);
        nd = load_at(dinv, at);
      };
      load_row(0);
      D.template fetch<false>(lp, 0, &sh.bad);
      __syncthreads();
#pragma unroll
      for (int j = 0; j < RPT; ++j) {
        if (j == kHalf) {
          __syncthreads();
          D.template fetch<true>(up, 0, &sh.bad);
          __syncthreads();
        }
        double vr[ND];
#pragma unroll
        for (int d = 0; d < ND; ++d) vr[d] = nv[d];
        const double s = ns, dv = nd;
        // every LDS read of the row and the next row's loads before the first use
        const double pi = lc[j * kThreads];
        double c[ND], acc = 0.0;
#pragma unroll
        for (int d = 0; d < ND; ++d) {
          const double *p = bp[d] + j * kThreads;
          // past the last row: the upper halo in the lower one's place
          if (j >= kHalf && d >= ND / 2)
            if (ti >= a.rows - a.off[d] - j * kThreads) p -= H + a.rows;
          c[d] = *p;
        }
        if (j + 1 < RPT) load_row(j + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int d = 0; d < ND; ++d) acc = __builtin_fma(vr[d], c[d] - pi, acc);
        const double qi = __builtin_fma(s, pi, acc);
        q[j] = ti + j * kThreads < mine ? qi : 0.0;
        pin(q[j]);
        fn(j, pi, dv);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  double rr = 0.0, rz = 0.0, bb = 0.0;
  if constexpr (!kStream) {
    D.template fetch<false>(lp, 0, &sh.bad);
    D.template fetch<true>(up, 0, &sh.bad);
    __syncthreads();
  }
  sweep([&](int, double, double) {});
  __syncthreads();
  // r = b - A x, p = D^-1 r; r (GHOST) or p travels
  ++D.tag;
  const Publisher pub1(D);
#pragma unroll
  for (int j = RPT - 1; j >= 0; --j) {
    const int32_t i = t + j * kThreads;
    if (i < mine) {
      const double bi = a.b[D.r0 + i];
      r[j] = bi - q[j];
      const double z = (kStream ? dinv[i] : di[kStream ? 0 : j]) * r[j];
      lp[H + i] = z;
      pub1(w0 + j * kThreads, i, kGhost ? r[j] : z);
      bb += bi * bi;
      rr += r[j] * r[j];
      rz += r[j] * z;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  int iter = 0, converged = 0;
  bool run = true, ok;
  double thr, rr_out;
  {
    double s[2] = {bb, rr};
    ok = team_sum(tm, sh, s, [&] {
      if constexpr (kGhost) {
        D.template fetch<false>(gr, kIdle, &sh.bad);
        D.template fetch<true>(gr + H, kIdle, &sh.bad);
      }
    });
    bb = s[0];
    rr_out = s[1];
    thr = a.tol2 * bb;
    thr = thr > 2.2250738585072014e-308 ? thr : 2.2250738585072014e-308;
    if (bb == 0.0 || s[1] < thr) {
      converged = 1;
      run = false;
    } else if (a.maxit <= 0) {
      run = false;
    }
  }
  if constexpr (kGhost) {
    for (int32_t h = t; h < 2 * H; h += kThreads) lp[h < H ? h : D.rows + h] = gd[h] * gr[h];
  }
  for (int k = 0; run && ok; ++k) {
    double s[5] = {0.0, 0.0, 0.0, rr, rz};
    if constexpr (KIND == HALO) {
      D.template fetch<false>(lp, 0, &sh.bad);
      D.template fetch<true>(up, 0, &sh.bad);
    }
    if constexpr (kGhost) ++D.tag;
    if constexpr (!kStream) __syncthreads();
    {
      const int32_t wi = opaque_uniform(w0);
      const int32_t tp = opaque(t);
      const Publisher pub(D);
      sweep([&](int j, double pi, double dv) {
        if constexpr (kGhost) pub(wi + j * kThreads, tp + j * kThreads, q[j]);
        const double dq = dv * q[j];
        s[0] = __builtin_fma(pi, q[j], s[0]);
        s[1] = __builtin_fma(dq, r[j], s[1]);
        s[2] = __builtin_fma(dq, q[j], s[2]);
        pin(s[0]), pin(s[1]), pin(s[2]);
      });
    }
    ok = team_sum(tm, sh, s, [&] {
      if constexpr (kGhost) {
        D.template fetch<false>(gq, kIdle, &sh.bad);
        D.template fetch<true>(gq + H, kIdle, &sh.bad);
      }
    });
    if (!ok) break;
    rr_out = s[3];
    if (s[3] < thr) {
      converged = 1;
      iter = k > 0 ? k - 1 : 0;
      break;
    }
    iter = k;
    if (k >= a.maxit) break;
    const double rho = s[4], alpha = rho / s[0];
    const double rho_next = rho - 2.0 * alpha * s[1] + alpha * alpha * s[2];
    const double beta = rho_next / rho;
    rr = rz = 0.0;
    if constexpr (!kGhost) ++D.tag;
    const Publisher pub(D);
    const int32_t ti = opaque(t), wi = opaque_uniform(w0);
    double *lc = lp + H + ti;
    // the next row's streamed values
    double nd = 0.0, nx = 0.0;
    auto load_update = [&](int j) {
      const uint32_t at = (uint32_t)min(ti + j * kThreads, mine - 1) * 8u;
      if constexpr (kStream) nd = load_at(dinv, at);
      if (j >= XR) nx = load_at(xg, at);
    };
    load_update(RPT - 1);
#pragma unroll
    for (int j = RPT - 1; j >= 0; --j) {
      const int32_t i = ti + j * kThreads;
      const double dv = kStream ? nd : di[kStream ? 0 : j];
      const double xi = j < XR ? x[j < XR ? j : 0] : nx;
      if (j > 0) load_update(j - 1);
      // (the rows past the end: q, r and their sums stay zero; what they
      // read of p is finite where the solve is)
      const double pi = lc[j * kThreads];
      const double xn = __builtin_fma(alpha, pi, xi);
      if (j < XR) x[j < XR ? j : 0] = xn;
      r[j] = __builtin_fma(-alpha, q[j], r[j]);
      const double z = dv * r[j];
      const double p = __builtin_fma(beta, pi, z);
      rr = __builtin_fma(r[j], r[j], rr);
      rz = __builtin_fma(r[j], z, rz);
      if (i < mine) {
        lc[j * kThreads] = p;
        if (j >= XR) xg[i] = xn;
      }
      if constexpr (!kGhost) pub(wi + j * kThreads, i, p);
      pin(r[j]), pin(rr), pin(rz);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (kGhost) {
      for (int32_t h = t; h < 2 * H; h += kThreads) {
        const double rn = __builtin_fma(-alpha, gq[h], gr[h]);
        gr[h] = rn;
        const int32_t at = h < H ? h : D.rows + h;
        lp[at] = __builtin_fma(beta, lp[at], gd[h] * rn);
      }
    }
  }
  if (ok) {
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      const int32_t i = t + j * kThreads;
      if (i < mine) {
        if (bb == 0.0) xg[i] = 0.0;
        else if (j < XR) xg[i] = x[j < XR ? j : 0];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (D.rank == 0 && t == 0) {
    a.st->rr = rr_out;
    a.st->bb = bb;
    a.st->iter = iter;
    a.st->converged = converged;
    a.st->refinements = 0;
    a.st->aborted = ok ? 0 : 1;
  }
}

__global__ void k_zero_words(word_t *p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0;
}

constexpr size_t kPartWords = (size_t)2 * 2 * kSums * kMaxTeam;
constexpr size_t kTotalWords = (size_t)2 * kLeaders * 2 * kSums;
constexpr size_t kLdsBytes = 160 * 1024;
// LDS of the team sums, rounded up (static, beside the dynamic lp array)
constexpr size_t kLdsStatic = (sizeof(SumLds) + 1023) / 1024 * 1024;

typedef void (*DiaKernel)(DiaArgs);
struct DiaVariant {
  int kind, rpt;
  DiaKernel fn;
};

// In order of preference: the smallest number of rows per thread with which
// the team and its LDS fit.
const DiaVariant kDiaVariants[] = {
    {GHOST, 1, k_res_dia<GHOST, 1, 1>},   {GHOST, 3, k_res_dia<GHOST, 3, 3>},
    {GHOST, 5, k_res_dia<GHOST, 5, 5>},   {GHOST, 7, k_res_dia<GHOST, 7, 7>},
    {GHOST, 9, k_res_dia<GHOST, 9, 9>},   {HALO, 9, k_res_dia<HALO, 9, 9>},
    {STREAM, 17, k_res_dia<STREAM, 17, 17>},
    {STREAM, 25, k_res_dia<STREAM, 25, 17>},
    {STREAM, 33, k_res_dia<STREAM, 33, 8>},
};

}  // namespace

namespace lfgpu {

void resident_free(ResidentBufs *b) {
  dfree(b->halo);
  dfree(b->sums);
  dfree(b->state);
  *b = ResidentBufs{};
}

int resident_pcg_dia(lfgpu_ctx *ctx, ResidentBufs *bufs, const ResidentDia &A, const double *b,
                     double *x, double rtol, int maxit, ResidentState *st, bool *taken) {
  *taken = false;
  if (A.n <= 0 || A.ndiag > ND) return LFGPU_OK;
  int32_t H = 0;
  for (int d = 0; d < A.ndiag; ++d) H = std::max(H, std::abs(A.off[d]));
  const int cus = std::min(ctx->cus, kMaxTeam);
  const DiaVariant *pick = nullptr;
  int team = 0;
  int32_t rows = 0;
  size_t lds = 0;  // in doubles
  for (const DiaVariant &v : kDiaVariants) {
    if (v.kind == STREAM && !(A.sym && A.ndiag == ND)) continue;
    const int64_t cap = (int64_t)v.rpt * kThreads;
    team = (int)((A.n + cap - 1) / cap);
    if (team > cus) continue;
    // rows in 128-byte steps, evenly over the team
    rows = (int32_t)(((A.n + team - 1) / team + 15) / 16 * 16);
    rows = (int32_t)std::min<int64_t>(rows, cap);
    team = (int)((A.n + rows - 1) / rows);
    if (team > 1 && H > rows) continue;
    // STREAM: the first half's rows must not read the upper halo nor the
    // second half's the lower one (they share their place)
    const int32_t half = (v.rpt + 1) / 2 * kThreads;
    if (v.kind == STREAM && (half < H || half > rows - H)) continue;
    // p with both halos (STREAM: one) and, for GHOST, three more halo arrays;
    // the rows up to rpt * 512 are read
    lds = (size_t)cap + (v.kind == GHOST ? 8 : v.kind == HALO ? 2 : 1) * (size_t)H;
    if (lds * sizeof(double) + kLdsStatic > kLdsBytes) continue;
    pick = &v;
    break;
  }
  if (!pick) return LFGPU_OK;
  const int32_t slots = std::min(rows, 2 * H);
  const size_t words = (size_t)2 * team * 2 * std::max(slots, 1);
  hipStream_t s = ctx->stream;
  if (!bufs->sums) {
    LFG_TRY(dalloc(&bufs->sums, kPartWords + kTotalWords, "resident PCG sums"));
    LFG_TRY(dalloc(&bufs->state, 2, "resident PCG state"));
    bufs->abort = reinterpret_cast<int *>(bufs->state + 1);
    bufs->epoch = 0xffffffffu;  // forces the clearing below
  }
  if (words > bufs->halo_words) {
    dfree(bufs->halo);
    bufs->halo = nullptr;
    bufs->halo_words = 0;
    LFG_TRY(dalloc(&bufs->halo, words, "resident PCG halo"));
    bufs->halo_words = words;
    bufs->epoch = 0xffffffffu;
  }
  // tags of this solve: one exchange and one sum an iteration and two more
  const uint64_t need = (uint64_t)maxit + 4;
  if (bufs->epoch + need > 0xfffffff0ull) {
    hipLaunchKernelGGL(k_zero_words, dim3(256), dim3(256), 0, s, bufs->halo, bufs->halo_words);
    hipLaunchKernelGGL(k_zero_words, dim3(8), dim3(256), 0, s, bufs->sums,
                       kPartWords + kTotalWords);
    hipLaunchKernelGGL(k_zero_words, dim3(1), dim3(64), 0, s,
                       reinterpret_cast<word_t *>(bufs->state),
                       2 * sizeof(ResidentState) / sizeof(word_t));
    LFG_HIP(hipGetLastError());
    bufs->epoch = 0;
  }
  DiaArgs a{};
  a.n = A.n;
  a.rows = rows;
  a.halo = H;
  a.slots = std::max(slots, 1);
  a.lds = (int32_t)lds;
  lds *= sizeof(double);
  a.ndiag = A.ndiag;
  for (int d = 0; d < kMaxD; ++d) a.off[d] = d < A.ndiag ? A.off[d] : 0;
  a.val = A.val;
  a.rowsum = A.rowsum;
  a.dinv = A.dinv;
  a.b = b;
  a.x = x;
  a.halo_words = bufs->halo;
  a.part = bufs->sums;
  a.total = bufs->sums + kPartWords;
  a.abort = bufs->abort;
  a.tag0 = bufs->epoch;
  a.tol2 = rtol * rtol;
  a.maxit = maxit;
  a.st = bufs->state;
  const void *fn = reinterpret_cast<const void *>(pick->fn);
  LFG_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  void *args[] = {&a};
  if (team == 1) {
    LFG_HIP(hipLaunchKernel(fn, dim3(1), dim3(kThreads), args, lds, s));
  } else {
    // all workgroups of the team must run at once
    const hipError_t e = hipLaunchCooperativeKernel(fn, dim3(team), dim3(kThreads), args,
                                                    (unsigned)lds, s);
    if (e == hipErrorCooperativeLaunchTooLarge) {
      (void)hipGetLastError();
      return LFGPU_OK;
    }
    LFG_HIP(e);
  }
  bufs->epoch += (uint32_t)need;
  LFG_HIP(hipMemcpyAsync(st, bufs->state, sizeof(ResidentState), hipMemcpyDeviceToHost, s));
  *taken = true;
  return LFGPU_OK;
}

}  // namespace lfgpu
