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
// sweeps against this, in us:
//              64^2   512^2   1023x770   1024^2   2048x256   1400^2   2048^2
//   FP64     12.6/2.4 17.6/3.4 29.8/4.8 32.0/6.3  20.8/4.0 55.1/14.4  101/37
//   FP32     15.2/3.4 14.4/3.9 19.6/5.2 21.8/5.9  17.0/4.6 31.6/13.8 57.6/26
//   FP32 mat 17.4/3.5 16.7/4.1 24.3/5.2 30.5/6.4  21.1/4.5 46.6/13.2 85.3/47
//
// One iteration (the recurrences and the stopping test of the two-sweep
// solver, with one team sum instead of two):
//   q = A p; team sum of p.q, (q, D^-1 r), (q, D^-1 q) and of ||r||^2 and
//   (r, D^-1 r) left by the previous update; stop if ||r||^2 < thr;
//   alpha = rho / p.q, beta from rho' = rho - 2 alpha (q, D^-1 r) +
//   alpha^2 (q, D^-1 q); x += alpha p, r -= alpha q, p = D^-1 r + beta p.
// The product that runs beside the stopping test of the last iteration is
// discarded, x is what the test was made on.
//
// The matrix lives on a lattice: S rows a line, L lines, every off-diagonal
// couples a row to one of its eight lattice neighbours (the P1 matrix of a
// structured mesh).  A workgroup owns a tile of the lattice.  Runs of
// consecutive rows would need no lattice, but their halo is two lines a
// workgroup: at 2048 x 256 (2560 rows and 4100 halo values a workgroup)
// exchanging them took half of an iteration (11.5 us).
#include <hip/hip_bf16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <vector>

#include "lfgpu_reduce.h"
#include "lfgpu_resident.h"
#include "lfgpu_resident_device.h"

using namespace lfgpu;
using namespace lfgpu::res;

namespace {

constexpr int ND = 6;  // off-diagonals of a P1 matrix on a structured mesh

// One problem of a batch: its lattice, tiles and place in the buffers.
struct TileJob {
  int32_t index, lo;  // problem number, first row
  int32_t S, L, TW, TH, TX, team, slots, ghosts, ndiag;
  int32_t off[ND], shift[ND];
  uint64_t halo_at, sums_at;  // words
};

struct TileArgs {
  int32_t n;            // rows of the storage (a diagonal's stride)
  int32_t S, L;         // lattice: rows a line, lines
  int32_t TW, TH, TX;   // tile width and height, tiles a line
  int32_t slots;        // values a workgroup publishes, 2 (TW + TH)
  int32_t ghosts;       // most halo cells of a workgroup
  int ndiag;
  int32_t off[ND];      // row offset of diagonal d
  int32_t shift[ND];    // its offset in the padded tile
  const double *__restrict__ val;
  const double *__restrict__ rowsum;
  const double *__restrict__ dinv;
  const double *__restrict__ b;
  double *x;
  word_t *halo_words;  // [2][team][2][slots]
  word_t *part, *total;
  ResidentAbort *abort;
  uint32_t tag0;
  double tol2;
  int maxit;
  ResidentState *st;
  // mixed modes
  const float *__restrict__ val32;
  const float *__restrict__ rowsum32;
  const float *__restrict__ dinv32;
  const __hip_bfloat16 *__restrict__ dinv16;
  double *xlo;
  double delta2;
  int max_interval;
  // batches: the jobs, each slot's job and rank in its team, and the counter
  // that hands out the slots
  const TileJob *__restrict__ jobs;
  const int2 *__restrict__ job_slots;
  int nslots;
  int *ticket, *running, *arrived;
};

// The workgroup's tile: tw x th cells of the lattice, padded by one halo cell
// on each side to lines of P = TW + 2 cells.  Cell i = line * P + c (c = 0 and
// c > tw are halo cells) is thread i % 512's cell number i / 512; it sits in
// an LDS array at P + 1 + i, so that every neighbour is at a fixed distance.
struct Tile {
  int32_t S, P, tw, th, x0, y0, n, g0;
  int32_t rank, team, TW, TH, TX, L, slots;
  word_t *words;
  ResidentAbort *abort;
  uint32_t tag;
  int32_t *gpos, *gsrc, *ppos;  // LDS tables of the exchange
  int32_t ng, np;

  __device__ __forceinline__ Tile(const TileArgs &a, int32_t rank_, int32_t team_)
      : S(a.S), P(a.TW + 2), n(a.n), rank(rank_), team(team_), TW(a.TW), TH(a.TH), TX(a.TX),
        L(a.L), slots(a.slots), words(a.halo_words), abort(a.abort), tag(a.tag0) {
    x0 = rank % TX * TW;
    y0 = rank / TX * TH;
    tw = min(TW, S - x0);
    th = min(TH, L - y0);
    g0 = y0 * S + x0;
    ng = 2 * (tw + 2) + 2 * th;
    np = team > 1 ? slots : 0;
    gpos = gsrc = ppos = nullptr;
  }

  // Walks this thread's cells in order: column c and row g of cell number j.
  struct Walk {
    int32_t c, g, line;
  };
  __device__ __forceinline__ Walk first(int32_t t) const {
    Walk w;
    w.line = t / P;
    w.c = t - w.line * P;
    w.g = g0 + w.line * S + w.c - 1;
    return w;
  }
  __device__ __forceinline__ void next(Walk &w) const {
    const int32_t lines = kThreads / P, cols = kThreads - lines * P;  // uniform
    w.c += cols;
    w.g += lines * S + cols;
    w.line += lines;
    if (w.c >= P) {
      w.c -= P;
      w.g += S - P;
      w.line += 1;
    }
  }
  __device__ __forceinline__ bool alive(const Walk &w) const {
    return w.line < th && w.c >= 1 && w.c <= tw;
  }

  // Halo cell h: its place in an LDS array and the word its owner publishes
  // it in (-1: outside the lattice).  Every workgroup publishes the cells of
  // its tile's rim: top line, bottom line, left and right column; a cell on
  // two of them is read from the first.
  __device__ void tables(int32_t t) {
    for (int32_t h = t; h < ng; h += kThreads) {
      int32_t line, c;
      if (h < 2 * (tw + 2)) {
        line = h < tw + 2 ? -1 : th;
        c = h < tw + 2 ? h : h - (tw + 2);
      } else {
        const int32_t k = h - 2 * (tw + 2);
        line = k < th ? k : k - th;
        c = k < th ? 0 : tw + 1;
      }
      gpos[h] = P + 1 + line * P + c;
      const int32_t gx = x0 + c - 1, gy = y0 + line;
      int32_t src = -1;
      if (gx >= 0 && gx < S && gy >= 0 && gy < L) {
        const int32_t ox = gx / TW, oy = gy / TH, lx = gx - ox * TW, ly = gy - oy * TH;
        const int32_t oth = min(TH, L - oy * TH);
        const int32_t s = ly == 0 ? lx : ly == oth - 1 ? TW + lx
                          : lx == 0 ? 2 * TW + ly : 2 * TW + TH + ly;
        src = (oy * TX + ox) * 2 * slots + s;
      }
      gsrc[h] = src;
    }
    for (int32_t s = t; s < slots; s += kThreads) {
      int32_t line, lx;
      if (s < 2 * TW) {
        line = s < TW ? 0 : th - 1;
        lx = s < TW ? s : s - TW;
      } else {
        const int32_t k = s - 2 * TW;
        line = k < TH ? k : k - TH;
        lx = k < TH ? 0 : tw - 1;
      }
      ppos[s] = lx < tw && line < th ? P + 1 + line * P + lx + 1 : -1;
    }
  }

  // Publishes the rim cells of src (indexed like an LDS array of the tile),
  // with the threads from `first` on.
  template <class VT, class A>
  __device__ __forceinline__ void publish(const A *src, int first) const {
    if ((int)threadIdx.x < first) return;
    word_t *w = words + ((size_t)(tag & 1u) * team + rank) * 2 * slots;
    for (int32_t s = (int32_t)threadIdx.x - first; s < np; s += kThreads - first) {
      const int32_t at = ppos[s];
      if (at < 0) continue;
      if constexpr (sizeof(VT) == 8) {
        const double v = (double)src[at];
        put(&w[s], low_word(v, tag));
        put(&w[slots + s], high_word(v, tag));
      } else {
        put(&w[s], ((word_t)__float_as_uint((float)src[at]) << 32) | tag);
      }
    }
  }
  // The same from an array with a value for every slot.
  template <class VT>
  __device__ __forceinline__ void publish_slots(const VT *src, int first) const {
    static_assert(sizeof(VT) == 8, "two words a value");
    if ((int)threadIdx.x < first) return;
    word_t *w = words + ((size_t)(tag & 1u) * team + rank) * 2 * slots;
    for (int32_t s = (int32_t)threadIdx.x - first; s < np; s += kThreads - first) {
      put(&w[s], low_word(src[s], tag));
      put(&w[slots + s], high_word(src[s], tag));
    }
  }
  // Waits for the halo cells and hands (h, place, value) to fn, two cells per
  // thread in flight, with the threads from `first` on.
  template <class VT, class F>
  __device__ __forceinline__ void fetch(int first, int *bad, F &&fn) const {
    if (team == 1 || (int)threadIdx.x < first) return;
    const word_t *w = words + (size_t)(tag & 1u) * team * 2 * slots;
    const int32_t step = kThreads - first;
    for (int32_t h0 = (int32_t)threadIdx.x - first; h0 < ng; h0 += 2 * step) {
      int32_t src[2];
      word_t lo[2], hi[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) src[u] = h0 + u * step < ng ? gsrc[h0 + u * step] : -1;
      bool ok;
      Wait wait(abort);
      do {
        ok = true;
#pragma unroll
        for (int u = 0; u < 2; ++u)
          if (src[u] >= 0) {
            lo[u] = get(&w[src[u]]);
            if constexpr (sizeof(VT) == 8) hi[u] = get(&w[src[u] + slots]);
          }
#pragma unroll
        for (int u = 0; u < 2; ++u)
          if (src[u] >= 0) {
            ok = ok && tagged(lo[u], tag);
            if constexpr (sizeof(VT) == 8) ok = ok && tagged(hi[u], tag);
          }
      } while (!ok && wait.more());
      if (!ok) *bad = 1;
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (src[u] >= 0) {
          VT v;
          if constexpr (sizeof(VT) == 8) v = from_words(lo[u], hi[u]);
          else v = __uint_as_float((uint32_t)(lo[u] >> 32));
          fn(h0 + u * step, gpos[h0 + u * step], v);
        }
    }
  }
  // The halo of an LDS array whose values are VTs, from the neighbours' rims;
  // a workgroup barrier has to precede it and to follow it.
  template <class VT, class A>
  __device__ __forceinline__ void exchange(A *arr, int *bad) {
    ++tag;
    publish<VT>(arr, 0);
    fetch<VT>(0, bad, [&](int32_t, int32_t at, VT v) { arr[at] = (A)v; });
  }
};

// How a variant keeps the matrix and the halo.
//   GHOST: the matrix stays in registers.  The halo cells' r, q, D^-1 and p
//     are kept here as well and updated by the same operations as their
//     owners', so that what travels is q: it is published beside the partial
//     sums and arrives while the team sum runs, which takes the exchange off
//     the iteration's critical path.
//   STREAM: the matrix (its upper half: symmetric values) is read from memory
//     every iteration, the next rows' loads in flight while a row is worked
//     on; in the mixed modes p travels between the update and the next product.
enum { GHOST, STREAM };

// From this many cells a thread the GHOST variants keep row sums and D^-1 in
// LDS (9 cells' r, q, x and six diagonals take 162 of the 256 registers; with
// the two others in registers too 1024^2 spilled and took 11.7 us an iteration
// instead of 8.2).
constexpr int kLdsDiag = 7;

// LDS: p (FP64 in every mode: converting the neighbours' values of an FP32 p
// in every product costs more than the bytes), q (GHOST) and the exchange's
// tables.
template <int KIND, class VT, int RPT>
struct TileLds {
  static constexpr bool kDiag = KIND == GHOST && RPT >= kLdsDiag;
  double *lp;           // padded tile of p (and of the vectors of a reliable update)
  double *rs, *di;      // kDiag: row sums and D^-1 of cell j of thread t at t + 512 j
  VT *lq, *gr, *gq, *gd;
  __device__ __forceinline__ TileLds(double *base, const TileArgs &a, Tile &T) {
    const int32_t n = cells(a.TW);
    lp = base;
    base += n;
    rs = di = nullptr;
    if (kDiag) {
      rs = base;
      di = rs + RPT * kThreads;
      base = di + RPT * kThreads;
    }
    VT *v = reinterpret_cast<VT *>(base);
    lq = v;
    gr = gq = gd = nullptr;
    if (KIND == GHOST) {
      gr = v + n;
      gq = gr + a.ghosts;
      gd = gq + a.ghosts;
      v = gd + a.ghosts;
    }
    T.gpos = reinterpret_cast<int32_t *>(v);
    T.gsrc = T.gpos + a.ghosts;
    T.ppos = T.gsrc + a.ghosts;
  }
  // cells of one padded array: what any cell number's neighbours reach
  static __host__ __device__ int32_t cells(int32_t TW) {
    return (kThreads * RPT + 2 * (TW + 3) + 1) / 2 * 2;
  }
  static size_t bytes(const TileArgs &a) {
    const size_t n = (size_t)cells(a.TW);
    return n * 8 + (kDiag ? 2 * (size_t)RPT * kThreads * 8 : 0) +
           (KIND == GHOST ? (n + 3 * (size_t)a.ghosts) * sizeof(VT) : 0) +
           4 * (2 * (size_t)a.ghosts + a.slots) + 16;
  }
};

// GHOST in FP64.  RPT: cells per thread.
template <int RPT, bool BATCH>
__device__ __forceinline__ bool tile_solve(const TileArgs &a, int rank, int team, double *dyn,
                                           SumLds &sh) {
  const int t = threadIdx.x;
  Tile T(a, rank, team);
  typedef TileLds<GHOST, double, RPT> Lds;
  const Lds M(dyn, a, T);
  constexpr bool kRegDiag = !Lds::kDiag;
  double *const lp = M.lp;
  // (a batch's smaller tiles leave the last cell numbers empty)
  const int nj = BATCH ? (T.th * T.P + kThreads - 1) / kThreads : RPT;
  Team tm{T.rank, T.team, a.part, a.total, a.abort, a.tag0};
  if (t == 0) sh.bad = 0;
  // Moves the loops by 48 B.  The kernel of one cell a thread waits in short
  // poll loops most of the time, and the same code takes 2.30 us an iteration on
  // 65 x 65 rows this way, 2.52 without, 2.58 with all loops on 32 or 64 B.  Why
  // is not established (the loops' place in the instruction cache, or the phase
  // in which their polls meet the words); to be measured again when that kernel's
  // code changes.
  if constexpr (RPT == 1 && !BATCH) asm volatile(".rept 12\n s_nop 0\n .endr");
  T.tables(t);
  const int32_t cells = Lds::cells(a.TW);
  for (int32_t i = t; i < cells; i += kThreads) lp[i] = 0.0;
  for (int32_t h = t; h < T.ng; h += kThreads) M.gr[h] = M.gq[h] = M.gd[h] = 0.0;
  const int32_t at0 = T.P + 1 + t;  // LDS place of the thread's first cell

  double x[RPT], r[RPT], q[RPT];
  double v[RPT][ND], rs[kRegDiag ? RPT : 1], di[kRegDiag ? RPT : 1];
  uint64_t live = 0;  // the thread's cells that are rows of the tile
  __syncthreads();
  {
    Tile::Walk w = T.first(t);
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      r[j] = q[j] = x[j] = 0.0;
      if constexpr (kRegDiag) rs[j] = di[j] = 0.0;
      else M.rs[t + j * kThreads] = M.di[t + j * kThreads] = 0.0;
#pragma unroll
      for (int d = 0; d < ND; ++d) v[j][d] = 0.0;
      if (T.alive(w)) {
        live |= 1ull << j;
        x[j] = a.x[w.g];
        lp[at0 + j * kThreads] = x[j];
        if constexpr (kRegDiag) {
          rs[j] = a.rowsum[w.g];
          di[j] = a.dinv[w.g];
        } else {
          M.rs[t + j * kThreads] = a.rowsum[w.g];
          M.di[t + j * kThreads] = a.dinv[w.g];
        }
#pragma unroll
        for (int d = 0; d < ND; ++d)
          if (d < a.ndiag) v[j][d] = a.val[(int64_t)d * a.n + w.g];
      }
      T.next(w);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();
  T.template exchange<double>(lp, &sh.bad);
  __syncthreads();

  // q_j = (A p)_i in difference form from LDS, handed to fn with p_i and
  // D^-1_i; cells that are no rows give q = 0
  auto sweep = [&](auto &&fn) {
    const double *lc = lp + opaque(at0);
    const double *bp[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) bp[d] = lc + a.shift[d];
    const double *lrs = M.rs + opaque(t), *ldi = M.di + opaque(t);
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      if (BATCH && j >= nj) break;
      // every LDS read of the row before the first use
      const double pi = lc[j * kThreads];
      double c[ND], acc = 0.0;
#pragma unroll
      for (int d = 0; d < ND; ++d) c[d] = bp[d][j * kThreads];
      const double s = kRegDiag ? rs[kRegDiag ? j : 0] : lrs[j * kThreads];
      const double dv = kRegDiag ? di[kRegDiag ? j : 0] : ldi[j * kThreads];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int d = 0; d < ND; ++d) acc = __builtin_fma(v[j][d], c[d] - pi, acc);
      q[j] = __builtin_fma(s, pi, acc);
      pin(q[j]);
      fn(j, pi, dv);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  double rr = 0.0, rz = 0.0, bb = 0.0;
  sweep([&](int, double, double) {});
  __syncthreads();
  // r = b - A x, p = D^-1 r
  {
    Tile::Walk w = T.first(opaque(t));
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      if ((live >> j) & 1) {
        const double bi = a.b[w.g];
        r[j] = bi - q[j];
        const double z = (kRegDiag ? di[kRegDiag ? j : 0] : M.di[t + j * kThreads]) * r[j];
        lp[at0 + j * kThreads] = z;
        M.lq[at0 + j * kThreads] = r[j];
        bb = __builtin_fma(bi, bi, bb);
        rr = __builtin_fma(r[j], r[j], rr);
        rz = __builtin_fma(r[j], z, rz);
      }
      T.next(w);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // the halo cells' r, D^-1 and p = D^-1 r
  __syncthreads();
  ++T.tag;
  T.template publish<double>(M.lq, 0);
  T.template fetch<double>(0, &sh.bad, [&](int32_t h, int32_t at, double rv) {
    const int32_t cell = at - T.P - 1 + T.P;  // from the line above the tile
    const int32_t line = cell / T.P - 1, c = cell - (line + 1) * T.P;
    const double d = a.dinv[T.g0 + line * T.S + c - 1];
    M.gr[h] = rv;
    M.gd[h] = d;
    lp[at] = d * rv;
  });
  int iter = 0, converged = 0;
  bool run = true, ok;
  double thr, rr_out;
  {
    double s[2] = {bb, rr};
    ok = team_sum(tm, sh, s, [] {});
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
  for (int k = 0; run && ok; ++k) {
    double s[5] = {0.0, 0.0, 0.0, rr, rz};
    __syncthreads();
    double *lqc = M.lq + opaque(at0);
    sweep([&](int j, double pi, double dv) {
      lqc[j * kThreads] = q[j];
      const double dq = dv * q[j];
      s[0] = __builtin_fma(pi, q[j], s[0]);
      s[1] = __builtin_fma(dq, r[j], s[1]);
      s[2] = __builtin_fma(dq, q[j], s[2]);
      pin(s[0]), pin(s[1]), pin(s[2]);
    });
    ++T.tag;
    ok = team_sum(tm, sh, s, [&] {
      const int first = sums_threads(tm);
      T.template publish<double>(M.lq, first);
      T.template fetch<double>(first, &sh.bad,
                               [&](int32_t h, int32_t, double qv) { M.gq[h] = qv; });
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
    double *lc = lp + opaque(at0);
    const double *ldi = M.di + opaque(t);
    double np = lc[0];
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      if (BATCH && j >= nj) break;
      const double dv = kRegDiag ? di[kRegDiag ? j : 0] : ldi[j * kThreads];
      const double pi = np;
      if (j + 1 < RPT) np = lc[(j + 1) * kThreads];
      // (cells that are no rows: r, q and so their sums stay zero)
      x[j] = __builtin_fma(alpha, pi, x[j]);
      r[j] = __builtin_fma(-alpha, q[j], r[j]);
      const double z = dv * r[j];
      const double p = __builtin_fma(beta, pi, z);
      rr = __builtin_fma(r[j], r[j], rr);
      rz = __builtin_fma(r[j], z, rz);
      if ((live >> j) & 1) lc[j * kThreads] = p;
      pin(r[j]), pin(rr), pin(rz);
      __builtin_amdgcn_sched_barrier(0);
    }
    for (int32_t h = t; h < T.ng; h += kThreads) {
      const int32_t at = T.gpos[h];
      const double rn = __builtin_fma(-alpha, M.gq[h], M.gr[h]);
      M.gr[h] = rn;
      lp[at] = __builtin_fma(beta, lp[at], M.gd[h] * rn);
    }
  }
  if (ok) {
    Tile::Walk w = T.first(opaque(t));
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      if ((live >> j) & 1) a.x[w.g] = bb == 0.0 ? 0.0 : x[j];
      T.next(w);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (T.rank == 0 && t == 0) {
    a.st->rr = rr_out;
    a.st->bb = bb;
    a.st->iter = iter;
    a.st->converged = converged;
    a.st->refinements = 0;
    a.st->aborted = ok ? 0 : 1;
  }
  return ok;
}

template <int RPT>
__global__ __launch_bounds__(kThreads) void k_res_tile(TileArgs a) {
  extern __shared__ double dyn[];
  __shared__ SumLds sh;
  (void)tile_solve<RPT, false>(a, blockIdx.x, gridDim.x, dyn, sh);
}

// The streamed solve in FP64.  What bounds it is the matrix's trip through the
// chip's caches every iteration, so that it reads as little as it can: the
// three upper diagonals and the row sums (32 B a row), from which the lower
// ones (symmetric values), the diagonal (row sum minus the others) and D^-1
// follow.  z = D^-1 r and D^-1 q take the places of r and q, so that the update
// needs no D^-1: z -= alpha D^-1 q, p = z + beta p; r = D z is formed in the
// next product, for its sums.  D^-1 q travels during the team sum as GHOST's q
// does, from an LDS array of the rim.  Against 64 B a row and an exchange of p between update and product:
// 1400^2 20.0 -> 14.4, 2048^2 43.3 -> 36.6 us an iteration
// (18 of them the matrix, 9 the trips of x).  One row of the stream in flight
// a thread: two take 36.7, three spill.
//
// 1 / d to rounding, by Newton's iteration
__device__ __forceinline__ double reciprocal(double d) {
  double y = __builtin_amdgcn_rcp(d);
  y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
  return __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
}

template <int RPT>
struct StreamLds {
  double *lp;         // padded tile of p
  double *rim;        // D^-1 q of the rim, by slot, and 64 places for the other cells'
  double *gz, *gdq;   // the halo cells' z and D^-1 q
  __device__ __forceinline__ StreamLds(double *base, const TileArgs &a, Tile &T) {
    lp = base;
    rim = lp + TileLds<STREAM, double, RPT>::cells(a.TW);
    gz = rim + a.slots + 64;
    gdq = gz + a.ghosts;
    T.gpos = reinterpret_cast<int32_t *>(gdq + a.ghosts);
    T.gsrc = T.gpos + a.ghosts;
    T.ppos = T.gsrc + a.ghosts;
  }
  static size_t bytes(const TileArgs &a) {
    return (TileLds<STREAM, double, RPT>::cells(a.TW) + (size_t)a.slots + 64 +
            2 * (size_t)a.ghosts) *
               8 +
           4 * (2 * (size_t)a.ghosts + a.slots) + 16;
  }
};

// RPT: cells per thread.  XR: the cells j < XR keep their x in a register, the
// others' is read and written in every update (as many as the registers hold
// and LDS leave room for: all 17; 16 of 25, with 21 registers spilled; none of
// 33, with 4, since more of them spill more and take longer).  AHEAD: rows of a
// stream in flight.
template <int RPT, int XR, int AHEAD>
__global__ __launch_bounds__(kThreads) void k_res_stream(TileArgs a) {
  extern __shared__ double dyn[];
  __shared__ SumLds sh;
  constexpr int NU = ND / 2;  // upper diagonals: ND / 2.. of a.val
  const int t = threadIdx.x;
  Tile T(a, blockIdx.x, gridDim.x);
  const StreamLds<RPT> M(dyn, a, T);
  double *const lp = M.lp;
  Team tm{T.rank, T.team, a.part, a.total, a.abort, a.tag0};
  if (t == 0) sh.bad = 0;
  T.tables(t);
  const int32_t cells = TileLds<STREAM, double, RPT>::cells(a.TW);
  for (int32_t i = t; i < cells; i += kThreads) lp[i] = 0.0;
  for (int32_t i = t; i < a.slots; i += kThreads) M.rim[i] = 0.0;
  for (int32_t h = t; h < T.ng; h += kThreads) M.gz[h] = M.gdq[h] = 0.0;
  const int32_t at0 = T.P + 1 + t;  // LDS place of the thread's first cell

  double x[XR > 0 ? XR : 1], z[RPT], dq[RPT];
  uint64_t live = 0;  // the thread's cells that are rows of the tile
  __syncthreads();
  {
    Tile::Walk w = T.first(t);
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      z[j] = dq[j] = 0.0;
      if (j < XR) x[j] = 0.0;
      if (T.alive(w)) {
        live |= 1ull << j;
        const double xi = a.x[w.g];
        if (j < XR) x[j] = xi;
        lp[at0 + j * kThreads] = xi;
      }
      T.next(w);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();
  T.template exchange<double>(lp, &sh.bad);
  __syncthreads();

  // the next rows of the stream: the upper diagonals, the lower ones as the
  // mirrored upper ones (before the first row the last row's, which are zero:
  // a value changed after its load would be waited for at once), and the row
  // sum
  double nv[AHEAD][ND], ns[AHEAD];
  Tile::Walk lw;
  auto load_row = [&](int j) {
    const int k = j % AHEAD;
    const int32_t g = (live >> j) & 1 ? lw.g : T.g0;
    const uint32_t at = (uint32_t)g * 8u;
#pragma unroll
    for (int d = 0; d < NU; ++d) {
      const int32_t c = g + a.off[d];
      nv[k][d] = load_at(a.val + (int64_t)(ND - 1 - d) * a.n, (uint32_t)(c < 0 ? a.n - 1 : c) * 8u);
      nv[k][NU + d] = load_at(a.val + (int64_t)(NU + d) * a.n, at);
    }
    ns[k] = load_at(a.rowsum, at);
    T.next(lw);
  };
  auto prefetch = [&] {
    lw = T.first(opaque(t));
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) load_row(j);
  };
  // (A p)_i in difference form from LDS, the diagonal and p_i, handed to fn
  auto sweep = [&](auto &&fn) {
    // (LDS instructions reach 64 KB from a register: new bases every 16 rows)
    const double *lc = lp, *bp[ND];
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      if (j % 16 == 0) {
        lc = lp + opaque(at0 + j * kThreads);
#pragma unroll
        for (int d = 0; d < ND; ++d) bp[d] = lc + a.shift[d];
      }
      const int in = j % 16 * kThreads;
      double vr[ND];
#pragma unroll
      for (int d = 0; d < ND; ++d) vr[d] = nv[j % AHEAD][d];
      const double s = ns[j % AHEAD];
      const double pi = lc[in];
      double c[ND], acc = 0.0, diag = s;
#pragma unroll
      for (int d = 0; d < ND; ++d) c[d] = bp[d][in];
      if (AHEAD == 1 && j + 1 < RPT) load_row(j + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        acc = __builtin_fma(vr[d], c[d] - pi, acc);
        diag -= vr[d];
      }
      fn(j, __builtin_fma(s, pi, acc), diag, pi);
      __builtin_amdgcn_sched_barrier(0);
      if (AHEAD > 1 && j + AHEAD < RPT) load_row(j + AHEAD);
    }
  };

  double rr = 0.0, bb = 0.0;
  prefetch();
  sweep([&](int j, double qi, double, double) {
    dq[j] = (live >> j) & 1 ? qi : 0.0;
    pin(dq[j]);
  });
  __syncthreads();
  // r = b - A x, z = p = D^-1 r
  {
    Tile::Walk w = T.first(opaque(t));
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      if ((live >> j) & 1) {
        const double bi = a.b[w.g];
        const double ri = bi - dq[j];
        z[j] = a.dinv[w.g] * ri;
        lp[at0 + j * kThreads] = z[j];
        bb = __builtin_fma(bi, bi, bb);
        rr = __builtin_fma(ri, ri, rr);
      }
      T.next(w);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();
  ++T.tag;
  T.template publish<double>(lp, 0);
  T.template fetch<double>(0, &sh.bad, [&](int32_t h, int32_t at, double v) {
    M.gz[h] = v;
    lp[at] = v;
  });
  int iter = 0, converged = 0;
  bool run = true, ok;
  double thr, rr_out;
  {
    double s[2] = {bb, rr};
    ok = team_sum(tm, sh, s, [] {});
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
  for (int k = 0; run && ok; ++k) {
    double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    __syncthreads();
    {
      prefetch();
      Tile::Walk w = T.first(opaque(t));
      sweep([&](int j, double qi, double diag, double pi) {
        const bool row = (live >> j) & 1;
        qi = row ? qi : 0.0;
        const double d = row ? reciprocal(diag) * qi : 0.0;
        const double ri = diag * z[j];
        dq[j] = d;
        s[0] = __builtin_fma(pi, qi, s[0]);
        s[1] = __builtin_fma(qi, z[j], s[1]);
        s[2] = __builtin_fma(d, qi, s[2]);
        s[3] = __builtin_fma(ri, ri, s[3]);
        s[4] = __builtin_fma(ri, z[j], s[4]);
        const int32_t lx = w.c - 1;
        const int32_t line = w.line;
        int32_t to = a.slots + (t & 63);  // (no rim: a place that nobody reads)
        to = lx == T.tw - 1 ? 2 * T.TW + T.TH + line : to;
        to = lx == 0 ? 2 * T.TW + line : to;
        to = line == T.th - 1 ? T.TW + lx : to;
        to = line == 0 ? lx : to;
        M.rim[row ? to : a.slots + (t & 63)] = d;
        T.next(w);
        pin(dq[j]), pin(s[0]), pin(s[1]), pin(s[2]), pin(s[3]), pin(s[4]);
      });
    }
    ++T.tag;
    ok = team_sum(tm, sh, s, [&] {
      const int first = sums_threads(tm);
      T.template publish_slots<double>(M.rim, first);
      T.template fetch<double>(first, &sh.bad,
                               [&](int32_t h, int32_t, double v) { M.gdq[h] = v; });
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
    double *lc = lp;
    // the streamed x: kX rows in flight
    constexpr int kX = 4;
    double nx[kX];
    uint32_t nat[kX];
    Tile::Walk w = T.first(opaque(t));
    auto load_x = [&](int j) {
      nat[j % kX] = (uint32_t)((live >> j) & 1 ? w.g : T.g0) * 8u;
      nx[j % kX] = load_at(a.x, nat[j % kX]);
      T.next(w);
    };
    // (streamed cells first: their loads run while the others are updated)
    if constexpr (XR < RPT) {
#pragma unroll
      for (int j = 0; j < XR; ++j) T.next(w);
#pragma unroll
      for (int j = XR; j < XR + kX && j < RPT; ++j) load_x(j);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      if (j % 16 == 0) lc = lp + opaque(at0 + j * kThreads);
      const int in = j % 16 * kThreads;
      const double pi = lc[in];
      if (j < XR) {
        x[j < XR ? j : 0] = __builtin_fma(alpha, pi, x[j < XR ? j : 0]);
      } else {
        const double xn = __builtin_fma(alpha, pi, nx[j % kX]);
        if ((live >> j) & 1)
          *reinterpret_cast<double *>(reinterpret_cast<char *>(a.x) + nat[j % kX]) = xn;
        if (j + kX < RPT) load_x(j + kX);
      }
      // (cells that are no rows: z and D^-1 q stay zero)
      z[j] = __builtin_fma(-alpha, dq[j], z[j]);
      const double p = __builtin_fma(beta, pi, z[j]);
      if ((live >> j) & 1) lc[in] = p;
      pin(z[j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    for (int32_t h = t; h < T.ng; h += kThreads) {
      const int32_t at = T.gpos[h];
      const double zn = __builtin_fma(-alpha, M.gdq[h], M.gz[h]);
      M.gz[h] = zn;
      lp[at] = __builtin_fma(beta, lp[at], zn);
    }
  }
  if (ok) {
    Tile::Walk w = T.first(opaque(t));
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      if ((live >> j) & 1) {
        if (bb == 0.0) a.x[w.g] = 0.0;
        else if (j < XR) a.x[w.g] = x[j < XR ? j : 0];
      }
      T.next(w);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (T.rank == 0 && t == 0) {
    a.st->rr = rr_out;
    a.st->bb = bb;
    a.st->iter = iter;
    a.st->converged = converged;
    a.st->refinements = 0;
    a.st->aborted = ok ? 0 : 1;
  }
}

// A batch: the workgroups take slots (a problem and a rank in its team) from
// a counter, in order.  A problem's slots are consecutive and a team has at
// most as many members as there are workgroups, all of which run, so the
// first unfinished problem always gets its team together.
template <class F>
__device__ __forceinline__ void batch_loop(const TileArgs &base, F &&solve) {
  __shared__ int slot, up;
  if (threadIdx.x == 0) atomicAdd(base.running, 1);
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) slot = atomicAdd(base.ticket, 1);
    __syncthreads();
    const int k = __builtin_amdgcn_readfirstlane(slot);
    if (k >= base.nslots) return;
    const int2 jr = base.job_slots[k];
    // (the job is read after the wait: held across it, the mixed kernels of 7
    // cells a thread spill 82 registers instead of 7, and 64 problems of 32 to
    // 512 lines take 59 ms instead of 46)
    if (!team_assembles(base.arrived + jr.x, base.jobs[jr.x].team, base.running, base.abort, up))
      return;
    const TileJob &jb = base.jobs[jr.x];
    TileArgs a = base;
    a.S = jb.S;
    a.L = jb.L;
    a.TW = jb.TW;
    a.TH = jb.TH;
    a.TX = jb.TX;
    a.slots = jb.slots;
    a.ghosts = jb.ghosts;
    a.ndiag = jb.ndiag;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      a.off[d] = jb.off[d];
      a.shift[d] = jb.shift[d];
    }
    a.val += jb.lo;
    a.rowsum += jb.lo;
    a.dinv += jb.lo;
    a.b += jb.lo;
    a.x += jb.lo;
    a.val32 += jb.lo;
    a.rowsum32 += jb.lo;
    a.dinv32 += jb.lo;
    a.dinv16 += jb.lo;
    a.xlo += jb.lo;
    a.halo_words += jb.halo_at;
    a.part += jb.sums_at;
    a.total = a.part + part_words(jb.team);
    a.st += jb.index;
    if (!solve(a, jr.y, jb.team)) return;
  }
}

template <int RPT>
__global__ __launch_bounds__(kThreads) void k_res_tile_batch(TileArgs base) {
  extern __shared__ double dyn[];
  __shared__ SumLds sh;
  batch_loop(base, [&](const TileArgs &a, int rank, int team) {
    return tile_solve<RPT, true>(a, rank, team, dyn, sh);
  });
}

// ---------------------------------------------------------------------------
// Mixed precision: the reliable-update scheme of k_mx_a / k_mx_b
// (lfgpu_solver.hip).  Matrix values and row sums in FP32, the Krylov vectors
// in VT (float: D^-1 in bfloat16; double: D^-1 in FP32), row sums and dot
// products in FP64.  x (high part) and its low part stay in memory: they are
// touched by the reliable updates only.  A reliable update forms
// b - A x - A (xa + xlo) in FP64 with the FP64 matrix read from memory, the
// two vectors passing through LDS one after the other (p waits in the
// registers of q), folds xa into (x, xlo) by TwoSum and replaces r by the
// true residual, p by p + M (r_true - r).  The first residual b - A x is the
// same code.
// ---------------------------------------------------------------------------
template <class VT>
__device__ __forceinline__ float mixed_dinv(const TileArgs &a, int32_t g) {
  if constexpr (sizeof(VT) == 4) return __bfloat162float(a.dinv16[g]);
  else return a.dinv32[g];
}

template <int KIND, class VT, int RPT, int AHEAD, bool BATCH>
__device__ __forceinline__ bool tile_solve_mixed(const TileArgs &a, int rank, int team,
                                                 double *dyn, SumLds &sh) {
  constexpr bool kStream = KIND == STREAM, kGhost = KIND == GHOST;
  const int t = threadIdx.x;
  Tile T(a, rank, team);
  typedef TileLds<KIND, VT, RPT> Lds;
  const Lds M(dyn, a, T);
  constexpr bool kRegDiag = !kStream && !Lds::kDiag;
  const int nj = BATCH ? (T.th * T.P + kThreads - 1) / kThreads : RPT;
  double *const lp = M.lp;
  Team tm{T.rank, T.team, a.part, a.total, a.abort, a.tag0};
  if (t == 0) sh.bad = 0;
  T.tables(t);
  const int32_t cells = Lds::cells(a.TW);
  for (int32_t i = t; i < cells; i += kThreads) lp[i] = 0.0;
  const int32_t at0 = T.P + 1 + t;

  VT r[RPT], q[RPT], xa[RPT];
  // (the FP32 values, widened once)
  double v[kStream ? 1 : RPT][ND], rs[kRegDiag ? RPT : 1];
  VT di[kRegDiag ? RPT : 1];
  uint64_t live = 0;
  {
    Tile::Walk w = T.first(t);
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      r[j] = q[j] = xa[j] = (VT)0;
      if constexpr (!kStream) {
        if constexpr (kRegDiag) rs[j] = 0.0, di[j] = (VT)0;
        else M.rs[t + j * kThreads] = M.di[t + j * kThreads] = 0.0;
#pragma unroll
        for (int d = 0; d < ND; ++d) v[j][d] = 0.0;
      }
      if (T.alive(w)) {
        live |= 1ull << j;
        a.xlo[w.g] = 0.0;
        if constexpr (!kStream) {
          if constexpr (kRegDiag) {
            rs[j] = a.rowsum32[w.g];
            di[j] = mixed_dinv<VT>(a, w.g);
          } else {
            M.rs[t + j * kThreads] = a.rowsum32[w.g];
            M.di[t + j * kThreads] = mixed_dinv<VT>(a, w.g);
          }
#pragma unroll
          for (int d = 0; d < ND; ++d)
            if (d < a.ndiag) v[j][d] = a.val32[(int64_t)d * a.n + w.g];
        }
      }
      T.next(w);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if constexpr (kGhost)
    for (int32_t h = t; h < T.ng; h += kThreads) M.gr[h] = M.gq[h] = M.gd[h] = (VT)0;

  // q = A32 p, each row's q, p and D^-1 handed to fn
  auto sweep = [&](auto &&fn) {
    const double *lc = lp + opaque(at0);
    const double *bp[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) bp[d] = lc + a.shift[d];
    const double *lrs = M.rs + opaque(t), *ldi = M.di + opaque(t);
    float nv[AHEAD][ND], ns[AHEAD], nd[AHEAD];  // the next rows of a stream
    Tile::Walk w = T.first(opaque(t));
    auto load_row = [&](int j) {
      const int k = j % AHEAD;
      const int32_t g = (live >> j) & 1 ? w.g : T.g0;
      const uint32_t at = (uint32_t)g * 4u;
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        // (before the first row the last row's upper values, which are zero: a
        // value changed after its load would be waited for at once)
        const int32_t c = g + a.off[d];
        if (d < ND / 2)
          nv[k][d] = load_at(a.val32 + (int64_t)(ND - 1 - d) * a.n,
                             (uint32_t)(c < 0 ? a.n - 1 : c) * 4u);
        else
          nv[k][d] = load_at(a.val32 + (int64_t)d * a.n, at);
      }
      ns[k] = load_at(a.rowsum32, at);
      nd[k] = mixed_dinv<VT>(a, g);
      T.next(w);
    };
    if constexpr (kStream)
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) load_row(j);
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      if (BATCH && j >= nj) break;
      const int k = j % AHEAD;
      double vr[ND];
#pragma unroll
      for (int d = 0; d < ND; ++d) vr[d] = kStream ? (double)nv[k][d] : v[kStream ? 0 : j][d];
      const double pi = lc[j * kThreads];
      double c[ND], acc = 0.0;
#pragma unroll
      for (int d = 0; d < ND; ++d) c[d] = bp[d][j * kThreads];
      const double s = kRegDiag ? rs[kRegDiag ? j : 0]
                       : kStream ? (double)ns[k] : lrs[j * kThreads];
      const VT dv = kRegDiag ? di[kRegDiag ? j : 0]
                    : kStream ? (VT)nd[k] : (VT)ldi[j * kThreads];
      if (kStream && AHEAD == 1 && j + 1 < RPT) load_row(j + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int d = 0; d < ND; ++d) acc = __builtin_fma(vr[d], c[d] - pi, acc);
      VT qi = (VT)__builtin_fma(s, pi, acc);
      if (kStream) qi = (live >> j) & 1 ? qi : (VT)0;
      q[j] = qi;
      pin(q[j]);
      fn(j, pi, dv);
      __builtin_amdgcn_sched_barrier(0);
      if (kStream && AHEAD > 1 && j + AHEAD < RPT) load_row(j + AHEAD);
    }
  };

  bool first = true, ok = true;
  int itp = 0, last_refine = 0, refinements = 0, converged = 0;
  double rr = 0.0, rz = 0.0, bb = 0.0, thr = 0.0, rr_ref = 0.0, rr_out = 0.0;
  for (;;) {
    double s[5] = {0.0, 0.0, 0.0, rr, rz};
    bool refine = first;
    if (!first) {
      __syncthreads();
      if constexpr (kStream) {
        T.template exchange<VT>(lp, &sh.bad);
        __syncthreads();
      }
      VT *lqc = M.lq + opaque(at0);
      sweep([&](int j, double pi, VT dv) {
        if constexpr (kGhost) lqc[j * kThreads] = q[j];
        const double qd = (double)q[j], dq = (double)(dv * q[j]);
        s[0] = __builtin_fma(pi, qd, s[0]);
        s[1] = __builtin_fma(dq, (double)r[j], s[1]);
        s[2] = __builtin_fma(dq, qd, s[2]);
        pin(s[0]), pin(s[1]), pin(s[2]);
      });
      if constexpr (kGhost) ++T.tag;
      ok = team_sum(tm, sh, s, [&] {
        if constexpr (kGhost) {
          const int from = sums_threads(tm);
          T.template publish<VT>(M.lq, from);
          T.template fetch<VT>(from, &sh.bad, [&](int32_t h, int32_t, VT qv) { M.gq[h] = qv; });
        }
      });
      if (!ok) break;
      // (a step between two reliable updates, so that the loop ends)
      refine = itp > last_refine && (s[3] < thr || s[3] < a.delta2 * rr_ref ||
                                     itp - last_refine >= a.max_interval || itp >= a.maxit);
    }
    if (!refine) {
      itp += 1;
      const double rho = s[4], alpha = rho / s[0];
      const double rho_next = rho - 2.0 * alpha * s[1] + alpha * alpha * s[2];
      const VT fa = (VT)alpha, fb = (VT)(rho_next / rho);
      rr = rz = 0.0;
      double *lc = lp + opaque(at0);
      const double *ldi = M.di + opaque(t);
      Tile::Walk w = T.first(opaque(t));
      constexpr int kAhead = AHEAD > 1 ? 2 * AHEAD : 1;  // rows of D^-1 in flight
      float nd[kAhead];
      auto load_update = [&](int j) {
        if constexpr (kStream) {
          nd[j % kAhead] = mixed_dinv<VT>(a, (live >> j) & 1 ? w.g : T.g0);
          T.next(w);
        }
      };
#pragma unroll
      for (int j = 0; j < kAhead; ++j) load_update(j);
      double np = lc[0];
#pragma unroll
      for (int j = 0; j < RPT; ++j) {
        if (BATCH && j >= nj) break;
        const VT dv = kRegDiag ? di[kRegDiag ? j : 0]
                      : kStream ? (VT)nd[j % kAhead] : (VT)ldi[j * kThreads];
        if (j + kAhead < RPT) load_update(j + kAhead);
        const VT pi = (VT)np;
        if (j + 1 < RPT) np = lc[(j + 1) * kThreads];
        xa[j] = xa[j] + fa * pi;
        r[j] = r[j] - fa * q[j];
        const VT z = dv * r[j];
        const VT p = z + fb * pi;
        const double rd = (double)r[j];
        rr = __builtin_fma(rd, rd, rr);
        rz = __builtin_fma(rd, (double)z, rz);
        if ((live >> j) & 1) lc[j * kThreads] = (double)p;
        pin(r[j]), pin(xa[j]), pin(rr), pin(rz);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (kGhost) {
        for (int32_t h = t; h < T.ng; h += kThreads) {
          const int32_t at = T.gpos[h];
          const VT rn = M.gr[h] - fa * M.gq[h];
          M.gr[h] = rn;
          lp[at] = (double)(M.gd[h] * rn + fb * (VT)lp[at]);
        }
      }
      continue;
    }
    // reliable update (or the first residual): r64 = b - A x - A (xa + xlo)
    double r64[RPT];
    {
      Tile::Walk w = T.first(opaque(t));
#pragma unroll
      for (int j = 0; j < RPT; ++j) {
        const bool in = (live >> j) & 1;
        r64[j] = in ? a.b[w.g] : 0.0;
        if (!first) q[j] = (VT)lp[at0 + j * kThreads];  // p
        T.next(w);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (first) {
#pragma unroll
      for (int j = 0; j < RPT; ++j) bb = __builtin_fma(r64[j], r64[j], bb);
    }
    // (values of memory in groups of rows and the next rows' in flight, each
    // row waits for its own else; with 7 and 9 cells a thread more than this
    // spills registers of the iterations)
    constexpr int G = RPT <= 5 ? RPT : kGhost ? 2 : 4;
    for (int part = 0; part < (first ? 1 : 2); ++part) {
      __syncthreads();  // the last readers of LDS are done
      {
        const double *const y = part == 0 ? a.x : a.xlo;
        Tile::Walk w = T.first(opaque(t));
#pragma unroll
        for (int j0 = 0; j0 < RPT; j0 += G) {
          double yi[G];
#pragma unroll
          for (int j = j0; j < j0 + G && j < RPT; ++j) {
            yi[j - j0] = load_at(y, (uint32_t)((live >> j) & 1 ? w.g : T.g0) * 8u);
            T.next(w);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int j = j0; j < j0 + G && j < RPT; ++j)
            if ((live >> j) & 1)
              lp[at0 + j * kThreads] = part == 0 ? yi[j - j0] : yi[j - j0] + (double)xa[j];
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __syncthreads();
      T.template exchange<double>(lp, &sh.bad);
      __syncthreads();
      {
        constexpr int kNext = RPT <= 5 ? 2 : 1;
        double nv[kNext][ND], ns[kNext];
        Tile::Walk w = T.first(opaque(t));
        auto load_row = [&](int j) {
          const uint32_t g = (uint32_t)((live >> j) & 1 ? w.g : T.g0) * 8u;
#pragma unroll
          for (int d = 0; d < ND; ++d)
            nv[j % kNext][d] = d < a.ndiag ? load_at(a.val + (int64_t)d * a.n, g) : 0.0;
          ns[j % kNext] = load_at(a.rowsum, g);
          T.next(w);
        };
#pragma unroll
        for (int j = 0; j < kNext && j < RPT; ++j) load_row(j);
        const double *lc = lp + opaque(at0);
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
          const double yi = lc[j * kThreads];
          double acc = 0.0;
#pragma unroll
          for (int d = 0; d < ND; ++d)
            acc = __builtin_fma(nv[j % kNext][d], lc[j * kThreads + a.shift[d]] - yi, acc);
          acc = __builtin_fma(ns[j % kNext], yi, acc);
          if ((live >> j) & 1) r64[j] -= acc;
          pin(r64[j]);
          __builtin_amdgcn_sched_barrier(0);
          if (j + kNext < RPT) load_row(j + kNext);
        }
      }
    }
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
      Tile::Walk w = T.first(opaque(t));
#pragma unroll
      for (int j0 = 0; j0 < RPT; j0 += G) {
        double hi[G], lo[G];
        uint32_t at[G];
#pragma unroll
        for (int j = j0; j < j0 + G && j < RPT; ++j) {
          at[j - j0] = (uint32_t)((live >> j) & 1 ? w.g : T.g0) * 8u;
          hi[j - j0] = load_at(a.x, at[j - j0]);
          lo[j - j0] = load_at(a.xlo, at[j - j0]);
          T.next(w);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = j0; j < j0 + G && j < RPT; ++j) {
          const double h = hi[j - j0], dx = (double)xa[j];
          const double sm = h + dx, bp = sm - h;
          const double err = (h - (sm - bp)) + (dx - bp);
          if ((live >> j) & 1) {
            *reinterpret_cast<double *>(reinterpret_cast<char *>(a.x) + at[j - j0]) = sm;
            *reinterpret_cast<double *>(reinterpret_cast<char *>(a.xlo) + at[j - j0]) =
                lo[j - j0] + err;
          }
          xa[j] = (VT)0;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    rr_ref = u[0];
    if (stop) break;
    // r = r64, p += M (r64 - r); the first p is M r64
    rr = rz = 0.0;
    {
      Tile::Walk w = T.first(opaque(t));
#pragma unroll
      for (int j = 0; j < RPT; ++j) {
        if ((live >> j) & 1) {
          const VT rn = (VT)r64[j];
          const VT m = kRegDiag ? di[kRegDiag ? j : 0]
                       : kStream ? (VT)mixed_dinv<VT>(a, w.g) : (VT)M.di[t + j * kThreads];
          const VT z = m * rn;
          lp[at0 + j * kThreads] = (double)(first ? z : q[j] + m * (rn - r[j]));
          r[j] = rn;
          if constexpr (kGhost) M.lq[at0 + j * kThreads] = rn;
          // (the first rho, as the sweeps take it: with the FP64 D^-1 and residual)
          const double rd = first ? r64[j] : (double)rn;
          const double zd = first ? a.dinv[w.g] * rd : (double)z;
          rr = __builtin_fma(rd, rd, rr);
          rz = __builtin_fma(rd, zd, rz);
        }
        T.next(w);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (kGhost) {
      // the halo cells' p and r
      __syncthreads();
      T.template exchange<VT>(lp, &sh.bad);
      __syncthreads();  // no r before every thread has its p
      ++T.tag;
      T.template publish<VT>(M.lq, 0);
      T.template fetch<VT>(0, &sh.bad, [&](int32_t h, int32_t at, VT rv) {
        M.gr[h] = rv;
        if (first) {
          const int32_t cell = at - 1;  // from the line above the tile
          const int32_t line = cell / T.P - 1, c = cell - (line + 1) * T.P;
          M.gd[h] = (VT)mixed_dinv<VT>(a, T.g0 + line * T.S + c - 1);
        }
      });
    }
    first = false;
  }
  if (ok) {
    Tile::Walk w = T.first(opaque(t));
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      if ((live >> j) & 1) a.x[w.g] = bb == 0.0 ? 0.0 : a.x[w.g] + a.xlo[w.g];
      T.next(w);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (T.rank == 0 && t == 0) {
    a.st->rr = rr_out;
    a.st->bb = bb;
    a.st->iter = itp;
    a.st->converged = converged;
    a.st->refinements = refinements;
    a.st->aborted = ok ? 0 : 1;
  }
  return ok;
}

template <int KIND, class VT, int RPT, int AHEAD = 1>
__global__ __launch_bounds__(kThreads) void k_res_tile_mixed(TileArgs a) {
  extern __shared__ double dyn[];
  __shared__ SumLds sh;
  (void)tile_solve_mixed<KIND, VT, RPT, AHEAD, false>(a, blockIdx.x, gridDim.x, dyn, sh);
}

template <class VT, int RPT>
__global__ __launch_bounds__(kThreads) void k_res_tile_mixed_batch(TileArgs base) {
  extern __shared__ double dyn[];
  __shared__ SumLds sh;
  batch_loop(base, [&](const TileArgs &a, int rank, int team) {
    return tile_solve_mixed<GHOST, VT, RPT, 1, true>(a, rank, team, dyn, sh);
  });
}

__global__ void k_zero_words(word_t *p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0;
}
// (a bound of nothing: the flag is up from the start)
__device__ __forceinline__ void set_abort(ResidentAbort *a, uint64_t ticks) {
  a->raised = ticks == 0;
  a->ticks = ticks;
}
__global__ void k_set_abort(ResidentAbort *a, uint64_t ticks) {
  if (threadIdx.x == 0) set_abort(a, ticks);
}
__global__ void k_start_batch(ResidentControl *c, int *arrived, int jobs, uint64_t ticks) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < jobs) arrived[i] = 0;
  if (i == 0) {
    c->ticket = c->running = 0;
    set_abort(&c->abort, ticks);
  }
}

// The variants in order of preference (the smallest number of cells per
// thread with which the team and its LDS fit): FP64, FP32 vectors, FP64
// vectors with the FP32 matrix.  Registers that they spill: 29, 12 and 28 with 9
// cells; streamed, 0, 21, 4 in FP64, 0, 16, 92 with FP32 vectors and 0, 166, 368
// with FP64 ones, which is why the FP32 matrix is the slowest mode at 2048^2
// (47 us an iteration; FP64 37, FP32 vectors 26): its update reads D^-1 a second
// time and waits for p's exchange between update and product.
struct TileVariant {
  int kind, rpt;
  size_t (*lds)(const TileArgs &);
  void (*fn)(TileArgs);
};
#define LFG_TILE(R) {GHOST, R, &TileLds<GHOST, double, R>::bytes, &k_res_tile<R>}
#define LFG_TILEM(K, T, R, A) {K, R, &TileLds<K, T, R>::bytes, &k_res_tile_mixed<K, T, R, A>}
#define LFG_STREAM(R, ...) {STREAM, R, &StreamLds<R>::bytes, &k_res_stream<R, __VA_ARGS__>}
const std::vector<TileVariant> kTileVariants[3] = {
    {LFG_TILE(1), LFG_TILE(3), LFG_TILE(5), LFG_TILE(7), LFG_TILE(9), LFG_STREAM(17, 17, 1),
     LFG_STREAM(25, 16, 1), LFG_STREAM(33, 0, 1)},
    {LFG_TILEM(GHOST, float, 1, 1), LFG_TILEM(GHOST, float, 3, 1), LFG_TILEM(GHOST, float, 5, 1),
     LFG_TILEM(GHOST, float, 7, 1), LFG_TILEM(GHOST, float, 9, 1), LFG_TILEM(STREAM, float, 17, 4),
     LFG_TILEM(STREAM, float, 25, 4), LFG_TILEM(STREAM, float, 33, 4)},
    {LFG_TILEM(GHOST, double, 1, 1), LFG_TILEM(GHOST, double, 3, 1),
     LFG_TILEM(GHOST, double, 5, 1), LFG_TILEM(GHOST, double, 7, 1),
     LFG_TILEM(GHOST, double, 9, 1), LFG_TILEM(STREAM, double, 17, 4),
     LFG_TILEM(STREAM, double, 25, 3), LFG_TILEM(STREAM, double, 33, 2)},
};
#undef LFG_TILE
#undef LFG_STREAM
#undef LFG_TILEM

// Splits the lattice a.S x a.L into at most `most` tiles of at most cap padded
// cells whose LDS fits; among the splits, the one with the shortest rim (the
// halo travels every iteration) and, where every workgroup sums all members'
// partials, the smallest team.  STREAM: lines of a tile are read in 128-byte
// pieces, two of which at their ends another tile reads too, so a tile line
// counts as 16 cells more.  Returns the team, 0 if there is no such split.
int tile_split(TileArgs &a, int64_t cap, int most, bool stream, size_t (*lds)(const TileArgs &)) {
  int64_t best = -1;
  int team = 0;
  TileArgs pick = a;
  for (int32_t tx = 1; tx <= most && tx <= a.S; ++tx) {
    const int32_t TW = (a.S + tx - 1) / tx, TX = (a.S + TW - 1) / TW;
    const int32_t lines = (int32_t)std::min<int64_t>(cap / (TW + 2), a.L);  // lines a tile
    if (lines < 1 || TX > most) continue;
    int32_t TY = (a.L + lines - 1) / lines;
    if ((int64_t)TX * TY > most) continue;
    const int32_t TH = (a.L + TY - 1) / TY;
    TY = (a.L + TH - 1) / TH;
    TileArgs c = a;
    c.TW = TW;
    c.TH = TH;
    c.TX = TX;
    c.slots = 2 * (TW + TH);
    c.ghosts = (2 * (TW + 2) + 2 * TH + 1) / 2 * 2;
    if (lds(c) > kLdsDynamic) continue;
    const int32_t wgs = TX * TY;
    int64_t cost = wgs == 1 ? 0 : 2 * (TW + TH) + 7 * std::min(wgs, kFlatTeam);
    if (stream) cost += 16 * (int64_t)TH;
    if (best >= 0 && cost >= best) continue;
    best = cost;
    team = wgs;
    pick = c;
  }
  if (team > 0) a = pick;
  return team;
}

// Row offsets to offsets in the padded tile: off = dy S + dx with |dx|, |dy|
// <= 1.  (An offset that no row of this lattice has gets 0: its values are
// zero.)
template <class J>
void tile_shifts(J &a) {
  for (int d = 0; d < ND; ++d) {
    const int32_t o = d < a.ndiag ? a.off[d] : 0;
    const int32_t dy = o > 1 ? 1 : o < -1 ? -1 : 0, dx = o - dy * a.S;
    a.shift[d] = std::abs(dx) <= 1 ? dy * (a.TW + 2) + dx : 0;
  }
}

// the first variant that takes the lattice, or nullptr
const TileVariant *tile_plan(TileArgs &a, int mode, bool sym, bool diag, int cus, int *team) {
  for (const TileVariant &v : kTileVariants[mode]) {
    if (v.kind == STREAM && !(sym && a.ndiag == ND && (diag || mode != LFGPU_PCG_FP64))) continue;
    const int64_t cap = (int64_t)v.rpt * kThreads;
    if ((int64_t)a.S * a.L > cap * cus) continue;
    *team = tile_split(a, cap, cus, v.kind == STREAM, v.lds);
    if (*team > 0) return &v;
  }
  return nullptr;
}

// Batches: up to 3 and up to 7 cells a thread (with 9 FP32 cells 55 registers
// spill and 64 problems of 32 to 512 lines take 59 ms instead of 46; with 7, 7 of
// the FP32 and 18 of the FP64 vectors' kernel do, and none in FP64).
struct BatchVariant {
  int rpt;
  size_t (*lds)(const TileArgs &);
  void (*fn)(TileArgs);
};
const BatchVariant kBatchVariants[3][2] = {
    {{3, &TileLds<GHOST, double, 3>::bytes, &k_res_tile_batch<3>},
     {7, &TileLds<GHOST, double, 7>::bytes, &k_res_tile_batch<7>}},
    {{3, &TileLds<GHOST, float, 3>::bytes, &k_res_tile_mixed_batch<float, 3>},
     {7, &TileLds<GHOST, float, 7>::bytes, &k_res_tile_mixed_batch<float, 7>}},
    {{3, &TileLds<GHOST, double, 3>::bytes, &k_res_tile_mixed_batch<double, 3>},
     {7, &TileLds<GHOST, double, 7>::bytes, &k_res_tile_mixed_batch<double, 7>}},
};

}  // namespace

namespace lfgpu {

void resident_free(ResidentBufs *b) {
  dfree(b->halo);
  dfree(b->sums);
  dfree(b->outcome);
  *b = ResidentBufs{};
}

static void fill_args(TileArgs &a, const ResidentDia &A, const lfgpu_pcg_opts &opts,
                      const double *b, double *x) {
  a.n = A.n;
  a.val = A.val;
  a.rowsum = A.rowsum;
  a.dinv = A.dinv;
  a.b = b;
  a.x = x;
  a.tol2 = opts.rtol * opts.rtol;
  a.maxit = opts.maxit;
  a.val32 = A.val32;
  a.rowsum32 = A.rowsum32;
  a.dinv32 = A.dinv32;
  a.dinv16 = static_cast<const __hip_bfloat16 *>(A.dinv16);
  a.xlo = A.xlo;
  a.delta2 = opts.refine_delta > 0.0 ? opts.refine_delta * opts.refine_delta : 0.09;
  a.max_interval = opts.refine_max_interval > 0 ? opts.refine_max_interval : 2147483647;
}

int resident_clear(hipStream_t s, unsigned long long *words, size_t n) {
  if (n == 0) return LFGPU_OK;
  hipLaunchKernelGGL(k_zero_words, dim3((unsigned)std::min<size_t>(256, (n + 255) / 256)),
                     dim3(256), 0, s, words, n);
  LFG_HIP(hipGetLastError());
  return LFGPU_OK;
}

bool resident_will_clear(const ResidentBufs *bufs, size_t words, uint64_t need) {
  return !bufs->outcome || words > bufs->halo_words || bufs->epoch + need > 0xfffffff0ull;
}

int resident_start_batch(lfgpu_ctx *ctx, ResidentControl *control, int jobs) {
  hipLaunchKernelGGL(k_start_batch, dim3((unsigned)((jobs + 255) / 256)), dim3(256), 0,
                     ctx->stream, control, control->arrived(), jobs, ctx->wait_ticks);
  LFG_HIP(hipGetLastError());
  return LFGPU_OK;
}

int resident_prepare(lfgpu_ctx *ctx, ResidentBufs *bufs, size_t words, uint64_t need,
                     uint32_t *tag0) {
  hipStream_t s = ctx->stream;
  if (!bufs->outcome) {
    if (!bufs->sums) LFG_TRY(dalloc(&bufs->sums, kPartWords + kTotalWords, "resident PCG sums"));
    LFG_TRY(dalloc(&bufs->outcome, 1, "resident PCG state"));
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
  bool fresh = false;
  if (bufs->epoch + need > 0xfffffff0ull) {
    hipLaunchKernelGGL(k_zero_words, dim3(256), dim3(256), 0, s, bufs->halo, bufs->halo_words);
    hipLaunchKernelGGL(k_zero_words, dim3(8), dim3(256), 0, s, bufs->sums,
                       kPartWords + kTotalWords);
    bufs->epoch = 0;
    fresh = true;
  }
  if (fresh || bufs->ticks != ctx->wait_ticks) {
    bufs->ticks = ctx->wait_ticks;
    hipLaunchKernelGGL(k_set_abort, dim3(1), dim3(64), 0, s, &bufs->outcome->team,
                       bufs->ticks);
    LFG_HIP(hipGetLastError());
  }
  *tag0 = bufs->epoch;
  bufs->epoch = (uint32_t)std::min<uint64_t>(bufs->epoch + need, 0xffffffffull);
  return LFGPU_OK;
}

int resident_launch_team(hipStream_t s, const void *fn, int team, void *args, size_t lds,
                         bool *taken) {
  LFG_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  void *argv[] = {args};
  if (team == 1) {
    LFG_HIP(hipLaunchKernel(fn, dim3(1), dim3(kThreads), argv, lds, s));
  } else {
    // all workgroups of the team must run at once
    const hipError_t e =
        hipLaunchCooperativeKernel(fn, dim3(team), dim3(kThreads), argv, (unsigned)lds, s);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      return e == hipErrorCooperativeLaunchTooLarge ? LFGPU_OK : kResidentRefused;
    }
  }
  *taken = true;
  return LFGPU_OK;
}

int resident_launch(hipStream_t s, ResidentBufs *bufs, const void *fn, int team, void *args,
                    size_t lds, ResidentOutcome *out, bool *taken) {
  LFG_TRY(resident_launch_team(s, fn, team, args, lds, taken));
  if (*taken)
    LFG_HIP(hipMemcpyAsync(out, bufs->outcome, sizeof(ResidentOutcome), hipMemcpyDeviceToHost, s));
  return LFGPU_OK;
}

int resident_pcg_dia(lfgpu_ctx *ctx, ResidentBufs *bufs, const ResidentDia &A,
                     const lfgpu_pcg_opts &opts, const double *b, double *x,
                     ResidentOutcome *out, bool *taken, bool *ask) {
  *taken = false;
  if (A.n <= 0 || A.width <= 0 || A.ndiag > ND) return LFGPU_OK;
  TileArgs a{};
  a.n = A.n;
  a.S = A.width;
  a.L = A.n / A.width;
  a.ndiag = A.ndiag;
  int team = 0;
  const int cus = std::min(ctx->cus, kMaxTeam);
  const TileVariant *v = tile_plan(a, opts.mode, A.sym, A.diag, cus, &team);
  if (!v && ask) *ask = tile_plan(a, opts.mode, true, true, cus, &team) != nullptr;
  if (!v) return LFGPU_OK;
  for (int d = 0; d < A.ndiag; ++d) a.off[d] = A.off[d];
  tile_shifts(a);
  // tags of this solve: one exchange and one sum an iteration, six for a
  // reliable update (at most one an iteration), and a few at the start
  hipStream_t s = ctx->stream;
  LFG_TRY(resident_prepare(ctx, bufs, (size_t)2 * team * 2 * a.slots,
                           (uint64_t)opts.maxit * (opts.mode == LFGPU_PCG_FP64 ? 1 : 7) + 16,
                           &a.tag0));
  fill_args(a, A, opts, b, x);
  a.halo_words = bufs->halo;
  a.part = bufs->sums;
  a.total = bufs->sums + kPartWords;
  a.abort = &bufs->outcome->team;
  a.st = &bufs->outcome->solve;
  bufs->kept = v->kind == STREAM && opts.mode == LFGPU_PCG_FP64;
  if (bufs->kept)
    LFG_HIP(hipMemcpyAsync(A.keep, x, (size_t)A.n * 8, hipMemcpyDeviceToDevice, s));
  return resident_launch(s, bufs, reinterpret_cast<const void *>(v->fn), team, &a, v->lds(a), out,
                         taken);
}


// ---------------------------------------------------------------------------
// batches
// ---------------------------------------------------------------------------
struct ResidentTiles {
  bool fits = false;
  int nslots = 0, njobs = 0, variant = 0;
  size_t lds = 0;
  size_t halo_words = 0, sums_words = 0;
  TileJob *jobs = nullptr;
  int2 *slots = nullptr;
  word_t *words = nullptr;  // sums, then halos
  ResidentControl *control = nullptr;
  uint32_t epoch = 0xffffffffu;
};

void resident_tiles_free(ResidentTiles *p) {
  if (!p) return;
  dfree(p->jobs);
  dfree(p->slots);
  dfree(p->words);
  dfree(p->control);
  delete p;
}

// Team sizes: the problems run side by side, so that the batch takes as long
// as its longest problem while all teams fit the chip; iterations grow with
// the square root of the rows, an iteration takes about 2.5 us and 0.8 ns a
// cell of a workgroup.  The cells a workgroup takes follow from the smallest
// common finishing time with which the teams fit; where none does, every
// workgroup takes as many as it can hold and the longest problems go first.
int resident_tiles_plan(lfgpu_ctx *ctx, const std::vector<ResidentProblem> &probs, int mode,
                        ResidentTiles **out) {
  ResidentTiles *p = new ResidentTiles();
  *out = p;
  const int cus = std::min(ctx->cus, kMaxTeam);
  const BatchVariant &big = kBatchVariants[mode][1];
  const int64_t cap = (int64_t)big.rpt * kThreads;
  const size_t np = probs.size();
  if (np == 0) return LFGPU_OK;
  auto iterations = [&](const ResidentProblem &q) { return std::sqrt((double)q.n); };
  auto split = [&](const ResidentProblem &q, int64_t cells, TileArgs &a) {
    a = TileArgs{};
    a.S = q.width;
    a.L = q.n / q.width;
    return tile_split(a, cells, cus, false, big.lds);
  };
  // teams for a common finishing time tau; 0 if one does not fit
  std::vector<int> team(np);
  std::vector<TileArgs> geo(np);
  auto total = [&](double tau) {
    int64_t sum = 0;
    for (size_t k = 0; k < np; ++k) {
      const double c = tau > 0.0 ? (tau / iterations(probs[k]) - 2.5) / 0.0008 : (double)cap;
      const int64_t cells = (int64_t)std::min<double>((double)cap, std::max(c, 128.0));
      team[k] = split(probs[k], cells, geo[k]);
      if (team[k] == 0) team[k] = split(probs[k], cap, geo[k]);
      if (team[k] == 0) return (int64_t)-1;
      sum += team[k];
    }
    return sum;
  };
  int64_t all = total(0.0);
  if (all < 0) return LFGPU_OK;
  if (all <= cus) {
    double hi = 0.0;
    for (const ResidentProblem &q : probs)
      hi = std::max(hi, iterations(q) * (2.5 + 0.0008 * (double)cap));
    double lo = 0.0;
    for (int step = 0; step < 10; ++step) {
      const double mid = 0.5 * (lo + hi);
      if (total(mid) <= cus) hi = mid;
      else lo = mid;
    }
    all = total(hi);
  }
  std::vector<size_t> order(np);
  for (size_t k = 0; k < np; ++k) order[k] = k;
  auto cost = [&](size_t k) {
    return iterations(probs[k]) * (2.5 + 0.0008 * (geo[k].TW + 2) * geo[k].TH);
  };
  std::stable_sort(order.begin(), order.end(),
                   [&](size_t i, size_t j) { return cost(i) > cost(j); });
  std::vector<TileJob> jobs(np);
  std::vector<int2> slots;
  int64_t most = 0;
  for (size_t o = 0; o < np; ++o) {
    const size_t k = order[o];
    const ResidentProblem &q = probs[k];
    const TileArgs &g = geo[k];
    TileJob &j = jobs[o];
    j.index = q.index;
    j.lo = q.lo;
    j.S = g.S;
    j.L = g.L;
    j.TW = g.TW;
    j.TH = g.TH;
    j.TX = g.TX;
    j.team = team[k];
    j.slots = g.slots;
    j.ghosts = g.ghosts;
    j.ndiag = q.ndiag;
    for (int d = 0; d < ND; ++d) j.off[d] = d < q.ndiag ? q.off[d] : 0;
    tile_shifts(j);
    j.halo_at = p->halo_words;
    j.sums_at = p->sums_words;
    if (j.team > 1) {  // (a workgroup alone exchanges nothing)
      p->halo_words += (size_t)2 * j.team * 2 * j.slots;
      p->sums_words += part_words(j.team) + kTotalWords;
    }
    most = std::max<int64_t>(most, (int64_t)(g.TW + 2) * g.TH);
    for (int r = 0; r < j.team; ++r) slots.push_back(int2{(int)o, r});
  }
  p->variant = most <= (int64_t)kBatchVariants[mode][0].rpt * kThreads ? 0 : 1;
  for (size_t k = 0; k < np; ++k)
    p->lds = std::max(p->lds, kBatchVariants[mode][p->variant].lds(geo[k]));
  p->nslots = (int)slots.size();
  hipStream_t s = ctx->stream;
  LFG_TRY(dalloc(&p->jobs, np, "resident batch jobs"));
  LFG_TRY(dalloc(&p->slots, slots.size(), "resident batch slots"));
  LFG_TRY(dalloc(&p->words, p->sums_words + p->halo_words, "resident batch words"));
  p->njobs = (int)np;
  LFG_TRY(ResidentControl::alloc(&p->control, np));
  LFG_HIP(hipMemcpyAsync(p->jobs, jobs.data(), np * sizeof(TileJob), hipMemcpyHostToDevice, s));
  LFG_HIP(hipMemcpyAsync(p->slots, slots.data(), slots.size() * sizeof(int2),
                         hipMemcpyHostToDevice, s));
  LFG_HIP(hipStreamSynchronize(s));
  p->fits = true;
  return LFGPU_OK;
}

bool resident_tiles_fit(const ResidentTiles *p) { return p && p->fits; }

void resident_tiles_reset(ResidentTiles *p) { p->epoch = 0xffffffffu; }

int resident_tiles_run(lfgpu_ctx *ctx, ResidentTiles *p, const ResidentDia &A,
                       const lfgpu_pcg_opts &opts, const double *b, double *x, ResidentState *st,
                       ResidentAbort *ab, bool *taken) {
  *taken = false;
  hipStream_t s = ctx->stream;
  const uint64_t need = (uint64_t)opts.maxit * (opts.mode == LFGPU_PCG_FP64 ? 1 : 7) + 16;
  if (p->epoch + need > 0xfffffff0ull) {
    hipLaunchKernelGGL(k_zero_words, dim3(256), dim3(256), 0, s, p->words,
                       p->sums_words + p->halo_words);
    p->epoch = 0;
  }
  LFG_TRY(resident_start_batch(ctx, p->control, p->njobs));
  TileArgs a{};
  fill_args(a, A, opts, b, x);
  a.halo_words = p->words + p->sums_words;
  a.part = p->words;
  a.abort = &p->control->abort;
  a.tag0 = p->epoch;
  a.st = st;
  a.jobs = p->jobs;
  a.job_slots = p->slots;
  a.nslots = p->nslots;
  a.ticket = &p->control->ticket;
  a.running = &p->control->running;
  a.arrived = p->control->arrived();
  p->epoch = (uint32_t)std::min<uint64_t>(p->epoch + need, 0xffffffffull);
  const int team = std::min(p->nslots, std::min(ctx->cus, kMaxTeam));
  LFG_TRY(resident_launch_team(
      s, reinterpret_cast<const void *>(kBatchVariants[opts.mode][p->variant].fn), team, &a,
      p->lds, taken));
  LFG_HIP(hipMemcpyAsync(ab, a.abort, sizeof(ResidentAbort), hipMemcpyDeviceToHost, s));
  return LFGPU_OK;
}

}  // namespace lfgpu
