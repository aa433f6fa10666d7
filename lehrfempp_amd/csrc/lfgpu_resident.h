// Resident Jacobi-PCG (lfgpu_resident.hip): the whole solve in one launch.
#pragma once

#include <algorithm>
#include <chrono>
#include <cstdint>
#include <vector>

#include "lfgpu_internal.h"

namespace lfgpu {

// Outcome of a resident solve as the device leaves it.
struct ResidentState {
  double rr, bb;
  int iter, converged, refinements, aborted;
};

// The bound on the waits of a launch, and the flag by which a workgroup that
// gave one up ends all teams of the launch.  The flag alone tells whether a
// solve is whole: a workgroup that gives up in the last sum leaves its part of
// x unwritten, while the one that reports may have got its total and found
// convergence.
struct ResidentAbort {
  int raised, pad;
  uint64_t ticks;
};
// What the host reads after a solve.
struct ResidentOutcome {
  ResidentState solve;
  ResidentAbort team;
};

// When the resident solves of a matrix or a batch may run again after one that
// gave up or was refused: the sweeps take over for 16 times as long as it cost, twice as long
// after each further one in a row, so that a lasting cause (a part of the chip
// held by another process) costs a few per cent and a passing one not the
// resident solves for good.
struct ResidentPause {
  double until = 0.0, times = 16.0;
  static double now() {
    return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch())
        .count();
  }
  bool over() const { return until == 0.0 || now() >= until; }
  void start(double lost) {
    until = now() + times * lost;
    times = std::min(2.0 * times, 1e6);
  }
};

// Communication buffers of the resident solves on one matrix (owned by the
// solver cache); epoch is the last tag any exchange in them has used.
struct ResidentBufs {
  unsigned long long *halo = nullptr;
  size_t halo_words = 0;
  unsigned long long *sums = nullptr;  // team sums (fixed size)
  ResidentOutcome *outcome = nullptr;
  uint64_t ticks = 0;  // outcome->team.ticks
  bool kept = false;   // the last solve's start is in its ResidentDia::keep
  uint32_t epoch = 0;
};
void resident_free(ResidentBufs *b);
// Buffers for a solve that exchanges through `words` words and uses at most
// `need` tags; *tag0 the tag before its first.
int resident_prepare(lfgpu_ctx *ctx, ResidentBufs *bufs, size_t words, uint64_t need,
                     uint32_t *tag0);
// Whether resident_prepare would clear the buffers.
bool resident_will_clear(const ResidentBufs *bufs, size_t words, uint64_t need);
int resident_clear(hipStream_t s, unsigned long long *words, size_t n);
// What the workgroups of a batch share: the counter that hands out the slots,
// the number of workgroups that run, the abort flag and, behind them, every
// problem's number of workgroups that have come to it; set before every launch.
struct ResidentControl {
  int ticket, running;
  ResidentAbort abort;
  int *arrived() { return reinterpret_cast<int *>(this + 1); }
  static int alloc(ResidentControl **out, size_t jobs) {
    void *p = nullptr;
    const int rc = dmalloc(&p, sizeof(ResidentControl) + jobs * sizeof(int),
                           "resident batch counters");
    *out = static_cast<ResidentControl *>(p);
    return rc;
  }
};
int resident_start_batch(lfgpu_ctx *ctx, ResidentControl *control, int jobs);
// Status of a cooperative launch that the runtime refused: while another
// process that has made such launches lives on the device, they fail with
// hipErrorIllegalState, and the sweeps have to do.
constexpr int kResidentRefused = -1;
int resident_launch_team(hipStream_t s, const void *fn, int team, void *args, size_t lds,
                         bool *taken);
// Queues kernel fn (one argument struct) on `team` workgroups that all run at
// once, and the copy of its outcome to *st; *taken = false where the chip
// does not hold them.
int resident_launch(hipStream_t s, ResidentBufs *bufs, const void *fn, int team, void *args,
                    size_t lds, ResidentOutcome *out, bool *taken);

// A matrix on DIA storage (val[d * n + row], offsets ascending) whose rows
// form a lattice: `width` rows a line, n / width lines, no entry but between
// lattice neighbours (dia_lattice in lfgpu_solver.hip).
struct ResidentDia {
  int32_t n = 0, width = 0;
  int ndiag = 0;
  const int32_t *off = nullptr;
  const double *val = nullptr, *rowsum = nullptr, *dinv = nullptr;
  bool sym = false;  // lower diagonals equal the mirrored upper ones bit for bit
  bool diag = false;  // 1 / dinv is the row sum less the off-diagonal values, to 1e-13
  // mixed modes: the FP32 copies, D^-1 in bfloat16 (FP32 vectors) or FP32,
  // and the solution's low part
  const float *val32 = nullptr, *rowsum32 = nullptr, *dinv32 = nullptr;
  const void *dinv16 = nullptr;
  double *xlo = nullptr;
  // n values for the start of the streamed FP64 solve, which updates x in memory.
  // A workgroup that gives up in a team sum still sends what it has, and the
  // others may take one step with that before they see the flag; the other
  // solves write x only after a later sum, which then does not come.
  double *keep = nullptr;
};

// Jacobi-PCG in opts.mode on the context stream (rtol, maxit, mode and the
// refinement options of lfgpu_pcg), queued without synchronisation; *out
// (pinned) receives the outcome.  *taken = false (and nothing queued) when
// the system does not fit the chip; *ask (unless null) is set then if it would
// with A.sym and A.diag.
int resident_pcg_dia(lfgpu_ctx *ctx, ResidentBufs *bufs, const ResidentDia &A,
                     const lfgpu_pcg_opts &opts, const double *b, double *x,
                     ResidentOutcome *out, bool *taken, bool *ask);

// The lattice problems of a batch, side by side in one launch.  st (device)
// receives the outcome of problem `index` at st[index], *ab (pinned) the flag.
struct ResidentProblem {
  int32_t index, lo, n, width, ndiag;
  int32_t off[8];
};
struct ResidentTiles;
int resident_tiles_plan(lfgpu_ctx *ctx, const std::vector<ResidentProblem> &probs, int mode,
                        ResidentTiles **out);
bool resident_tiles_fit(const ResidentTiles *p);
void resident_tiles_free(ResidentTiles *p);
// After an aborted solve: the next one clears the words.
void resident_tiles_reset(ResidentTiles *p);
// (A.width, A.ndiag and A.off are the problems' own)
int resident_tiles_run(lfgpu_ctx *ctx, ResidentTiles *p, const ResidentDia &A,
                       const lfgpu_pcg_opts &opts, const double *b, double *x, ResidentState *st,
                       ResidentAbort *ab, bool *taken);

// Sliced-ELL storage split over a team for the resident solves: a workgroup
// owns a run of storage rows and keeps their p in LDS, with the values of the
// rows it reads of others behind them (lfgpu_resident_ell.hip).
struct ResidentEllPlan;
void resident_ell_free(ResidentEllPlan *p);
bool resident_ell_fits(const ResidentEllPlan *p);

// A matrix on sliced-ELL storage with 16-bit column offsets.
struct ResidentEll {
  int32_t n = 0;  // storage rows
  int64_t slots = 0;
  // perm: storage row -> row of x and b (-1: an empty row); null: the same
  const int32_t *slice_off = nullptr, *perm = nullptr;
  const int16_t *dcol = nullptr;
  const double *val = nullptr, *rowsum = nullptr, *dinv = nullptr;
  const float *val32 = nullptr, *rowsum32 = nullptr, *dinv32 = nullptr;
  const void *dinv16 = nullptr;
  double *xlo = nullptr;  // in storage order
};
// As resident_pcg_dia; *plan is built by the first call.
int resident_pcg_ell(lfgpu_ctx *ctx, ResidentBufs *bufs, ResidentEllPlan **plan,
                     const ResidentEll &A, const lfgpu_pcg_opts &opts, const double *b, double *x,
                     ResidentOutcome *out, bool *taken);
// The problems of a batch that are no lattices: problem q owns the storage
// rows from q.lo (a multiple of 64) on, q.n of them.
int resident_ell_batch_plan(lfgpu_ctx *ctx, const ResidentEll &A,
                            const std::vector<ResidentProblem> &probs, ResidentEllPlan **out);
int resident_ell_batch_run(lfgpu_ctx *ctx, ResidentBufs *bufs, ResidentEllPlan *plan,
                           const ResidentEll &A, const lfgpu_pcg_opts &opts, const double *b,
                           double *x, ResidentState *st, ResidentAbort *ab, bool *taken);

}  // namespace lfgpu
