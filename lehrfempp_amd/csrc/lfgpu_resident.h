// Resident Jacobi-PCG (lfgpu_resident.hip): the whole solve in one launch.
#pragma once

#include <cstdint>

#include "lfgpu_internal.h"

namespace lfgpu {

// Outcome of a resident solve as the device leaves it.
struct ResidentState {
  double rr, bb;
  int iter, converged, refinements, aborted;
};

// Communication buffers of the resident solves on one matrix (owned by the
// solver cache); epoch is the last tag any exchange in them has used.
struct ResidentBufs {
  unsigned long long *halo = nullptr;
  size_t halo_words = 0;
  unsigned long long *sums = nullptr;  // team sums (fixed size)
  ResidentState *state = nullptr;      // followed by the abort flag
  int *abort = nullptr;
  uint32_t epoch = 0;
};
void resident_free(ResidentBufs *b);

// A matrix on DIA storage (val[d * n + row], offsets ascending) whose rows
// form a lattice: `width` rows a line, n / width lines, no entry but between
// lattice neighbours (dia_lattice in lfgpu_solver.hip).
struct ResidentDia {
  int32_t n = 0, width = 0;
  int ndiag = 0;
  const int32_t *off = nullptr;
  const double *val = nullptr, *rowsum = nullptr, *dinv = nullptr;
  bool sym = false;  // lower diagonals equal the mirrored upper ones bit for bit
  // mixed modes: the FP32 copies, D^-1 in bfloat16 (FP32 vectors) or FP32,
  // and the solution's low part
  const float *val32 = nullptr, *rowsum32 = nullptr, *dinv32 = nullptr;
  const void *dinv16 = nullptr;
  double *xlo = nullptr;
};

// Jacobi-PCG in opts.mode on the context stream (rtol, maxit, mode and the
// refinement options of lfgpu_pcg), queued without synchronisation; *st
// (pinned) receives the outcome.  *taken = false (and nothing queued) when
// the system does not fit the chip.
int resident_pcg_dia(lfgpu_ctx *ctx, ResidentBufs *bufs, const ResidentDia &A,
                     const lfgpu_pcg_opts &opts, const double *b, double *x, ResidentState *st,
                     bool *taken);

}  // namespace lfgpu
