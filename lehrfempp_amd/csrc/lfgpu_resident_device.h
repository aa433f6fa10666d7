// Communication between the workgroups of one resident solve.
//
// A resident solve keeps a system's vectors in the registers and LDS of a
// team of workgroups that stay on the chip for the whole solve, one per CU,
// launched cooperatively (all of them run at once).  Workgroups exchange the
// boundary values of the search direction and their partial sums through
// device memory in self-validating words: every 8-byte word carries 32 bits
// of payload and a 32-bit tag, the number of the exchange, and is stored and
// loaded whole by relaxed agent-scope atomics.  A reader polls a word until
// its tag is the one it waits for, so no ordering between different words is
// needed: no fences, no cache write-backs or invalidations.  Slots are double
// buffered by the exchange number; a workgroup writes exchange e + 2 only
// after it has read exchange e + 1 of every workgroup that reads its slot, and
// those wrote e + 1 after they had read e.
//
// Every wait is bounded by the real-time clock: a workgroup that waits longer
// than ResidentAbort::ticks raises the team's abort flag and leaves, the others see the
// flag in their own waits and leave too; the caller then runs the sweeps.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "lfgpu_resident.h"

namespace lfgpu {
namespace res {

typedef unsigned long long word_t;

constexpr int kThreads = 512;  // 8 wavefronts: 256 registers per lane
constexpr int kWaves = kThreads / 64;
constexpr int kMaxTeam = 256;  // workgroups of a team (one leader thread per member)
constexpr int kSums = 5;       // values of one team sum
// Teams of fewer workgroups read every member's partial sums in every
// workgroup (one hop: 32 members a wavefront); in larger ones each of kLeaders
// workgroups sums a group of the members and every workgroup reads the
// leaders' sums (two hops).  A member's leader is the one of the same rank
// modulo 8, which puts a group on one XCD when the ranks are the workgroup
// numbers.  A sum of five values, workgroup's part included, takes 1.3 us
// with 2 members, 1.8 with 32, 2.0 with 63, 2.3 with 64 and 2.5 with 256 (8
// leaders that poll all 256 members, five separate wavefront sums and 40 LDS
// reads a thread took 3.9).
constexpr int kFlatTeam = 64;
constexpr int kLeaders = 8;

__device__ __forceinline__ void put(word_t *p, word_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ word_t get(const word_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ word_t low_word(double v, uint32_t tag) {
  return ((word_t)__double_as_longlong(v) << 32) | tag;
}
__device__ __forceinline__ word_t high_word(double v, uint32_t tag) {
  return ((word_t)__double_as_longlong(v) & 0xffffffff00000000ull) | tag;
}
__device__ __forceinline__ double from_words(word_t lo, word_t hi) {
  return __longlong_as_double((long long)((lo >> 32) | (hi & 0xffffffff00000000ull)));
}
__device__ __forceinline__ bool tagged(word_t w, uint32_t tag) { return (uint32_t)w == tag; }

// A value of an array at a uniform base and a 32-bit byte offset per lane (one
// address register for all the arrays of a row).
template <class T>
__device__ __forceinline__ T load_at(const T *base, uint32_t bytes) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + bytes);
}
// Hides a value from the optimiser, which else keeps every row's addresses
// and masks in registers across the iterations (several hundred of them).
__device__ __forceinline__ int32_t opaque(int32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}
// Keeps a row's result where it is computed (the compiler else sinks whole
// rows past the next barrier and spills their operands).
template <class T>
__device__ __forceinline__ void pin(T &v) {
  asm volatile("" : "+v"(v));
}

// A bounded wait: returns false once the team has been aborted.
struct Wait {
  ResidentAbort *abort;
  uint64_t t0 = 0;
  uint32_t polls = 0;
  __device__ __forceinline__ explicit Wait(ResidentAbort *a) : abort(a) {}
  __device__ __forceinline__ bool more() {
    if ((++polls & 255u) != 0) return true;
    const uint64_t now = wall_clock64();
    if (t0 == 0) t0 = now;
    if (__hip_atomic_load(&abort->raised, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      return false;
    if (now - t0 > __hip_atomic_load(&abort->ticks, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
      __hip_atomic_store(&abort->raised, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
    return true;
  }
};

// The workgroups of a batch draw their slots in order, so that the first ones
// of a team find it incomplete until the others have ended the problems that
// they are at, whatever those take: that wait has no bound of time once all
// workgroups of the launch run (`running` says how many do).  It ends, since the
// earlier problems' workgroups are all there and end, or raise the flag.  Before
// that the bound holds, as a workgroup may never come while others hold its CU.
// Returns false, in all threads, once the flag is up.  `scratch` is shared.
__device__ __forceinline__ bool team_assembles(int *arrived, int team, const int *running,
                                               ResidentAbort *abort, int &scratch) {
  if (threadIdx.x == 0) {
    int up = 0;
    const uint64_t from = wall_clock64();
    __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    while (team > 1 && !up &&
           __hip_atomic_load(arrived, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < team) {
      up = __hip_atomic_load(&abort->raised, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (!up &&
          __hip_atomic_load(running, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < (int)gridDim.x &&
          wall_clock64() - from >
              __hip_atomic_load(&abort->ticks, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
        __hip_atomic_store(&abort->raised, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        up = 1;
      }
      __builtin_amdgcn_s_sleep(2);
    }
    scratch = up;
  }
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(scratch) == 0;
}

// Lane l's 32 bits from the lane that the DPP control CTRL names.
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppRor8 = 0x128;

// a summed over lane pairs (l, l + 32) in the lower half of the result, b in
// the upper half; and the same over (l, l + 16) in the even and odd rows.
__device__ __forceinline__ double fold32(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a),
                                                   (unsigned)__double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a),
                                                   (unsigned)__double2hiint(b), false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ __forceinline__ double fold16(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a),
                                                   (unsigned)__double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a),
                                                   (unsigned)__double2hiint(b), false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}

// Up to five values summed over the wavefront in a fixed order, the values
// folded into one register on the way (35 instructions; five separate DPP
// sums take 90).  PAIRS: both lanes of a pair (2i, 2i + 1) hold the same, one
// of them counts.  The result of value wave_value(l) is in lane l; every
// value is in the two lanes of which wave_owner(l) >= 0 (0 and 1).
template <bool PAIRS, int K>
__device__ __forceinline__ double wave_sums(const double (&v)[K]) {
  static_assert(K <= kSums, "too many sums");
  auto val = [&](int k) { return k < K ? v[k < K ? k : 0] : 0.0; };
  const double a = fold32(val(0), K > 1 ? val(1) : val(0));
  const double b = K > 2 ? fold32(val(2), K > 3 ? val(3) : val(2)) : a;
  double d = fold16(a, b);
  if constexpr (K > 4) {
    double c = fold32(val(4), val(4));
    c = fold16(c, c);
    const bool up = (threadIdx.x & 8) != 0;
    d = (up ? c : d) + dpp<kDppRor8>(up ? d : c);
  } else {
    d += dpp<kDppRor8>(d);
  }
  d += dpp<kDppHalfMirror>(d);
  d += dpp<kDppXor2>(d);
  if constexpr (!PAIRS) d += dpp<kDppXor1>(d);
  return d;
}
__device__ __forceinline__ int wave_value(int l) {
  return (l & 8) ? 4 : (l >> 4 & 1) * 2 + (l >> 5);
}
__device__ __forceinline__ int wave_owner(int l) {
  return (l & 14) == 0 || (l & 62) == 8 ? l & 1 : -1;
}

// The value whose low and high words the lanes 2i and 2i + 1 hold.
__device__ __forceinline__ double join_words(word_t w) {
  const int mine = (int)(w >> 32);
  const int other = __builtin_amdgcn_update_dpp(0, mine, kDppXor1, 0xf, 0xf, false);
  return (threadIdx.x & 1) ? __hiloint2double(mine, other) : __hiloint2double(other, mine);
}

// Workgroup-shared scratch of the team sums.
struct SumLds {
  double part[2][kWaves][kSums];
  double total[2][2][kSums];
  int bad;
};

// words of the team sums' buffers: a line of 16 (10 in use) per member and
// per leader
constexpr int kLine = 16;
constexpr size_t part_words(int team) { return (size_t)2 * kLine * team; }
constexpr size_t kPartWords = part_words(kMaxTeam);
constexpr size_t kTotalWords = (size_t)2 * kLine * kLeaders;
// LDS a resident kernel may take dynamically (beside SumLds)
constexpr size_t kLdsDynamic = 160 * 1024 - (sizeof(SumLds) + 1023) / 1024 * 1024;

// The team as one workgroup sees it.
struct Team {
  int rank, size;
  word_t *part;   // [2][size][kLine] partial sums of every member
  word_t *total;  // [2][kLeaders][kLine] sums over a leader's group
  ResidentAbort *abort;
  uint32_t tag;   // number of the last team sum
};

// The first sums_threads() threads of a workgroup carry a team sum, the
// others are free between its barriers.
__device__ __forceinline__ int sums_threads(const Team &tm) {
  return tm.size > 32 && tm.size < kFlatTeam ? 128 : 64;
}

// Polls N words per lane (word u at src + u * step; lanes that are not `in`
// count as arrived) until all of the wavefront's carry the tag.  (A second
// poll in flight half a round trip behind gains 1 %.)
template <int N>
__device__ __forceinline__ bool poll_words(const word_t *src, int step, bool in, uint32_t tag,
                                           ResidentAbort *abort, word_t (&a)[N]) {
  Wait wait(abort);
  for (;;) {
#pragma unroll
    for (int u = 0; u < N; ++u) a[u] = get(src + u * step);
    bool ok = true;
#pragma unroll
    for (int u = 0; u < N; ++u) ok = ok && tagged(a[u], tag);
    if (__all(ok || !in)) return true;
    if (!wait.more()) return false;
  }
}

// Sums v over all threads of the team; every thread of every workgroup gets
// the same bits: every step adds in a fixed order.  Returns false when the
// team has been aborted (in every thread of the workgroup).  Contains
// workgroup barriers: LDS written before the call is visible after it.  All
// threads run `meanwhile` between the first of them, when the workgroup's
// partials are about to go out, and the wait for the team; it must leave the
// first sums_threads() threads to themselves.
template <int K, class F>
__device__ __forceinline__ bool team_sum(Team &tm, SumLds &sh, double (&v)[K], F &&meanwhile) {
  const int t = threadIdx.x, w = t >> 6, l = t & 63;
  const uint32_t tag = ++tm.tag;
  const int par = (int)(tag & 1u);
  {
    const double s = wave_sums<false>(v);
    if (wave_owner(l) == 0 && wave_value(l) < K) sh.part[par][w][wave_value(l)] = s;
  }
  __syncthreads();
  // the workgroup's sums: waves in a fixed tree
  auto group = [&](int k) {
    const double(*p)[kSums] = sh.part[par];
    return ((p[0][k] + p[1][k]) + (p[2][k] + p[3][k])) +
           ((p[4][k] + p[5][k]) + (p[6][k] + p[7][k]));
  };
  if (tm.size == 1) {
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = group(k);
    return true;
  }
  word_t *pb = tm.part + (size_t)par * kLine * tm.size;
  if (t < 2 * K) {
    const double s = group(t >> 1);
    put(&pb[tm.rank * kLine + t], (t & 1) ? high_word(s, tag) : low_word(s, tag));
  }
  meanwhile();
  const bool flat = tm.size < kFlatTeam;
  // sums over a group of up to 32 members: lane 2i + h holds word h of member i
  auto members = [&](int first, int stride, int count) {
    word_t a[K];
    const int i = l >> 1;
    const bool in = i < count;
    const word_t *src = pb + (in ? first + i * stride : first) * kLine + (l & 1);
    if (!poll_words(src, 2, in, tag, tm.abort, a)) sh.bad = 1;
    double r[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      r[k] = join_words(a[k]);
      r[k] = in ? r[k] : 0.0;
    }
    return wave_sums<true>(r);
  };
  const int k = wave_value(l);
  if (flat) {
    if (w < 2 && w * 32 < tm.size) {
      const double s = members(w * 32, 1, tm.size - w * 32);
      if (wave_owner(l) == 0 && k < K) sh.total[par][w][k] = s;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < K; ++q) v[q] = sh.total[par][0][q];
    if (tm.size > 32)
#pragma unroll
      for (int q = 0; q < K; ++q) v[q] += sh.total[par][1][q];
    return sh.bad == 0;
  }
  if (w == 0) {
    word_t *tb = tm.total + (size_t)par * kLine * kLeaders;
    if (tm.rank < kLeaders) {
      const double s =
          members(tm.rank, kLeaders, (tm.size - tm.rank + kLeaders - 1) / kLeaders);
      const int h = wave_owner(l);
      if (h >= 0 && k < K)
        put(&tb[tm.rank * kLine + 2 * k + h], h ? high_word(s, tag) : low_word(s, tag));
    }
    // lane 8 g + j: word j of leader g, and word 8 + j % 2 (the fifth value's)
    double r[2] = {0.0, 0.0};
    const int j = l & 7;
    word_t a[K > 4 ? 2 : 1];
    if (!poll_words(tb + (l >> 3) * kLine + j, 8 - (j & 6), j < 2 * K, tag, tm.abort, a))
      sh.bad = 1;
    r[0] = join_words(a[0]);
    if constexpr (K > 4) r[1] = join_words(a[1]);
    double s = fold32(r[0], r[1]);
    s = fold16(s, s);
    s += dpp<kDppRor8>(s);
    if ((l & 57) == 0 && (l >> 1) < K) sh.total[par][0][l >> 1] = s;
    if (K > 4 && l == 32) sh.total[par][0][K > 4 ? 4 : 0] = s;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < K; ++q) v[q] = sh.total[par][0][q];
  return sh.bad == 0;
}

}  // namespace res
}  // namespace lfgpu
