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
// than kWaitTicks raises the team's abort flag and leaves, the others see the
// flag in their own waits and leave too.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace lfgpu {
namespace res {

typedef unsigned long long word_t;

constexpr int kThreads = 512;  // 8 wavefronts: 256 registers per lane
constexpr int kWaves = kThreads / 64;
constexpr int kMaxTeam = 256;  // workgroups of a team (one leader thread per member)
constexpr int kSums = 5;       // values of one team sum
// Teams of fewer workgroups read every member's partial sums in every
// workgroup (one hop); larger ones let kLeaders workgroups sum them and
// publish the totals (two hops).  One hop costs 2.6 us with one workgroup (to
// memory and back, five values), 3.9 with 64, 5.0 with 128 and 6.6 with 256,
// which poll 256 x 10 words each; the second hop costs about 1.7.
constexpr int kFlatTeam = 64;
constexpr int kLeaders = 8;
constexpr uint64_t kWaitTicks = 400000000ull;  // 4 s of the 100 MHz real-time clock

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
  int *abort;
  uint64_t t0 = 0;
  uint32_t polls = 0;
  __device__ __forceinline__ explicit Wait(int *a) : abort(a) {}
  __device__ __forceinline__ bool more() {
    if ((++polls & 255u) != 0) return true;
    const uint64_t now = wall_clock64();
    if (t0 == 0) t0 = now;
    if (__hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
    if (now - t0 > kWaitTicks) {
      __hip_atomic_store(abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
    return true;
  }
};

// One step of a wavefront sum: v + (v of the lane that CTRL names, 0 where
// there is none or ROWS masks the row out).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, false);
  return v + __hiloint2double(hi, lo);
}
// Sum over the wavefront, valid in lane 63 (row shifts by 1, 2, 4, 8, then
// the row broadcasts; a fixed order).  Register moves only: the shuffle form
// goes through LDS and costs about 0.3 us for five values.
__device__ __forceinline__ double wave_sum63(double v) {
  v = dpp_add<0x111, 0xf>(v);
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);
  v = dpp_add<0x143, 0xc>(v);
  return v;
}

// Workgroup-shared scratch of the team sums.
struct SumLds {
  double part[2][kWaves][kSums];
  double lead[2][4][kSums];
  double total[2][kSums];
  int bad;
};

// words of the team sums' buffers
constexpr size_t kPartWords = (size_t)2 * 2 * kSums * kMaxTeam;
constexpr size_t kTotalWords = (size_t)2 * kLeaders * 2 * kSums;
// LDS a resident kernel may take dynamically (beside SumLds)
constexpr size_t kLdsDynamic = 160 * 1024 - (sizeof(SumLds) + 1023) / 1024 * 1024;

// The team as one workgroup sees it.
struct Team {
  int rank, size;
  word_t *part;   // [2][2 kSums][size] partial sums of every member
  word_t *total;  // [2][kLeaders][2 kSums] totals, one copy per leader
  int *abort;
  uint32_t tag;   // number of the last team sum
};

// Sums v over all threads of the team; every thread of every workgroup gets
// the same bits: wavefronts in order within a workgroup, then the members'
// partials in a fixed tree over their ranks.  Returns false when the team has
// been aborted (in every thread of the workgroup).  Contains workgroup
// barriers: LDS written before the call is visible after it.  All threads run
// `meanwhile` between the first of them, when the workgroup's partials are
// about to go out, and the wait for the team; it must leave to itself the
// threads that have a part in the sum: the first wavefront, and the first
// kMaxTeam threads where sums_members() holds.
__device__ __forceinline__ bool sums_members(const Team &tm) {
  return tm.size < kFlatTeam || tm.rank < kLeaders;
}
template <int K, class F>
__device__ __forceinline__ bool team_sum(Team &tm, SumLds &sh, double (&v)[K], F &&meanwhile) {
  static_assert(K <= kSums, "too many sums");
  const int t = threadIdx.x, w = t >> 6, l = t & 63;
  const uint32_t tag = ++tm.tag;
  const int par = (int)(tag & 1u);
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = wave_sum63(v[k]);
  if (l == 63)
#pragma unroll
    for (int k = 0; k < K; ++k) sh.part[par][w][k] = v[k];
  __syncthreads();
  if (tm.size == 1) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      double s = sh.part[par][0][k];
#pragma unroll
      for (int q = 1; q < kWaves; ++q) s += sh.part[par][q][k];
      v[k] = s;
    }
    return true;
  }
  word_t *pb = tm.part + (size_t)par * 2 * kSums * tm.size;
  if (t < 2 * K) {
    const int k = t >> 1;
    double s = sh.part[par][0][k];
#pragma unroll
    for (int q = 1; q < kWaves; ++q) s += sh.part[par][q][k];
    put(&pb[(size_t)t * tm.size + tm.rank], (t & 1) ? high_word(s, tag) : low_word(s, tag));
  }
  meanwhile();
  const bool flat = tm.size < kFlatTeam;
  if (sums_members(tm)) {
    if (t < kMaxTeam) {
      double r[K];
#pragma unroll
      for (int k = 0; k < K; ++k) r[k] = 0.0;
      if (t < tm.size) {
        word_t a[2 * K];
        Wait wait(tm.abort);
        bool ok;
        do {
          ok = true;
#pragma unroll
          for (int k = 0; k < 2 * K; ++k) a[k] = get(&pb[(size_t)k * tm.size + t]);
#pragma unroll
          for (int k = 0; k < 2 * K; ++k) ok = ok && tagged(a[k], tag);
        } while (!ok && wait.more());
        if (!ok) sh.bad = 1;
#pragma unroll
        for (int k = 0; k < K; ++k) r[k] = from_words(a[2 * k], a[2 * k + 1]);
      }
#pragma unroll
      for (int k = 0; k < K; ++k) r[k] = wave_sum63(r[k]);
      if (l == 63)
#pragma unroll
        for (int k = 0; k < K; ++k) sh.lead[par][w][k] = r[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
      double s = sh.lead[par][0][k];
#pragma unroll
      for (int q = 1; q < kMaxTeam / 64; ++q) s += sh.lead[par][q][k];
      v[k] = s;
    }
    if (!flat && t < 2 * K) {
      double s = v[0];
#pragma unroll
      for (int k = 1; k < K; ++k)
        if ((t >> 1) == k) s = v[k];
      put(&tm.total[((size_t)par * kLeaders + tm.rank) * 2 * kSums + t],
          (t & 1) ? high_word(s, tag) : low_word(s, tag));
    }
    return sh.bad == 0;
  }
  if (t < 2 * K) {
    const word_t *src =
        &tm.total[((size_t)par * kLeaders + (tm.rank & (kLeaders - 1))) * 2 * kSums + t];
    word_t a;
    Wait wait(tm.abort);
    bool ok;
    do {
      a = get(src);
      ok = tagged(a, tag);
    } while (!ok && wait.more());
    if (!ok) sh.bad = 1;
    // the payload halves of one value sit in neighbouring lanes
    reinterpret_cast<uint32_t *>(&sh.total[par][0])[t] = (uint32_t)(a >> 32);
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = sh.total[par][k];
  return sh.bad == 0;
}

}  // namespace res
}  // namespace lfgpu
