// Persistent Krylov solves: the pieces a single launch needs to iterate on
// its own. Every workgroup of such a launch is resident (the launch is
// cooperative), keeps its part of the vectors in registers and LDS, and meets
// the others twice per iteration in a round: each workgroup publishes its
// partial sums and reads everyone's.
//
// A round needs no fence and waits for no store: everything the workgroups
// tell each other goes out as 8-byte words of 32 value bits and the round's
// tag, stored and polled at agent scope (past the XCD's own L2), so a word
// that shows the tag also holds its value. An L2 writeback fence instead costs
// about 35 ns per workgroup and launch; waiting for exchanged values' stores
// before publishing, and reading them after, two more trips to memory per
// round.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.hpp"

namespace msim {

constexpr int kPersistThreads = 512;
constexpr uint32_t kRoundBlocks = 256;  // most workgroups of a round
constexpr int kRoundWords = 4;          // words a workgroup publishes in one round, at most
// Two generations by tag parity: a workgroup can be one round ahead of the
// slowest, never two.
constexpr size_t kRoundSlots = 2ull * kRoundWords * kRoundBlocks;
// A thread that waits this long for words (100 MHz ticks: 0.2 s, where a round
// takes microseconds) gives the launch up; the others then do too, so the launch
// always ends, and its caller starts over without it. Short, because the halo
// entries of a wide grid are waited for one after the other, some 30 at most.
constexpr uint64_t kRoundTicks = 20'000'000ull;
constexpr uint32_t kRoundStalled = 6;  // failure of a launch given up that way

__device__ inline void word_store(uint64_t* at, uint32_t tag, uint32_t bits) {
  __hip_atomic_store(at, (static_cast<uint64_t>(tag) << 32) | bits, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline uint64_t word_load(const uint64_t* at) {
  return __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline bool word_has(uint64_t w, uint32_t tag) {
  return static_cast<uint32_t>(w >> 32) == tag;
}

// A value per entry of an exchange array of `n` entries: one word of a float,
// two (n apart) of a double.
template <typename T>
struct Exchange {
  static constexpr int kWords = sizeof(T) / 4;
  uint64_t* words;
  uint32_t n;
  __device__ void put(uint32_t i, uint32_t tag, T v) const {
    if constexpr (kWords == 1) {
      word_store(words + i, tag, __float_as_uint(v));
    } else {
      const uint64_t bits = static_cast<uint64_t>(__double_as_longlong(v));
      word_store(words + i, tag, static_cast<uint32_t>(bits));
      word_store(words + n + i, tag, static_cast<uint32_t>(bits >> 32));
    }
  }
  __device__ void load(uint32_t i, uint64_t (&w)[kWords]) const {
#pragma unroll
    for (int k = 0; k < kWords; ++k) w[k] = word_load(words + static_cast<size_t>(k) * n + i);
  }
  __device__ static bool has(const uint64_t (&w)[kWords], uint32_t tag) {
    bool all = true;
#pragma unroll
    for (int k = 0; k < kWords; ++k) all = all && word_has(w[k], tag);
    return all;
  }
  __device__ static T value(const uint64_t (&w)[kWords]) {
    if constexpr (kWords == 1) {
      return __uint_as_float(static_cast<uint32_t>(w[0]));
    } else {
      return __longlong_as_double(
          static_cast<long long>((w[1] << 32) | (w[0] & 0xffffffffull)));
    }
  }
};

// Sum over a wavefront, in its lane 63: quads, half rows and rows by DPP
// moves, then the rows. A fixed pattern; a sixth of the latency of shuffles
// through LDS.
template <int kControl>
__device__ inline double dpp_add(double v) {
  const uint64_t bits = static_cast<uint64_t>(__double_as_longlong(v));
  const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(bits), kControl, 0xf, 0xf, true);
  const int hi =
      __builtin_amdgcn_update_dpp(0, static_cast<int>(bits >> 32), kControl, 0xf, 0xf, true);
  return v + __longlong_as_double(static_cast<long long>(
                 (static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) |
                 static_cast<uint32_t>(lo)));
}

__device__ inline double wave_sum_last(double v) {
  v = dpp_add<0xb1>(v);   // quad_perm 1 0 3 2
  v = dpp_add<0x4e>(v);   // quad_perm 2 3 0 1
  v = dpp_add<0x141>(v);  // mirror within half rows
  v = dpp_add<0x140>(v);  // mirror within rows
  v = dpp_add<0x142>(v);  // lane 15 of each row to the next row
  v = dpp_add<0x143>(v);  // lane 31 to rows 2 and 3
  return v;
}

struct RoundLds {
  double mine[2 * (kPersistThreads / kWave)];
  double all[2 * (kPersistThreads / kWave)];
  int stalled;
};

// Polls: `issue` loads words, `done` says whether all of them show their tag.
// The pace of this loop is the rounds' and moves with any change of it: asking
// among the ticks whether another thread has given up costs the FP32 pressure
// iterations of 1024x512 sites 7 %, an unused argument of the kernel 4 %.
template <class Issue, class Done>
__device__ inline void poll_words(RoundLds& L, Issue&& issue, Done&& done) {
  uint64_t since = 0;
  for (uint32_t spins = 1;; ++spins) {
    issue();
    if (done()) return;
    if ((spins & 255u) == 0) {
      const uint64_t now = wall_clock64();
      if (since == 0) since = now;
      if (now - since > kRoundTicks) {
        L.stalled = 1;
        return;
      }
    }
  }
}

// v[k] becomes the sum over every thread of every workgroup, the same bits in
// each: waves in order within a workgroup, then workgroups by index in one
// fixed tree. Consecutive rounds take consecutive tags. The words `issue`
// loads are polled for along with the sums. False: stalled.
template <int K, class Issue, class Done>
__device__ inline bool round_sums(double (&v)[K], uint64_t* slots, uint32_t tag, RoundLds& L,
                                  Issue&& issue, Done&& done) {
  static_assert(2 * K <= kRoundWords);
  constexpr int kWaves = kPersistThreads / kWave;
  const int t = threadIdx.x, wave = t / kWave;
  const bool last = (t & (kWave - 1)) == kWave - 1;
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = wave_sum_last(v[k]);
  if (last) {
#pragma unroll
    for (int k = 0; k < K; ++k) L.mine[k * kWaves + wave] = v[k];
  }
  __syncthreads();
  uint64_t* base = slots + static_cast<size_t>(tag & 1u) * kRoundWords * kRoundBlocks;
  if (t < 2 * K) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s += L.mine[(t / 2) * kWaves + w];
    const uint64_t bits = static_cast<uint64_t>(__double_as_longlong(s));
    word_store(base + t * kRoundBlocks + blockIdx.x, tag,
               static_cast<uint32_t>((t & 1) != 0 ? bits >> 32 : bits));
  }
  uint64_t w[2 * K];
#pragma unroll
  for (int j = 0; j < 2 * K; ++j) w[j] = static_cast<uint64_t>(tag) << 32;  // 0.0
  const bool reads = t < static_cast<int>(gridDim.x);
  poll_words(
      L,
      [&] {
        if (reads) {
#pragma unroll
          for (int j = 0; j < 2 * K; ++j) w[j] = word_load(base + j * kRoundBlocks + t);
        }
        issue();
      },
      [&] {
        bool here = done();
#pragma unroll
        for (int j = 0; j < 2 * K; ++j) here = here && word_has(w[j], tag);
        return here;
      });
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const double got = wave_sum_last(__longlong_as_double(
        static_cast<long long>((w[2 * k + 1] << 32) | (w[2 * k] & 0xffffffffull))));
    if (last) L.all[k * kWaves + wave] = got;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < K; ++k) {
    double s = 0.0;
#pragma unroll
    for (int w2 = 0; w2 < kWaves; ++w2) s += L.all[k * kWaves + w2];
    v[k] = s;
  }
  return L.stalled == 0;
}

}  // namespace msim
