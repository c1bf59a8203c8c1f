// wave.h — wavefront-level helpers (64-lane CDNA wavefronts).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dyn_math.h"

namespace dyn {

constexpr int kWaveLanes = 64;

// A unique rank for every lane with valid set among the lanes that share its
// key: counters[key] grows by the number of such lanes.  Lanes of one key
// take consecutive ranks from one atomic, and the atomics of all the wave's
// keys are issued together (one round trip, whatever the number of keys).
// Every lane of the wave must call it.  Ranks depend on the order in which
// waves reach the counters.
__device__ __forceinline__ uint32_t wave_rank(uint32_t key, bool valid,
                                              uint32_t* __restrict__ counters) {
  const int lane = (int)(threadIdx.x & (kWaveLanes - 1));
  unsigned long long todo = __ballot(valid);
  int leader = lane;
  unsigned long long peers = 0ull;
  while (todo) {
    const int l = __ffsll((long long)todo) - 1;
    const uint32_t kl = __shfl(key, l, kWaveLanes);
    const unsigned long long p = __ballot(key == kl) & todo;
    if ((p >> lane) & 1ull) {
      leader = l;
      peers = p;
    }
    todo &= ~p;
  }
  uint32_t base = 0;
  if (peers && leader == lane) base = atomicAdd(&counters[key], (uint32_t)__popcll(peers));
  base = __shfl(base, leader, kWaveLanes);
  return base + (uint32_t)__popcll(peers & ((1ull << lane) - 1ull));
}

// Adds e to M[key] (2⁻³² fixed point) for every lane with key ≥ 0: one
// atomic for the wave when all such lanes share the key.  All lanes of the
// wave must be active.
__device__ __forceinline__ void wave_add_fx(int64_t* __restrict__ M, int key, double e) {
  const unsigned long long live = __ballot(key >= 0);
  if (!live) return;
  const int kf = __shfl(key, __ffsll((long long)live) - 1, kWaveLanes);
  if (__ballot(key >= 0 && key != kf) == 0ull) {
    double x = key >= 0 ? e : 0.0;
    for (int m = 1; m < kWaveLanes; m <<= 1) x += __shfl_xor(x, m, kWaveLanes);
    if ((threadIdx.x & (kWaveLanes - 1)) == 0)
      atomicAdd(reinterpret_cast<unsigned long long*>(M + kf),
                (unsigned long long)dyn_fx64(x));
  } else if (key >= 0) {
    atomicAdd(reinterpret_cast<unsigned long long*>(M + key),
              (unsigned long long)dyn_fx64(e));
  }
}

}  // namespace dyn
