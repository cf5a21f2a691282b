// walk.h -- a wave walks the adjacency lists its lanes hold.
#pragma once

#include "wave.h"

namespace sme {

__device__ __forceinline__ uint32_t WaveLane32(uint32_t v, uint32_t lane) {
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), static_cast<int>(lane)));
}

__device__ __forceinline__ uint64_t WaveLane64(uint64_t v, uint32_t lane) {
  return (static_cast<uint64_t>(WaveLane32(static_cast<uint32_t>(v >> 32), lane)) << 32) |
         WaveLane32(static_cast<uint32_t>(v), lane);
}

constexpr uint32_t kFlight = 4;                   // loads a lane keeps in flight
constexpr uint32_t kWalkStep = kFlight * kWave;  // entries per step

// Per-wave scratch of WalkLists.
struct WalkLds {
  uint64_t from[kWave];  // k-th list: its first entry less its first item
  uint32_t mid[kWave];
  union {
    uint8_t flag[kWalkStep];
    uint32_t clear[kWave];
  };
};
static_assert(kWalkStep == 4 * kWave, "a lane clears one word of flags");
constexpr uint32_t kLongList = kWalkStep;  // lists from here on are streamed one by one

// Calls f(w, t, mid) for every entry e (w = cols[e]; t = tri[e] with kT) of the
// lanes' lists cols[lb, lb + len): long lists one after another, the others
// together as one flat list of items, kWalkStep entries per step with all of a
// step's loads issued before the first use.  f may use no wave operation.
// (Streaming lists from 48 entries on one by one, and 64 items per step, left
// one or two loads in flight: 59 against 44 ms for the tile kernel of the house
// on R-MAT scale 19, 3.1 against 2.3 ms for the light 4-cycle kernel.)
template <bool kT, class F>
__device__ __forceinline__ void WalkLists(const uint32_t* cols, const uint32_t* tri, uint64_t lb, uint32_t len,
                                          uint32_t mid, WalkLds& s, int lane, F f) {
  for (unsigned long long m = __ballot(len >= kLongList); m; m &= m - 1) {
    const uint32_t src = static_cast<uint32_t>(__builtin_ctzll(m));
    const uint64_t b = WaveLane64(lb, src);
    const uint32_t n = WaveLane32(len, src), md = WaveLane32(mid, src);
    for (uint32_t i = static_cast<uint32_t>(lane); i < n; i += kWalkStep) {
      uint32_t w[kFlight], t[kFlight];
#pragma unroll
      for (uint32_t h = 0; h < kFlight; ++h) {
        const bool in = i + h * kWave < n;
        w[h] = in ? cols[b + i + h * kWave] : 0u;
        t[h] = kT && in ? tri[b + i + h * kWave] : 0u;
      }
#pragma unroll
      for (uint32_t h = 0; h < kFlight; ++h)
        if (i + h * kWave < n) f(w[h], t[h], md);
    }
  }
  const uint32_t items = len < kLongList ? len : 0;
  uint32_t total;
  const uint32_t start = WavePrefix(items, lane, &total);
  if (total == 0) return;
  const unsigned long long upto = ~0ull >> (kWave - 1 - lane);
  const unsigned long long work = __ballot(items != 0);
  WaveSync();  // the previous walk's readers are done
  if (items) {
    const int at = static_cast<int>(__popcll(work & (upto >> 1)));
    s.from[at] = lb - start;
    s.mid[at] = mid;
  }
  uint32_t before = 0;  // lists that started before this step
  for (uint32_t t0 = 0; t0 < total; t0 += kWalkStep) {
    s.clear[lane] = 0;
    WaveSync();
    if (items && start >= t0 && start - t0 < kWalkStep) s.flag[start - t0] = 1;
    WaveSync();
    uint32_t w[kFlight], t[kFlight], md[kFlight];
#pragma unroll
    for (uint32_t h = 0; h < kFlight; ++h) {
      w[h] = t[h] = md[h] = 0;
      if (t0 + h * kWave >= total) continue;
      const unsigned long long starts = __ballot(s.flag[h * kWave + lane] != 0);
      const uint32_t own = before + static_cast<uint32_t>(__popcll(starts & upto)) - 1;
      before += static_cast<uint32_t>(__popcll(starts));
      const uint32_t it = t0 + h * kWave + static_cast<uint32_t>(lane);
      if (it < total) {
        const uint64_t e = s.from[own] + it;
        w[h] = cols[e];
        if (kT) t[h] = tri[e];
        md[h] = s.mid[own];
      }
    }
#pragma unroll
    for (uint32_t h = 0; h < kFlight; ++h)
      if (t0 + h * kWave + static_cast<uint32_t>(lane) < total) f(w[h], t[h], md[h]);
  }
}

}  // namespace sme
