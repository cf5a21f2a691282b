// wave.h -- wave64 device helpers shared by the kernel files.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.h"

namespace sme {

constexpr int kWave = 64;

// Orders the LDS accesses of a wave: every lane's earlier accesses complete
// before any lane's later ones.
__device__ __forceinline__ void WaveSync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ unsigned long long WaveSum(unsigned long long v) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// Exclusive prefix sum over the wave's lanes; *total gets the sum.
__device__ __forceinline__ uint32_t WavePrefix(uint32_t v, int lane, uint32_t* total) {
  uint32_t s = v;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t y = __shfl_up(s, o);
    if (lane >= o) s += y;
  }
  *total = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(s), kWave - 1));
  return s - v;
}

// A sum and where it goes (nullptr, the same for all threads: nowhere).
struct Into {
  unsigned long long* p;
  unsigned long long v;
};

// Adds each sum's v over the workgroup of kThr threads to its *p.  Every
// thread must reach it.  One atomic instruction per workgroup, thread n for
// sum n: the counters share a line, and device atomics to it complete about 6
// ns apart (3.5e6 paths counted by 55,000 waves: 0.67 ms of 0.70 were spent
// there; 2,048 workgroups with three instructions each: 37 us).
template <int kThr, class... T>
__device__ __forceinline__ void BlockAdd(T... sums) {
  constexpr int N = sizeof...(T);
  __shared__ unsigned long long part[N][kThr / kWave];
  const Into in[N] = {sums...};
  __syncthreads();  // an earlier call's readers are done
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const unsigned long long v = WaveSum(in[n].v);
    if ((threadIdx.x & (kWave - 1)) == 0) part[n][threadIdx.x / kWave] = v;
  }
  __syncthreads();
  if (threadIdx.x < N) {
    unsigned long long* p = nullptr;
#pragma unroll
    for (int n = 0; n < N; ++n)
      if (static_cast<int>(threadIdx.x) == n) p = in[n].p;
    unsigned long long v = 0;
    for (int w = 0; w < kThr / kWave; ++w) v += part[threadIdx.x][w];
    if (p && v) atomicAdd(p, v);
  }
}

// The same by each wave alone, for kernels whose waves end at very different
// times: a wave that waits for its workgroup keeps its place from the next one
// (the pair counts of the solar square on R-MAT scale 12: 25.0 against 23.7 ms).
template <class... T>
__device__ __forceinline__ void WaveAdd(T... sums) {
  constexpr int N = sizeof...(T);
  const Into in[N] = {sums...};
  const int lane = threadIdx.x & (kWave - 1);
  unsigned long long* p = nullptr;
  unsigned long long mine = 0;
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const unsigned long long v = WaveSum(in[n].v);
    if (lane == n) {
      p = in[n].p;
      mine = v;
    }
  }
  if (p && mine) atomicAdd(p, mine);
}

constexpr unsigned long long kNoBucket = ~0ull;

// Bucket of start vertex v: largest k with bounds[k] <= v.
__device__ __forceinline__ unsigned long long BucketOf(const BucketRef& b, uint32_t v) {
  if (b.table) return b.table[v - b.base];
  uint64_t lo = 0, hi = b.nbuckets - 1;
  while (lo < hi) {
    const uint64_t mid = (lo + hi + 1) >> 1;
    if (b.bounds[mid] <= v)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// Per-wave running bucket sum (wave-uniform).  Bucket counts are added
// into it while the wave's keys stay on one bucket and written with one
// atomic when the bucket changes, so a wave issues about one atomic per
// bucket it touches instead of one per chunk (a few buckets would otherwise
// serialize every wave on the same counters).
struct BucketAcc {
  unsigned long long key;
  unsigned long long sum;
};

__device__ __forceinline__ void BucketFlush(const BucketRef& b, BucketAcc* acc) {
  if ((threadIdx.x & (kWave - 1)) == 0 && acc->sum && acc->key != kNoBucket)
    atomicAdd(b.counts + acc->key, acc->sum);
  acc->key = kNoBucket;
  acc->sum = 0;
}

// Adds each lane's value under its bucket key (keys non-decreasing across
// the wave; kNoBucket for lanes with nothing).  Must be reached by all 64
// lanes.  Runs before the wave's last bucket are written at once; the last
// one stays in the accumulator.
__device__ __forceinline__ void BucketAccAdd(const BucketRef& b, BucketAcc* acc, unsigned long long key,
                                             unsigned long long val) {
  const int lane = threadIdx.x & (kWave - 1);
  if (__ballot(key != kNoBucket && key != acc->key) == 0) {
    acc->sum += WaveSum(val);
    return;
  }
  BucketFlush(b, acc);
  unsigned long long v = val;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const unsigned long long y = __shfl_up(v, o);
    const unsigned long long k2 = __shfl_up(key, o);
    if (lane >= o && k2 == key) v += y;
  }
  const unsigned long long next = __shfl_down(key, 1);
  const bool run_end = lane == kWave - 1 || next != key;
  const unsigned long long live = __ballot(key != kNoBucket);  // not 0: some key differed from acc
  const int last = kWave - 1 - __clzll(static_cast<long long>(live));
  const unsigned long long last_key = __shfl(key, last);
  const unsigned long long last_sum = __shfl(v, last);
  if (run_end && key != kNoBucket && key != last_key && v) atomicAdd(b.counts + key, v);
  acc->key = last_key;
  acc->sum = last_sum;
}

}  // namespace sme
