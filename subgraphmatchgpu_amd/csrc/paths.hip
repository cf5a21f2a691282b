// paths.hip -- counting levels whose paths share all but one adjacency list
// (PathRunArgs in kernels.h).
//
// The reference intersects every path's lists from scratch, one warp per path
// (src/gpu/utils/ops/GPSMBinSearch.cuh:36-63).  Paths come ordered by the
// vertices matched first, so consecutive ones share every list but that of the
// vertex matched last: the shared intersection is built once per run of paths
// as an LDS bitmap, and each path streams its own list against it.
#include "kernels.h"
#include "wave.h"

namespace sme {

namespace {

using u64 = unsigned long long;

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;

__device__ __forceinline__ uint32_t Gather(const ColSet& cs, int w, uint64_t p) {
  const uint32_t* col = cs.inst[w];
  return col ? col[p] : cs.iota[w] + static_cast<uint32_t>(p);
}

__device__ __forceinline__ uint32_t Lane32(uint32_t v, uint32_t lane) {
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), static_cast<int>(lane)));
}

__device__ __forceinline__ uint64_t Lane64(uint64_t v, uint32_t lane) {
  return (static_cast<uint64_t>(Lane32(static_cast<uint32_t>(v >> 32), lane)) << 32) |
         Lane32(static_cast<uint32_t>(v), lane);
}

// First index in [lo, hi) with a[i] >= key.
__device__ __forceinline__ uint64_t Lower(const uint32_t* a, uint64_t lo, uint64_t hi, uint32_t key) {
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if (a[mid] < key)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// Calls f(x) for every value of cols[b, e), 64 consecutive ones per load, four
// loads in flight.
template <class F>
__device__ __forceinline__ void Stream(const uint32_t* cols, uint64_t b, uint32_t n, int lane, F f) {
  for (uint32_t i = static_cast<uint32_t>(lane); i < n; i += 4 * kWave) {
    uint32_t x[4];
#pragma unroll
    for (uint32_t h = 0; h < 4; ++h) x[h] = i + h * kWave < n ? cols[b + i + h * kWave] : 0u;
#pragma unroll
    for (uint32_t h = 0; h < 4; ++h)
      if (i + h * kWave < n) f(x[h]);
  }
}

// A wave takes 64 consecutive paths at a time.  One bitmap holds the shared
// list (of two, the shorter), the other the intersection of both; the bits set
// for a run are taken back by walking the same lists.  A path whose own list is
// over kOwnRatio times the shortest shared one walks that and searches the
// other lists instead.
//
// Bound by the latency of the list loads and the LDS bit tests.  Near-5-clique
// on R-MAT scale 13, its two path-count levels (3.5e6 paths): 1.6 ms, where the
// item schedule, whose 64-item chunks mostly straddle paths, bisected lists in
// memory for every item (15.2 ms).  Both bitmaps in LDS limit the ids: 1 KB
// each up to 8,192, 4 KB up to 32,768; beyond that the item schedule stays.
template <uint32_t kWords>
__global__ __launch_bounds__(kThreads) void PathRunKernel(PathRunArgs a) {
  __shared__ uint32_t lds_a[kWaves][kWords];
  __shared__ uint32_t lds_b[kWaves][kWords];
  const int lane = threadIdx.x & (kWave - 1);
  uint32_t* first = lds_a[threadIdx.x / kWave];
  uint32_t* both = lds_b[threadIdx.x / kWave];
  const uint64_t wave = (blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x) / kWave;
  const uint64_t nwaves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  const bool two = a.nshared == 2;
  const uint32_t* shared = two ? both : first;
  for (uint32_t k = lane; k < kWords; k += kWave) first[k] = both[k] = 0;
  WaveSync();
  u64 total = 0;
  BucketAcc bacc{kNoBucket, 0};
  for (uint64_t p0 = wave * kWave; p0 < a.npaths; p0 += nwaves * kWave) {
    const uint64_t p = p0 + lane;
    const bool live = p < a.npaths;
    uint32_t s0 = 0, s1 = 0, len = 0, ne0 = 0, ne1 = 0, wlo = 0, whi = 0xffffffffu;
    uint64_t lb = 0;
    if (live) {
      s0 = Gather(a.cs, a.shared_v[0], p);
      if (two) s1 = Gather(a.cs, a.shared_v[1], p);
      uint64_t lo = 0, hi = 0x100000000ull;
      for (int i = 0; i < a.ngt; ++i) {
        const uint64_t v = Gather(a.cs, a.gt_v[i], p) + 1ull;
        lo = v > lo ? v : lo;
      }
      for (int i = 0; i < a.nlt; ++i) {
        const uint64_t v = Gather(a.cs, a.lt_v[i], p);
        hi = v < hi ? v : hi;
      }
      const uint32_t own = Gather(a.cs, a.own_v, p);
      lb = a.rp[own];
      uint64_t le = a.rp[own + 1];
      if (lo >= hi) {
        le = lb;
      } else {
        if (lo > 0) lb = Lower(a.cols, lb, le, static_cast<uint32_t>(lo));
        if (hi <= 0xffffffffull) le = Lower(a.cols, lb, le, static_cast<uint32_t>(hi));
      }
      len = static_cast<uint32_t>(le - lb);
      wlo = static_cast<uint32_t>(lo <= 0xffffffffull ? lo : 0xffffffffull);
      whi = static_cast<uint32_t>(hi <= 0xffffffffull ? hi : 0xffffffffull);  // (no vertex is 2^32 - 1)
      if (a.nne > 0) ne0 = Gather(a.cs, a.ne_v[0], p);
      if (a.nne > 1) ne1 = Gather(a.cs, a.ne_v[1], p);
    }
    const uint32_t up0 = __shfl_up(s0, 1), up1 = __shfl_up(s1, 1);
    const u64 alive = __ballot(live);
    u64 runs = __ballot(live && (lane == 0 || up0 != s0 || up1 != s1));
    uint32_t mine = 0;  // this lane's path's count
    while (runs) {
      const uint32_t q0 = static_cast<uint32_t>(__builtin_ctzll(runs));
      runs &= runs - 1;
      const uint32_t q1 = runs ? static_cast<uint32_t>(__builtin_ctzll(runs))
                               : kWave - static_cast<uint32_t>(__clzll(static_cast<long long>(alive)));
      uint32_t v0 = Lane32(s0, q0), v1 = Lane32(s1, q0);
      uint64_t b0 = a.rp[v0], b1 = two ? a.rp[v1] : 0;
      uint32_t n0 = static_cast<uint32_t>(a.rp[v0 + 1] - b0);
      uint32_t n1 = two ? static_cast<uint32_t>(a.rp[v1 + 1] - b1) : 0;
      if (two && n1 < n0) {
        const uint64_t tb = b0;
        b0 = b1;
        b1 = tb;
        const uint32_t tn = n0;
        n0 = n1;
        n1 = tn;
      }
      WaveSync();
      Stream(a.cols, b0, n0, lane, [&](uint32_t x) { atomicOr(first + (x >> 5), 1u << (x & 31)); });
      WaveSync();
      if (two) {
        Stream(a.cols, b1, n1, lane, [&](uint32_t x) {
          if ((first[x >> 5] >> (x & 31)) & 1u) atomicOr(both + (x >> 5), 1u << (x & 31));
        });
        WaveSync();
      }
      for (uint32_t q = q0; q < q1; ++q) {
        const uint32_t n = Lane32(len, q);
        if (n == 0) continue;
        const uint64_t b = Lane64(lb, q);
        const uint32_t e0 = Lane32(ne0, q), e1 = Lane32(ne1, q);
        uint32_t hits = 0;
        if (n > kOwnRatio * n0) {
          const uint32_t lo = Lane32(wlo, q), hi = Lane32(whi, q);
          Stream(a.cols, b0, n0, lane, [&](uint32_t x) {
            if (x < lo || x >= hi || !((shared[x >> 5] >> (x & 31)) & 1u)) return;
            if ((a.nne > 0 && x == e0) || (a.nne > 1 && x == e1)) return;
            const uint64_t at = Lower(a.cols, b, b + n, x);
            hits += at < b + n && a.cols[at] == x ? 1u : 0u;
          });
        } else {
          Stream(a.cols, b, n, lane, [&](uint32_t x) {
            if ((a.nne > 0 && x == e0) || (a.nne > 1 && x == e1)) return;
            hits += (shared[x >> 5] >> (x & 31)) & 1u;
          });
        }
        hits = static_cast<uint32_t>(WaveSum(hits));
        if (static_cast<uint32_t>(lane) == q) mine = hits;
      }
      WaveSync();
      Stream(a.cols, b0, n0, lane, [&](uint32_t x) {
        first[x >> 5] = 0;
        if (two) both[x >> 5] = 0;
      });
    }
    if (live && a.out_len) a.out_len[p] = mine;
    total += mine;
    if (a.bk.bounds && a.acc) {
      const u64 key = live ? BucketOf(a.bk, Gather(a.cs, a.bk.start_v, p)) : kNoBucket;
      BucketAccAdd(a.bk, &bacc, key, mine);
    }
  }
  if (a.bk.bounds && a.acc) BucketFlush(a.bk, &bacc);
  BlockAdd<kThreads>(Into{a.acc, total}, Into{a.acc_level, total});
}

}  // namespace

void LaunchPathRuns(const PathRunArgs& a, hipStream_t stream) {
  if (a.npaths == 0) return;
  const uint64_t need = (a.npaths + kThreads - 1) / kThreads;
  // 1 KB bitmaps let 32 waves share a CU, 4 KB ones 20
  if (a.n <= 8192)
    hipLaunchKernelGGL(PathRunKernel<256>, dim3(need < 4096 ? need : 4096), dim3(kThreads), 0, stream, a);
  else
    hipLaunchKernelGGL(PathRunKernel<kPathRunIds / 32>, dim3(need < 4096 ? need : 4096), dim3(kThreads), 0, stream, a);
}

}  // namespace sme
