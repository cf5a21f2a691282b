// paths.hip -- counting levels whose paths share all but one adjacency list
// (PathRunArgs in kernels.h).
//
// The reference intersects every path's lists from scratch, one warp per path
// (src/gpu/utils/ops/GPSMBinSearch.cuh:36-63).  Paths come ordered by the
// vertices matched first, so consecutive ones share every list but that of the
// vertex matched last: the shared intersection is built once per run of paths
// as an LDS bitmap, and each path streams its own list against it.
#include "kernels.h"
#include "walk.h"
#include "wave.h"

namespace sme {

namespace {

using u64 = unsigned long long;

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr uint32_t kNone = 0xffffffffu;  // (no vertex)

__device__ __forceinline__ uint32_t Gather(const ColSet& cs, int w, uint64_t p) {
  const uint32_t* col = cs.inst[w];
  return col ? col[p] : cs.iota[w] + static_cast<uint32_t>(p);
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

__device__ __forceinline__ bool Holds(const uint32_t* cols, uint32_t b, uint32_t n, uint32_t x) {
  const uint64_t at = Lower(cols, b, b + n, x);
  return at < b + n && cols[at] == x;
}

// Calls f(x) for every value of cols[b, b + n), 64 consecutive ones per load, four
// loads in flight, kDeep sixteen while the list is long: one wave reads a hub's
// list, and few others hide its waits (diamonds from the last 2 % of 30,000
// vertices, 3 of them joined to 21,000: 0.29 ms by fours, 0.16 by sixteens, 0.14 on
// the item schedule).
constexpr uint32_t kLongStep = 16 * kWave;

template <bool kDeep, class F>
__device__ __forceinline__ void Stream(const uint32_t* cols, uint64_t b, uint32_t n, int lane, F f) {
  uint32_t i = static_cast<uint32_t>(lane);
  if (kDeep)
    for (; i < n / kLongStep * kLongStep; i += kLongStep) {
      uint32_t x[16];
#pragma unroll
      for (uint32_t h = 0; h < 16; ++h) x[h] = cols[b + i + h * kWave];
#pragma unroll
      for (uint32_t h = 0; h < 16; ++h) f(x[h]);
    }
  for (; i < n; i += 4 * kWave) {
    uint32_t x[4];
#pragma unroll
    for (uint32_t h = 0; h < 4; ++h) x[h] = i + h * kWave < n ? cols[b + i + h * kWave] : 0u;
#pragma unroll
    for (uint32_t h = 0; h < 4; ++h)
      if (i + h * kWave < n) f(x[h]);
  }
}

// A wave takes a.group (at most 64) consecutive paths at a time.  A run of paths
// is counted in one of two ways:
//   bitmaps: one holds the shared list (of two, the shorter), the other the
//     intersection of both; the bits set for a run are taken back by walking the
//     same lists.  Each path streams its own list against them; one whose own
//     list is over kOwnRatio times the shortest shared one walks that and
//     searches its own.
//   search: every path's shortest list is walked and the others are searched,
//     the lists of all such paths together as one flat list of items.
// Bitmaps cost what the shared lists hold, whatever is looked up in them, and a
// chain of waits per run and per path; a search costs each value walked two
// bisections.  In entries streamed: kRunCost, kPathCost and kSearchCost.  Level
// engine calls of which these levels are a part, on the item schedule, with
// bitmaps alone and with the rule (ms; the rule's numbers a factor of two either
// way change these by up to a quarter, mostly by a few percent):
//   near-5-clique, 1 hub over 32,768 ids, 65,536 edges   0.44   3.8    0.31
//   near-5-clique, 2 hubs over half of 32,768 ids        1.37   4.1    0.55
//   chordal roof, the same                               3.3    6.3    1.8
//   near-5-clique, G(20,000, 1e5)                        0.33   0.37   0.23
//   near-5-clique, G(8,192, 4e5)                         2.1    1.19   1.16
//   near-5-clique, R-MAT 13                             16.9    2.00   1.95
//
// Bound by the latency of the list loads and the LDS bit tests.  Near-5-clique
// on R-MAT scale 13, its two path-count levels (3.5e6 paths): 1.6 ms, where the
// item schedule, whose 64-item chunks mostly straddle paths, bisected lists in
// memory for every item (15.2 ms).  Both bitmaps in LDS limit the ids: 1 KB
// each up to 8,192, 4 KB up to 32,768; beyond that the item schedule stays.
constexpr uint32_t kSearchCost = 12, kRunCost = 512, kPathCost = 32;

template <uint32_t kWords>
union RunLds {
  uint32_t bits[2][kWords];  // zero between runs
  struct {
    WalkLds walk;
    // per path: the lists searched, the values passed over, the count
    uint32_t a_beg[kWave], a_len[kWave], b_beg[kWave], b_len[kWave], ne[2][kWave], hits[kWave];
  } s;
};

template <uint32_t kWords>
__global__ __launch_bounds__(kThreads) void PathRunKernel(PathRunArgs a) {
  __shared__ RunLds<kWords> lds_all[kWaves];
  const int lane = threadIdx.x & (kWave - 1);
  RunLds<kWords>& lds = lds_all[threadIdx.x / kWave];
  uint32_t* first = lds.bits[0];
  uint32_t* both = lds.bits[1];
  const uint64_t wave = (blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x) / kWave;
  const uint64_t nwaves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  const bool two = a.nshared == 2;
  constexpr bool kDeep = kWords > 256;  // (the others' lists are at most 8,192 long; it costs them a third of their waves)
  const uint32_t* shared = two ? both : first;
  for (uint32_t k = lane; k < kWords; k += kWave) first[k] = both[k] = 0;
  WaveSync();
  u64 total = 0;
  BucketAcc bacc{kNoBucket, 0};
  for (uint64_t p0 = wave * a.group; p0 < a.npaths; p0 += nwaves * a.group) {
    const uint64_t p = p0 + lane;
    const bool live = p < a.npaths && static_cast<uint32_t>(lane) < a.group;
    uint32_t s0 = 0, s1 = 0, len = 0, ne0 = kNone, ne1 = kNone, wlo = 0, whi = 0xffffffffu;
    // (at most 32,768 sorted lists of as many ids: entries are counted in 32 bits)
    uint32_t lb = 0, b0 = 0, n0 = 0, b1 = 0, n1 = 0;
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
      uint64_t b = a.rp[own], e = a.rp[own + 1];
      if (lo >= hi) {
        e = b;
      } else {
        if (lo > 0) b = Lower(a.cols, b, e, static_cast<uint32_t>(lo));
        if (hi <= 0xffffffffull) e = Lower(a.cols, b, e, static_cast<uint32_t>(hi));
      }
      lb = static_cast<uint32_t>(b);
      len = static_cast<uint32_t>(e - b);
      wlo = static_cast<uint32_t>(lo <= 0xffffffffull ? lo : 0xffffffffull);
      whi = static_cast<uint32_t>(hi <= 0xffffffffull ? hi : 0xffffffffull);  // (no vertex is 2^32 - 1)
      if (a.nne > 0) ne0 = Gather(a.cs, a.ne_v[0], p);
      if (a.nne > 1) ne1 = Gather(a.cs, a.ne_v[1], p);
      b0 = static_cast<uint32_t>(a.rp[s0]);
      n0 = static_cast<uint32_t>(a.rp[s0 + 1]) - b0;
      if (two) {
        b1 = static_cast<uint32_t>(a.rp[s1]);
        n1 = static_cast<uint32_t>(a.rp[s1 + 1]) - b1;
        if (n1 < n0) {  // the shorter first
          const uint32_t tb = b0, tn = n0;
          b0 = b1;
          n0 = n1;
          b1 = tb;
          n1 = tn;
        }
      }
    }
    const uint32_t up0 = __shfl_up(s0, 1), up1 = __shfl_up(s1, 1);
    const u64 alive = __ballot(live);
    u64 runs = __ballot(live && (lane == 0 || up0 != s0 || up1 != s1));
    // what a path looks up when its lists are searched, and what it streams past
    // the bitmaps: sums over the lanes before
    const uint32_t walked = len < n0 ? len : n0;
    const uint32_t passed = len > kOwnRatio * n0 ? n0 : len;
    uint32_t sum_walked, sum_passed;
    const uint32_t pre_walked = WavePrefix(walked, lane, &sum_walked);
    const uint32_t pre_passed = WavePrefix(passed, lane, &sum_passed);
    u64 searched = 0;  // paths that are
    uint32_t mine = 0;  // this lane's path's count
    while (runs) {
      const uint32_t q0 = static_cast<uint32_t>(__builtin_ctzll(runs));
      runs &= runs - 1;
      const uint32_t q1 = runs ? static_cast<uint32_t>(__builtin_ctzll(runs))
                               : kWave - static_cast<uint32_t>(__clzll(static_cast<long long>(alive)));
      const uint32_t rn0 = WaveLane32(n0, q0), rn1 = WaveLane32(n1, q0);
      const uint32_t search = (q1 < kWave ? WaveLane32(pre_walked, q1) : sum_walked) - WaveLane32(pre_walked, q0);
      if (search == 0) continue;  // (no path of the run has a candidate)
      const uint32_t stream = (q1 < kWave ? WaveLane32(pre_passed, q1) : sum_passed) - WaveLane32(pre_passed, q0);
      if (search * kSearchCost < 2 * rn0 + rn1 + stream + kRunCost + kPathCost * (q1 - q0)) {
        searched |= (q1 < kWave ? (1ull << q1) - 1 : ~0ull) & ~((1ull << q0) - 1);
        continue;
      }
      const uint32_t rb0 = WaveLane32(b0, q0), rb1 = WaveLane32(b1, q0);
      WaveSync();
      Stream<kDeep>(a.cols, rb0, rn0, lane, [&](uint32_t x) { atomicOr(first + (x >> 5), 1u << (x & 31)); });
      WaveSync();
      if (two) {
        Stream<kDeep>(a.cols, rb1, rn1, lane, [&](uint32_t x) {
          if ((first[x >> 5] >> (x & 31)) & 1u) atomicOr(both + (x >> 5), 1u << (x & 31));
        });
        WaveSync();
      }
      for (uint32_t q = q0; q < q1; ++q) {
        const uint32_t n = WaveLane32(len, q);
        if (n == 0) continue;
        const uint32_t b = WaveLane32(lb, q);
        const uint32_t e0 = WaveLane32(ne0, q), e1 = WaveLane32(ne1, q);
        uint32_t hits = 0;
        if (n > kOwnRatio * rn0) {
          const uint32_t lo = WaveLane32(wlo, q), hi = WaveLane32(whi, q);
          Stream<kDeep>(a.cols, rb0, rn0, lane, [&](uint32_t x) {
            if (x < lo || x >= hi || !((shared[x >> 5] >> (x & 31)) & 1u)) return;
            if (x == e0 || x == e1) return;
            hits += Holds(a.cols, b, n, x) ? 1u : 0u;
          });
        } else {
          Stream<kDeep>(a.cols, b, n, lane, [&](uint32_t x) {
            if (x == e0 || x == e1) return;
            hits += (shared[x >> 5] >> (x & 31)) & 1u;
          });
        }
        hits = static_cast<uint32_t>(WaveSum(hits));
        if (static_cast<uint32_t>(lane) == q) mine = hits;
      }
      WaveSync();
      if (kDeep && rn0 > kWords) {
        for (uint32_t k = lane; k < kWords; k += kWave) first[k] = both[k] = 0;
      } else {
        Stream<kDeep>(a.cols, rb0, rn0, lane, [&](uint32_t x) {
          first[x >> 5] = 0;
          if (two) both[x >> 5] = 0;
        });
      }
    }
    if (searched) {
      const bool in = (searched >> lane) & 1;
      uint32_t wb = 0, wn = 0;  // the list walked
      WaveSync();
      if (in) {
        if (len <= n0) {
          wb = lb;
          wn = len;
          lds.s.a_beg[lane] = b0;
          lds.s.a_len[lane] = n0;
        } else {
          // the shorter shared list's part within the path's window
          wb = static_cast<uint32_t>(Lower(a.cols, b0, b0 + n0, wlo));
          wn = static_cast<uint32_t>(Lower(a.cols, wb, b0 + n0, whi)) - wb;
          lds.s.a_beg[lane] = lb;
          lds.s.a_len[lane] = len;
        }
        lds.s.b_beg[lane] = b1;
        lds.s.b_len[lane] = n1;
        lds.s.ne[0][lane] = ne0;
        lds.s.ne[1][lane] = ne1;
        lds.s.hits[lane] = 0;
      }
      WaveSync();
      WalkLists<false>(a.cols, nullptr, wb, wn, static_cast<uint32_t>(lane), lds.s.walk, lane,
                       [&](uint32_t x, uint32_t, uint32_t q) {
                         if (x == lds.s.ne[0][q] || x == lds.s.ne[1][q]) return;
                         if (!Holds(a.cols, lds.s.a_beg[q], lds.s.a_len[q], x)) return;
                         if (two && !Holds(a.cols, lds.s.b_beg[q], lds.s.b_len[q], x)) return;
                         atomicAdd(lds.s.hits + q, 1u);
                       });
      WaveSync();
      if (in) mine = lds.s.hits[lane];
      WaveSync();
      for (uint32_t k = lane; k < kWords; k += kWave) first[k] = both[k] = 0;
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
  PathRunArgs b = a;
  // few paths: fewer per wave, so that their runs' chains of waits lie side by side
  const uint64_t per = a.npaths / 8192;
  b.group = static_cast<uint32_t>(per < 8 ? 8 : per > kWave ? kWave : per);
  const uint64_t waves = (a.npaths + b.group - 1) / b.group;
  const uint64_t need = (waves + kWaves - 1) / kWaves;
  // 1 KB bitmaps let 32 waves share a CU, 4 KB ones 20
  if (a.n <= 8192)
    hipLaunchKernelGGL(PathRunKernel<256>, dim3(need < 4096 ? need : 4096), dim3(kThreads), 0, stream, b);
  else
    hipLaunchKernelGGL(PathRunKernel<kPathRunIds / 32>, dim3(need < 4096 ? need : 4096), dim3(kThreads), 0, stream, b);
}

}  // namespace sme
