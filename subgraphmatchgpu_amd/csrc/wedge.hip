// wedge.hip -- 4-cycle and house counts from wedges per start vertex
// (WedgeArgs in kernels.h).
//
// The reference enumerates every (v0, v1, v2) path of the 4-cycle and
// intersects two lists for each (src/gpu/impl/light/op/LIGHTComputeCount.cuh:
// 13-119; the house likewise, one path per (v1, v2, v3)).  Here the wedges
// a - b - w of a start vertex are counted per end w in LDS, so a wedge costs
// one list entry and one LDS add instead of an intersection.
#include <type_traits>

#include "kernels.h"
#include "walk.h"
#include "wave.h"

namespace sme {

namespace {

using u64 = unsigned long long;

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;

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

// ---------------------------------------------------------------------------
// 4-cycles of start vertices with at most 64 middles and kLightItems list
// entries to look at, one wave each.  c is kept in LDS bytes (c <= 64): over
// the id span of the ends, kLightSpan ids per pass, when two passes cover it,
// otherwise in a hash table keyed by w.  Each add returns the c before it, and
// their sum is sum_w c (c - 1) / 2.
//
// Bound by the latency of a start vertex's chain (its list, the middles' list
// bounds, their entries, the LDS adds).  300 packed G(n, m) members (1.25e6
// vertices, 3.3e7 entries): 1.8 ms, where the level engine wrote every wedge
// as a path and intersected two lists for it (52 ms).  Two passes over 4,096
// ids cover the members (n <= 8,192) at 6 waves per SIMD; a start vertex above
// kLightItems would hold its wave for over 64 steps and goes to the tiles.
constexpr uint32_t kCutList = 48;       // lists up to here are walked whole and filtered
constexpr uint32_t kLightItems = 4096;
constexpr uint32_t kLightSpan = 4096;   // ids per pass of the byte counters
constexpr uint32_t kLightSlots = 1024;  // hash slots, at most half full
constexpr int kLightBits = 10;
constexpr uint32_t kEmpty = 0xffffffffu;

struct LightLds {
  uint32_t buf[kLightSlots + kLightSlots / 4];  // byte counters, or keys and byte counters
  WalkLds walk;
};
static_assert(kLightSpan <= kLightSlots * 4, "byte counters fit the keys' place");

__global__ __launch_bounds__(kThreads, 6) void SquareLightKernel(WedgeArgs a) {
  __shared__ LightLds lds_all[kWaves];
  const int lane = threadIdx.x & (kWave - 1);
  LightLds& s = lds_all[threadIdx.x / kWave];
  const uint64_t wave = (blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x) / kWave;
  const uint64_t nwaves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  const uint64_t nv = a.v_end - a.v_begin;
  u64 total = 0, nup = 0, nwedge = 0, looked = 0;
  BucketAcc bacc{kNoBucket, 0};
  for (uint64_t g = wave * a.group; g < nv; g += nwaves * a.group) {
    const uint64_t ge = g + a.group < nv ? g + a.group : nv;
    for (uint64_t x = g; x < ge; ++x) {
      const uint32_t v0 = a.v_begin + static_cast<uint32_t>(x);
      const uint64_t nb = a.up[v0], ne = a.rp[v0 + 1];
      const uint64_t d = ne - nb;
      if (lane == 0) nup += d;
      if (d == 0) continue;
      bool heavy = d > kWave;
      if (heavy && lane == 0) looked += kWave * d;
      uint64_t lb = 0;
      uint32_t len = 0, last = 0;
      uint32_t items = 0, most = 0;
      if (!heavy) {
        if (static_cast<uint64_t>(lane) < d) {
          const uint32_t v1 = a.cols[nb + lane];
          lb = a.rp[v1];
          const uint64_t le = a.rp[v1 + 1];
          // v0 lies in N(v1): short lists are walked whole and filtered
          if (le - lb >= kCutList) lb = Lower(a.cols, lb, le, v0);
          looked += le - lb;
          heavy = le - lb > kLightItems;
          len = heavy ? kLightItems : static_cast<uint32_t>(le - lb);
          last = a.cols[le - 1];
        }
        heavy = __ballot(heavy) != 0;
        WavePrefix(len, lane, &items);
        most = last;
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) {
          const uint32_t y = __shfl_xor(most, o);
          most = y > most ? y : most;
        }
        heavy = heavy || items > kLightItems;
      }
      const bool dense = !heavy && most - v0 <= 2 * kLightSpan;
      if (!dense && items > kLightSlots / 2) heavy = true;
      if (heavy) {
        if (lane == 0) a.heavy[atomicAdd(a.nheavy, 1ull)] = v0;
        continue;
      }
      u64 sum = 0;
      if (dense) {
        for (uint32_t o = 1; o <= most - v0; o += kLightSpan) {
          const uint32_t lo = v0 + o;
          WaveSync();
          for (uint32_t k = lane; k < kLightSpan / 4; k += kWave) s.buf[k] = 0;
          WaveSync();
          uint32_t seen = 0, pairs = 0;
          WalkLists<false>(a.cols, nullptr, lb, len, 0u, s.walk, lane, [&](uint32_t w, uint32_t, uint32_t) {
            const uint32_t k = w - lo;  // (w <= v0: wraps around)
            if (k >= kLightSpan) return;
            const uint32_t sh = 8 * (k & 3);
            pairs += (atomicAdd(s.buf + (k >> 2), 1u << sh) >> sh) & 0xffu;
            ++seen;
          });
          nwedge += seen;
          sum += pairs;
        }
      } else {
        WaveSync();
        for (uint32_t k = lane; k < kLightSlots; k += kWave) s.buf[k] = kEmpty;
        for (uint32_t k = lane; k < kLightSlots / 4; k += kWave) s.buf[kLightSlots + k] = 0;
        WaveSync();
        uint32_t seen = 0, pairs = 0;
        WalkLists<false>(a.cols, nullptr, lb, len, 0u, s.walk, lane, [&](uint32_t w, uint32_t, uint32_t) {
          if (w <= v0) return;
          uint32_t h = (w * 0x9E3779B1u) >> (32 - kLightBits);
          while (true) {
            const uint32_t old = atomicCAS(s.buf + h, kEmpty, w);
            if (old == kEmpty || old == w) break;
            h = (h + 1) & (kLightSlots - 1);
          }
          const uint32_t sh = 8 * (h & 3);
          pairs += (atomicAdd(s.buf + kLightSlots + (h >> 2), 1u << sh) >> sh) & 0xffu;
          ++seen;
        });
        nwedge += seen;
        sum += pairs;
      }
      total += sum;
      if (a.bk.bounds) BucketAccAdd(a.bk, &bacc, BucketOf(a.bk, v0), sum);
    }
  }
  if (a.bk.bounds) BucketFlush(a.bk, &bacc);
  BlockAdd<kThreads>(Into{a.acc, total}, Into{a.acc + 1, nup}, Into{a.acc + 2, nwedge}, Into{a.acc + 3, looked});
}

// ---------------------------------------------------------------------------
// One workgroup per start vertex and tile of kIds ids; 16-bit counters of c in
// LDS, two per word.  Workgroups take items from a counter, since start
// vertices differ by orders of magnitude; each ends when the counter passes
// the last item.  Graphs of up to 16,384 vertices use 32 KB of counters and
// four workgroups per CU; larger ones 128 KB and one of 1,024 threads, since a
// list has to be cut once per tile (tiles of 32,768 ids: 56 ms where these take
// 38, searching).  The cuts of every list at the tiles' bounds are kept in a
// table where there is room (one load instead of two searches: 38 -> 25 ms).
//
// Bound by the list reads: on R-MAT scale 19 (below) 121 GB past L2 in 24.5 ms,
// the rate of a large copy, with the VALU busy in 32 % of the cycles; on graphs
// that the caches hold by the latency of the walks.  House from a third of R-MAT scale
// 14's start vertices: 0.31 ms, where the level engine counted pairs for every
// (v1, v2, v3) path (11.1 ms).  House of R-MAT scale 19, edge factor 32, from
// its apexes (6.7e9 wedges walked twice): 25 ms, where one 64-bit device atomic
// per wedge into dense arrays and their reduction took 327 ms.
template <int kUse, uint32_t kIds, int kThr>
__global__ __launch_bounds__(kThr) void WedgeTileKernel(WedgeArgs a) {
  constexpr uint32_t kWv = kThr / kWave;
  __shared__ uint32_t cnt[kIds / 2];
  __shared__ uint32_t adj[kUse == kWedgeHouse ? kIds / 32 : 1];  // house: ids of N(a)
  __shared__ WalkLds walk_all[kWv];
  __shared__ u64 item_s;
  __shared__ u64 sum_s;
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t wid = threadIdx.x / kWave;
  WalkLds& s = walk_all[wid];
  const u64 napex = a.heavy ? *a.nheavy : a.v_end - a.v_begin;
  const u64 nitems = napex * a.ntiles;
  // (the same for all workgroups)
  if (kUse == kWedgeSquare && a.items_ratio && nitems > WedgeItemsMax(a.acc[3], a.items_ratio)) return;
  u64 total = 0, c1 = 0, c2 = 0, c3 = 0, c4 = 0, c5 = 0;
  while (true) {
    __syncthreads();  // the previous item's readers of item_s, sum_s and the counters are done
    if (threadIdx.x == 0) {
      item_s = atomicAdd(a.next, 1ull);
      sum_s = 0;
    }
    __syncthreads();
    const u64 item = item_s;
    if (item >= nitems) break;
    u64 x = a.ntiles == 1 ? item : item / a.ntiles;
    const uint32_t tile = a.ntiles == 1 ? 0 : static_cast<uint32_t>(item - x * a.ntiles);
    // the apexes were appended in about increasing id: heaviest first
    if (kUse == kWedgeApex) x = napex - 1 - x;
    const uint32_t v = a.heavy ? a.heavy[x] : a.v_begin + static_cast<uint32_t>(x);
    const uint64_t rb = a.rp[v], ub = a.up[v], re = a.rp[v + 1];
    // ends of this item: ids [lo, hi)
    uint32_t lo = tile * kIds, hi = a.n - lo < kIds ? a.n : lo + kIds;
    if (kUse == kWedgeHouse && tile == 0 && threadIdx.x == 0) {
      c1 += re - ub;
      c2 += re - rb;
      c4 += (re - ub) * (re - rb - (re > rb ? 1 : 0));
    }
    if (kUse == kWedgeSquare && hi <= v + 1) continue;  // no end above v
    if (kUse == kWedgeSquare && lo <= v) lo = v + 1;
    if (kUse == kWedgeApex && lo >= v) continue;         // no end below v
    if (kUse == kWedgeApex && hi > v) hi = v;
    // middles
    const uint64_t mb = kUse == kWedgeSquare ? ub : rb, me = kUse == kWedgeApex ? ub : re;
    if (kUse == kWedgeApex ? rb == ub : ub == re) continue;  // none, or no b > a
    const uint32_t words = (hi - lo + 1) / 2;
    for (uint32_t k = threadIdx.x; k < words; k += kThr) cnt[k] = 0;
    if (kUse == kWedgeHouse)
      for (uint32_t k = threadIdx.x; k < (hi - lo + 31) / 32; k += kThr) adj[k] = 0;
    __syncthreads();
    // a wave takes `per` middles at a time, all waves about the same number; a
    // second walk over the same middles finds the first ones' windows again
    uint64_t lb_kept = 0;
    uint32_t len_kept = 0;
    auto walk = [&](auto with_t, uint64_t b, uint64_t e, auto&& prep, auto&& f) {
      const uint64_t share = (e - b + kWv - 1) / kWv;
      const uint32_t per = share < kWave ? static_cast<uint32_t>(share) : kWave;
      for (uint64_t k0 = b + static_cast<uint64_t>(wid) * per; k0 < e; k0 += static_cast<uint64_t>(kWv) * per) {
        const uint64_t k = k0 + lane;
        uint64_t lb = 0;
        uint32_t len = 0, mid = 0;
        if (static_cast<uint32_t>(lane) < per && k < e) {
          if (kUse == kWedgeApex && decltype(with_t)::value && k0 == b + static_cast<uint64_t>(wid) * per) {
            lb = lb_kept;
            len = len_kept;
          } else {
            const uint32_t m = a.cols[k];
            lb = a.rp[m];
            uint64_t le = a.rp[m + 1];
            if (a.cuts) {
              // the tile's share of N(m), then the end or start within it
              const uint32_t* cut = a.cuts + static_cast<uint64_t>(m) * (a.ntiles + 1) + tile;
              le = lb + cut[1];
              lb += cut[0];
              if (lo != tile * kIds) lb = Lower(a.cols, lb, le, lo);
              if (hi != tile * kIds + kIds && hi != a.n) le = Lower(a.cols, lb, le, hi);
            } else {
              if (lo > 0) lb = Lower(a.cols, lb, le, lo);
              if (hi < a.n) le = Lower(a.cols, lb, le, hi);
            }
            len = static_cast<uint32_t>(le - lb);
          }
          mid = prep(k);
        }
        if (kUse == kWedgeApex && k0 == b + static_cast<uint64_t>(wid) * per) {
          lb_kept = lb;
          len_kept = len;
        }
        WalkLists<decltype(with_t)::value>(a.cols, a.t, lb, len, mid, s, lane, f);
      }
    };
    walk(std::false_type{}, mb, me, [](uint64_t) { return 0u; },
         [&](uint32_t w, uint32_t, uint32_t) {
           const uint32_t k = w - lo;
           atomicAdd(cnt + (k >> 1), 1u << (16 * (k & 1)));
         });
    if (kUse == kWedgeHouse) {
      uint64_t b = rb, e = re;
      if (lo > 0) b = Lower(a.cols, b, e, lo);
      if (hi < a.n) e = Lower(a.cols, b, e, hi);
      for (uint64_t k = b + threadIdx.x; k < e; k += kThr) {
        const uint32_t o = a.cols[k] - lo;
        atomicOr(adj + (o >> 5), 1u << (o & 31));
      }
    }
    __syncthreads();
    u64 sum = 0;
    if (kUse == kWedgeSquare) {
      for (uint32_t k = threadIdx.x; k < words; k += kThr) {
        const u64 p = cnt[k] & 0xffffu, q = cnt[k] >> 16;
        c2 += p + q;
        sum += (p ? p * (p - 1) / 2 : 0) + (q ? q * (q - 1) / 2 : 0);
      }
    } else if (kUse == kWedgeApex) {
      walk(std::true_type{}, rb, ub, [&](uint64_t k) { return a.t[k]; },
           [&](uint32_t w, uint32_t tbw, uint32_t tab) {
             const uint32_t k = w - lo;
             const uint32_t c = (cnt[k >> 1] >> (16 * (k & 1))) & 0xffffu;
             sum += static_cast<u64>(c - 1) * (tab + tbw);
           });
    } else {
      // b > a: t(a, b) (c(a, w) - 1) per end w, less the pairs whose apex is w
      // or the middle opposite b
      walk(std::true_type{}, ub, re,
           [&](uint64_t k) {
             const uint32_t tab = a.t[k];
             if (tile == 0) {
               c3 += tab;
               c5 += static_cast<u64>(tab) * (re - rb - 2);  // (tab > 0: d(a) >= 2)
             }
             return tab;
           },
           [&](uint32_t w, uint32_t tbw, uint32_t tab) {
             if (w == v) return;
             const uint32_t k = w - lo;
             const uint32_t c = (cnt[k >> 1] >> (16 * (k & 1))) & 0xffffu;
             sum += static_cast<u64>(tab) * (c - 1);
             if ((adj[k >> 5] >> (k & 31)) & 1u) sum -= static_cast<u64>(tbw) + c - 2;
           });
    }
    total += sum;
    if (a.bk.bounds) {
      sum = WaveSum(sum);
      if (lane == 0 && sum) atomicAdd(&sum_s, sum);
      __syncthreads();
      if (threadIdx.x == 0 && sum_s) atomicAdd(a.bk.counts + BucketOf(a.bk, v), sum_s);
    }
  }
  BlockAdd<kThr>(Into{a.acc, total});
  if (kUse == kWedgeSquare) {
    BlockAdd<kThr>(Into{a.acc + 2, c2});
  } else if (kUse == kWedgeHouse) {
    BlockAdd<kThr>(Into{a.acc + 1, c1},
                   Into{a.acc + 2, c2},
                   Into{a.acc + 3, c3},
                   Into{a.acc + 4, c4},
                   Into{a.acc + 5, c5});
  }
}

// ---------------------------------------------------------------------------
// 64 consecutive entries per wave; a lane finds its row between those of the
// wave's first and last entry.
__global__ __launch_bounds__(kThreads) void AsymmetricKernel(const uint64_t* rp, const uint32_t* cols, uint64_t n,
                                                             uint64_t nnz, uint64_t* flag) {
  const int lane = threadIdx.x & (kWave - 1);
  const uint64_t wave = (blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x) / kWave;
  const uint64_t nwaves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  // last row starting at or before entry e
  auto row_of = [&](uint64_t e, uint64_t lo, uint64_t hi) {
    while (lo < hi) {
      const uint64_t mid = (lo + hi + 1) >> 1;
      if (rp[mid] <= e)
        lo = mid;
      else
        hi = mid - 1;
    }
    return lo;
  };
  bool bad = false;
  for (uint64_t e0 = wave * kWave; e0 < nnz; e0 += nwaves * kWave) {
    const uint64_t e1 = e0 + kWave < nnz ? e0 + kWave : nnz;
    const uint64_t r0 = row_of(e0, 0, n - 1);
    const uint64_t r1 = row_of(e1 - 1, r0, n - 1);
    const uint64_t e = e0 + lane;
    if (e >= e1) continue;
    const uint32_t v = static_cast<uint32_t>(row_of(e, r0, r1)), u = cols[e];
    const uint64_t p = Lower(cols, rp[u], rp[u + 1], v);
    bad = bad || p >= rp[u + 1] || cols[p] != v;
  }
  if (__ballot(bad) && lane == 0) *flag = 1;
}

// 16,384 ids: 32 KB of counters, four workgroups per CU; 65,536: 128 KB, one
constexpr uint32_t kSmall = kWedgeSmallIds, kLarge = 65536;

__global__ __launch_bounds__(kThreads) void WedgeCutsKernel(WedgeArgs a, uint32_t* cuts) {
  const uint64_t per = a.ntiles + 1, total = per * a.n;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < total; i += stride) {
    const uint64_t v = i / per, b = a.rp[v], e = a.rp[v + 1], lo = (i - v * per) * kLarge;
    cuts[i] = static_cast<uint32_t>((lo < a.n ? Lower(a.cols, b, e, static_cast<uint32_t>(lo)) : e) - b);
  }
}

template <int kUse>
void LaunchTiles(const WedgeArgs& a, hipStream_t stream) {
  WedgeArgs b = a;
  const uint64_t nv = a.v_end - a.v_begin;
  if (a.n <= kSmall) {
    b.ntiles = 1;
    b.cuts = nullptr;
    const uint32_t grid = nv < 1024 ? static_cast<uint32_t>(nv) : 1024;
    hipLaunchKernelGGL((WedgeTileKernel<kUse, kSmall, 256>), dim3(grid), dim3(256), 0, stream, b);
  } else {
    b.ntiles = WedgeTiles(a.n);
    const uint64_t items = nv * b.ntiles;
    const uint32_t grid = items < 256 ? static_cast<uint32_t>(items) : 256;
    hipLaunchKernelGGL((WedgeTileKernel<kUse, kLarge, 1024>), dim3(grid), dim3(1024), 0, stream, b);
  }
}

}  // namespace

void LaunchSquareLight(const WedgeArgs& a, hipStream_t stream) {
  const uint64_t nv = a.v_end - a.v_begin;
  if (nv == 0) return;
  WedgeArgs b = a;
  // consecutive start vertices share a bucket: one bucket atomic per group
  const uint64_t per = nv / 8192;
  b.group = static_cast<uint32_t>(per < 1 ? 1 : per > 16 ? 16 : per);
  const uint64_t need = ((nv + b.group - 1) / b.group + kWaves - 1) / kWaves;
  // whole rounds of the six workgroups per CU that their LDS allows (2,048: 2.25 ms, 1,536: 1.92, 6,144: 1.82)
  hipLaunchKernelGGL(SquareLightKernel, dim3(need < 6144 ? need : 6144), dim3(kThreads), 0, stream, b);
}

uint32_t WedgeTiles(uint32_t n) { return n <= kSmall ? 1 : (n - 1) / kLarge + 1; }

void LaunchWedgeCuts(const WedgeArgs& a, uint32_t* cuts, hipStream_t stream) {
  WedgeArgs b = a;
  b.ntiles = WedgeTiles(a.n);
  const uint64_t need = ((b.ntiles + 1ull) * a.n + kThreads - 1) / kThreads;
  hipLaunchKernelGGL(WedgeCutsKernel, dim3(need < 8192 ? need : 8192), dim3(kThreads), 0, stream, b, cuts);
}

void LaunchWedgeTiles(const WedgeArgs& a, int use, hipStream_t stream) {
  if (a.v_end <= a.v_begin) return;
  if (use == kWedgeSquare)
    LaunchTiles<kWedgeSquare>(a, stream);
  else if (use == kWedgeHouse)
    LaunchTiles<kWedgeHouse>(a, stream);
  else
    LaunchTiles<kWedgeApex>(a, stream);
}

void LaunchAsymmetric(const uint64_t* rp, const uint32_t* cols, uint64_t n, uint64_t nnz, uint64_t* flag,
                      hipStream_t stream) {
  if (nnz == 0) return;
  const uint64_t need = (nnz + kThreads - 1) / kThreads;
  hipLaunchKernelGGL(AsymmetricKernel, dim3(need < 16384 ? need : 16384), dim3(kThreads), 0, stream, rp, cols, n, nnz,
                     flag);
}

}  // namespace sme
