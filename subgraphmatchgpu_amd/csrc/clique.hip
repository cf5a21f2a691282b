// clique.hip -- k-clique counting over bitmaps of upper neighbourhoods
// (CliqueArgs in kernels.h).
//
// Start vertices with at most 64 upper neighbours are counted by
// CliqueSmallKernel: a row is one u64, so every set below a row is one u64 and
// every step of the count is an LDS load, an AND and a popcount.  Larger
// neighbourhoods are counted in batches.  Their rows are found by
//   CliqueRowsTableKernel  d <= 4,096 and a span of fewer than 65,536 ids: N+(v)
//                          as an LDS table over its span (with per-edge counts on
//                          a ranked graph, CliqueMiddleKernel beside it);
//   CliqueRowsHashKernel   d <= 4,096, wider spans: N+(v) as an LDS hash;
//   CliqueRowsKernel       d > 4,096: binary search;
// which count triangles themselves and write rows to device memory for the
// larger cliques:
//   CliqueDenseKernel      4-cliques, d <= 512: all rows of a vertex in LDS;
//   CliqueCount4Kernel     4-cliques, the others: one wave per row;
//   CliquePackKernel       5- and 6-cliques, one wave per row of up to 128
//                          members, packed to those; CliqueLongKernel up to 512
//                          (5-cliques); CliqueUnpackedKernel the others.
//
// The reference counts the same cliques by intersecting sorted adjacency
// lists level by level (src/gpu/impl/light/op/LIGHTCompute.cuh,
// LIGHTComputeCount.cuh:13-119); here the lists of one start vertex's
// neighbourhood become bit rows, and one word operation replaces up to 64
// membership probes.
#include "kernels.h"
#include "walk.h"
#include "wave.h"

namespace sme {

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr uint32_t kWordsMax = kLocalMax / 64;  // words of the longest row
static_assert(2 * kRowsHashSmall <= (1u << 10) && 2 * kRowsHashMax <= (1u << 13), "hash tables at most half full");
constexpr uint64_t kMaxGrid = 16384;

using u64 = unsigned long long;

uint64_t Grid(uint64_t n, uint64_t per_block) {
  uint64_t g = (n + per_block - 1) / per_block;
  if (g < 1) g = 1;
  return g > kMaxGrid ? kMaxGrid : g;
}

__device__ __forceinline__ uint32_t Lane32(uint32_t v, uint32_t lane) {
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), static_cast<int>(lane)));
}

__device__ __forceinline__ u64 First64(u64 v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
  return (static_cast<u64>(hi) << 32) | lo;
}

// Does the sorted a[lo, hi) hold key?  *pos: where (when it does).
__device__ __forceinline__ bool Holds(const uint32_t* a, uint64_t lo, uint64_t hi, uint32_t key,
                                      uint64_t* pos) {
  const uint64_t end = hi;
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if (a[mid] < key)
      lo = mid + 1;
    else
      hi = mid;
  }
  *pos = lo;
  return lo < end && a[lo] == key;
}

__device__ __forceinline__ void AddBucket(const BucketRef& b, uint32_t v, u64 per_lane, int lane) {
  const u64 tot = WaveSum(per_lane);
  if (lane == 0 && tot) atomicAdd(b.counts + BucketOf(b, v), tot);
}

// ---------------------------------------------------------------------------
// Start vertices with d <= 64.  A wave takes kSmallGroup consecutive start
// vertices, packs as many whole ones as fit into 64 upper entries (lane =
// entry u_i of some N+(v)) and walks their entries' work as one flat list of
// items, 64 per step, so short neighbourhoods share a step.  An entry's work
// is the cheaper of
//   stream: the values x of N+(u_i), each looked up among the u_j (j > i)
//           staged in LDS (one coalesced load and at most 6 LDS steps);
//   search: the u_j (j > i), each searched in N+(u_i) (a chain of dependent
//           loads, log2 |N+(u_i)| long).
// A hit (i, j) is a triangle.  From K = 4 on it sets bit j of row i in LDS,
// and lane = row then counts the larger cliques by AND + popcount.
//
// Bound by the latency of the gathers (list bounds, then list values).  One
// wave per start vertex, searching one row after another with most lanes
// idle, took 10.2 ms on 1,000 packed G(n, m) members (5.4e7 entries, 13 per
// vertex) and 3.7 ms on R-MAT scale 20 (degree-ranked, 6 per vertex); the
// flat items take 2.4 and 1.1 ms.  Groups of 8 or 16 start vertices were
// slower (1.6, 1.7 ms on R-MAT: the heavy groups end last), and so was
// choosing the mode on rem * steps < len (67 against 87 us, R-MAT scale 14).
constexpr uint32_t kSmallGroup = 4;  // start vertices per wave step
constexpr uint32_t kSmallStream = 32;    // lists up to this length are streamed
// up to here one start vertex per wave step, since 4,096 waves of 4 vertices
// leave half the chip idle.  Whole triangle calls, one vertex and four a step:
// R-MAT 14 148 and 182 us, G(16,000, 160,000) 83 and 81; above the line
// G(24,000, 240,000) 87 and 83, G(32,000, 320,000) 91 and 87, R-MAT 15 357 and 367
constexpr uint64_t kSmallAlone = 16384;
// workgroups: what the chip holds at once; half of it up to 4 kSmallAlone start
// vertices, where each would get a few, since every one ends with atomics on the
// same counters (1,024 and 2,048 workgroups: G(40,000, 400,000) 90 and 160 us,
// R-MAT 18, factor 4, 1.13 and 1.04 ms)
constexpr uint64_t kSmallGrid = 2048, kSmallGridFew = 1024;

struct SmallLds {
  uint64_t beg[kWave];    // entry: N+(u_i) begins at cols[beg]
  u64 row[kWave];         // entry: row i (K >= 4)
  uint32_t key[kWave];    // entry: u_i
  uint32_t len[kWave];    // entry: |N+(u_i)|
  uint32_t base[kWave];   // entry: its vertex's first entry
  uint32_t last[kWave];   // entry: one past its vertex's last entry
  uint32_t start[kWave];  // k-th entry with work: its first item
  uint32_t edge[kWave];   // k-th entry with work: the entry, bit 31: search
  uint32_t flag[kWave];   // item of this step starts an entry
  uint32_t cnt[kWave];    // entry: triangles (per-edge counts or buckets)
};

// (8 waves per SIMD: at the 67 registers of free choice a CU holds 7 of the 8
// workgroups it is given, and the last ones run alone: 3.1 against 2.4 ms on the
// packed members, 1.37 against 1.12 on R-MAT scale 20.)
template <int K>
__global__ __launch_bounds__(kThreads, 8) void CliqueSmallKernel(CliqueArgs a) {
  __shared__ SmallLds lds_all[kWaves];
  const int lane = threadIdx.x & (kWave - 1);
  SmallLds& s = lds_all[threadIdx.x / kWave];
  const u64 upto = ~0ull >> (kWave - 1 - lane);  // lanes 0..lane
  const uint64_t wave = (blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x) / kWave;
  const uint64_t nwaves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  const uint64_t nv = a.v_end - a.v_begin;
  const bool counted = a.tc || a.bk.bounds;  // triangles are kept per entry
  u64 c1 = 0, c2 = 0, c3 = 0, c4 = 0, c5 = 0, c6 = 0;
  BucketAcc bacc{kNoBucket, 0};
  const uint64_t ngroups = (nv + a.group - 1) / a.group;
  for (uint64_t t = wave; t < ngroups; t += nwaves) {
    const uint64_t first = t * a.group;
    const uint32_t gn = static_cast<uint32_t>(first + a.group < nv ? a.group : nv - first);
    uint64_t nb_l = 0, d_l = 0;  // lane q: vertex q of the group
    if (static_cast<uint32_t>(lane) < gn) {
      const uint32_t v = a.v_begin + static_cast<uint32_t>(first) + lane;
      nb_l = a.up[v];
      d_l = a.rp[v + 1] - nb_l;
      if (d_l <= kLocalMax) {
        c1 += 1;
        c2 += d_l;
      }
      if (d_l > kLocalSmall) {
        // (big == nullptr: the caller already holds these lists)
        if (d_l <= kLocalMax) {
          if (a.big) {
            const u64 pos = atomicAdd(a.nbig, 1ull);
            a.big[pos] = v;
            a.big_d[pos] = static_cast<uint32_t>(d_l);
          }
        } else if (a.huge) {
          a.huge[atomicAdd(a.nhuge, 1ull)] = v;
        }
        d_l = 0;
      }
      if (d_l < 2) d_l = 0;  // no triangle from v
    }
    uint32_t dq[kSmallGroup];
    uint64_t nbq[kSmallGroup];
#pragma unroll
    for (uint32_t q = 0; q < kSmallGroup; ++q) {
      dq[q] = Lane32(static_cast<uint32_t>(d_l), q);
      nbq[q] = (static_cast<uint64_t>(Lane32(static_cast<uint32_t>(nb_l >> 32), q)) << 32) |
               Lane32(static_cast<uint32_t>(nb_l), q);
    }
    for (uint32_t q0 = 0; q0 < gn;) {
      // vertices q0.. of the group whose entries fit the wave together
      uint32_t ne = 0, d = 0, i = 0, end = 0, q1 = q0, mine = q0;
      uint64_t nb = 0;
      bool open = true;
#pragma unroll
      for (uint32_t q = 0; q < kSmallGroup; ++q) {
        if (q < q0 || q >= gn) continue;
        if (!open || ne + dq[q] > kWave) {
          open = false;
          continue;
        }
        if (static_cast<uint32_t>(lane) >= ne && static_cast<uint32_t>(lane) < ne + dq[q]) {
          d = dq[q];
          nb = nbq[q];
          i = static_cast<uint32_t>(lane) - ne;
          end = ne + dq[q];
          mine = q;
        }
        ne += dq[q];
        q1 = q + 1;
      }
      q0 = q1;
      if (ne == 0) continue;
      const bool entry = static_cast<uint32_t>(lane) < ne;
      uint32_t u = 0, len = 0;
      uint64_t lb = 0;
      if (entry) {
        u = a.cols[nb + i];
        if (i + 1 < d) {
          lb = a.up[u];
          len = static_cast<uint32_t>(a.rp[u + 1] - lb);
        }
      }
      const uint32_t rem = len ? d - 1 - i : 0;  // u_j above u_i
      const uint32_t steps = 32 - static_cast<uint32_t>(__clzll(static_cast<long long>(len))) + 32;
      // (a wave whose items mix both pays for both: short lists always stream)
      const bool search = len > kSmallStream && rem * steps < 2 * len;
      const uint32_t items = search ? rem : (rem ? len : 0);
      uint32_t total;
      const uint32_t start = WavePrefix(items, lane, &total);
      if (total == 0) continue;
      const u64 work = __ballot(items != 0);
      WaveSync();  // the previous step's readers are done
      s.key[lane] = u;
      s.beg[lane] = lb;
      s.len[lane] = len;
      s.base[lane] = end - d;
      s.last[lane] = end;
      if (K >= 4) s.row[lane] = 0;
      if (counted) s.cnt[lane] = 0;
      if (items) {
        const int at = static_cast<int>(__popcll(work & (upto >> 1)));
        s.start[at] = start;
        s.edge[at] = static_cast<uint32_t>(lane) | (search ? 0x80000000u : 0u);
      }
      uint32_t before = 0;  // entries with work that started before this step
      for (uint32_t t0 = 0; t0 < total; t0 += kWave) {
        s.flag[lane] = 0;
        WaveSync();
        if (items && start >= t0 && start - t0 < kWave) s.flag[start - t0] = 1;
        WaveSync();
        const u64 starts = __ballot(s.flag[lane] != 0);
        const uint32_t own = before + static_cast<uint32_t>(__popcll(starts & upto)) - 1;
        before += static_cast<uint32_t>(__popcll(starts));
        const uint32_t it = t0 + static_cast<uint32_t>(lane);
        if (it < total) {
          const uint32_t packed = s.edge[own];
          const uint32_t e = packed & 0x7fffffffu, k = it - s.start[own];
          uint64_t lo = s.beg[e];
          uint32_t j = e + 1;  // entry of the vertex holding the value
          bool hit;
          if (packed >> 31) {
            j += k;
            const uint32_t x = s.key[j];
            const uint64_t le = lo + s.len[e];
            uint64_t hi = le;
            while (lo < hi) {
              const uint64_t mid = (lo + hi) >> 1;
              if (a.cols[mid] < x)
                lo = mid + 1;
              else
                hi = mid;
            }
            hit = lo < le && a.cols[lo] == x;
          } else {
            lo += k;
            const uint32_t x = a.cols[lo], je = s.last[e];
            uint32_t hi = je;
            while (j < hi) {
              const uint32_t mid = (j + hi) >> 1;
              if (s.key[mid] < x)
                j = mid + 1;
              else
                hi = mid;
            }
            hit = j < je && s.key[j] == x;
          }
          if (hit) {
            if (K == 3) {
              ++c3;
              if (counted) atomicAdd(s.cnt + e, 1u);
              if (a.tc) {
                atomicAdd(s.cnt + j, 1u);
                atomicAdd(a.tc + lo, 1u);  // edge (u_i, u_j)
              }
            } else {
              atomicOr(s.row + e, 1ull << (j - s.base[e]));
            }
          }
        }
      }
      WaveSync();
      u64 vk = 0;  // this entry's share of the k-cliques from its vertex
      if (K == 3) {
        // edges (v, u_i): the triangles (v, u_i, x)
        if (counted) vk = s.cnt[lane];
        if (a.tc && entry && vk) atomicAdd(a.tc + nb + i, static_cast<uint32_t>(vk));
      } else if (entry) {
        const uint32_t base = end - d;
        const u64 s1 = s.row[lane];
        c3 += __popcll(s1);
        for (u64 m1 = s1; m1; m1 &= m1 - 1) {
          const u64 s2 = s1 & s.row[base + static_cast<uint32_t>(__builtin_ctzll(m1))];
          const u64 x4 = __popcll(s2);
          c4 += x4;
          if (K == 4) {
            vk += x4;
            continue;
          }
          for (u64 m2 = s2; m2; m2 &= m2 - 1) {
            const u64 s3 = s2 & s.row[base + static_cast<uint32_t>(__builtin_ctzll(m2))];
            const u64 x5 = __popcll(s3);
            c5 += x5;
            if (K == 5) {
              vk += x5;
              continue;
            }
            for (u64 m3 = s3; m3; m3 &= m3 - 1) {
              const u64 x6 = __popcll(s3 & s.row[base + static_cast<uint32_t>(__builtin_ctzll(m3))]);
              c6 += x6;
              vk += x6;
            }
          }
        }
      }
      if (a.bk.bounds)
        BucketAccAdd(a.bk, &bacc, entry ? BucketOf(a.bk, a.v_begin + static_cast<uint32_t>(first) + mine) : kNoBucket, vk);
    }
  }
  if (a.bk.bounds) BucketFlush(a.bk, &bacc);
  BlockAdd<kThreads>(Into{a.acc + 1, c1},
                     Into{a.acc + 2, c2},
                     Into{a.acc + 3, c3},
                     Into{K >= 4 ? a.acc + 4 : nullptr, c4},
                     Into{K >= 5 ? a.acc + 5 : nullptr, c5},
                     Into{K >= 6 ? a.acc + 6 : nullptr, c6});
  if (!a.publish) return;
  // the sums above were added by threads of wave 0, as is the ticket
  __shared__ bool last;
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "agent");
  if (threadIdx.x == 0) last = atomicAdd(a.done, 1ull) == gridDim.x - 1;
  __syncthreads();
  if (!last) return;
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "agent");
  if (threadIdx.x <= static_cast<unsigned>(kCliqueMaxK)) {
    a.publish[threadIdx.x] = atomicAdd(a.acc + threadIdx.x, 0ull);
    a.acc[threadIdx.x] = 0;
  }
  if (threadIdx.x == 0) *a.done = 0;
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "");  // (these are all of wave 0)
  if (threadIdx.x == 0) *const_cast<volatile unsigned long long*>(a.publish + kCliqueMaxK + 1) = a.call;
}

// ---------------------------------------------------------------------------
// Big vertices: row items.  Vertex x of the batch owns items
// [row_first[x], row_first[x+1]) - row_first[0]; the wave-uniform search
// finds it.
__device__ __forceinline__ uint64_t ItemVertex(const CliqueArgs& a, uint64_t t) {
  const uint64_t base = a.row_first[0];
  uint64_t lo = 0, hi = a.nverts - 1;
  while (lo < hi) {
    const uint64_t mid = (lo + hi + 1) >> 1;
    if (a.row_first[mid] - base <= t)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// The same by the whole wave: 64 evenly spaced entries per round, so that the
// chain of dependent loads is 3 long (60,000 vertices) instead of 16.
__device__ __forceinline__ uint64_t ItemVertexWave(const CliqueArgs& a, uint64_t t, int lane) {
  const uint64_t key = a.row_first[0] + t;
  uint64_t lo = 0, n = a.nverts;  // the vertex lies in [lo, lo + n)
  while (n > 1) {
    const uint64_t step = (n + kWave - 1) / kWave;
    const uint64_t at = lo + static_cast<uint64_t>(lane) * step;
    const u64 m = __ballot(static_cast<uint64_t>(lane) * step < n && a.row_first[at] <= key);
    const uint64_t skip = (__popcll(m) - 1) * step;  // lane 0 always holds
    lo += skip;
    n = n - skip < step ? n - skip : step;
  }
  return lo;
}

// One wave per row: word c of row i is the ballot of "u_j in N+(u_i)" over
// j = 64c + lane (j > i).  Words are gathered one per lane and stored 64 at
// a time.
__global__ __launch_bounds__(kThreads) void CliqueRowsKernel(CliqueArgs a) {
  const int lane = threadIdx.x & (kWave - 1);
  const uint64_t wave = (blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x) / kWave;
  const uint64_t nwaves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  u64 c3 = 0;  // triangles, when no count kernel follows (rows == nullptr)
  for (uint64_t t = wave; t < a.nitems; t += nwaves) {
    const uint64_t x = ItemVertex(a, t);
    const uint32_t v = a.verts[x];
    const uint32_t d = static_cast<uint32_t>(a.row_first[x + 1] - a.row_first[x]);
    const uint32_t i = static_cast<uint32_t>(t - (a.row_first[x] - a.row_first[0]));
    const uint32_t W = (d + 63) / 64;
    u64* rows = a.rows + (a.word_first[x] - a.word_first[0]);  // word w of row i at rows[w * d + i]
    const uint64_t nb = a.up[v];
    const uint32_t ui = a.cols[nb + i];
    const uint64_t lb = a.up[ui], le = a.rp[ui + 1];
    u64 keep = 0;
    uint32_t bits = 0;
    for (uint32_t c = 0; c < W; ++c) {
      const uint32_t j = c * 64 + static_cast<uint32_t>(lane);
      uint64_t pos = 0;
      const bool ok = j > i && j < d && Holds(a.cols, lb, le, a.cols[nb + j], &pos);
      const u64 w = __ballot(ok);
      if ((c & 63u) == static_cast<uint32_t>(lane)) keep = w;
      if ((c & 63u) == 63u || c + 1 == W) {
        if (a.rows && static_cast<uint32_t>(lane) <= (c & 63u))
          rows[static_cast<uint64_t>((c & ~63u) + lane) * d + i] = keep;
      }
      if (ok && a.tc) {
        atomicAdd(a.tc + pos, 1u);     // edge (u_i, u_j)
        atomicAdd(a.tc + nb + j, 1u);  // edge (v, u_j)
      }
      bits += static_cast<uint32_t>(__popcll(w));
    }
    // edge (v, u_i): one triangle per bit of row i
    if (a.tc && lane == 0 && bits) atomicAdd(a.tc + nb + i, bits);
    if (lane == 0) c3 += bits;
    if (!a.rows && a.bk.bounds) AddBucket(a.bk, v, lane == 0 ? bits : 0u, lane);
  }
  if (!a.rows) BlockAdd<kThreads>(Into{a.acc + 3, c3});
}

// Chunk t of a batch: largest x with chunk_first[x] - chunk_first[0] <= t.
__device__ __forceinline__ uint64_t ChunkVertex(const CliqueArgs& a, uint64_t t) {
  const uint64_t base = a.chunk_first[0];
  uint64_t lo = 0, hi = a.nverts - 1;
  while (lo < hi) {
    const uint64_t mid = (lo + hi + 1) >> 1;
    if (a.chunk_first[mid] - base <= t)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// Is vertex v (d upper neighbours from `base` to `vmax`) taken by
// CliqueRowsTableKernel?
__device__ __forceinline__ bool TableTakes(uint32_t d, uint32_t base, uint32_t vmax) {
  return d <= kRowsTableMax && vmax - base < kRowsTableRange;
}

// Are the triangles (v, u, w) found in row u of a table vertex v left to
// CliqueMiddleKernel for edge (u, w)?  By u's own upper neighbourhood.
__device__ __forceinline__ bool MiddleTakes(uint32_t d, uint32_t first, uint32_t last) {
  return d <= kMiddleMax && last - first < kRowsTableRange;
}

// Rows of a vertex v whose N+(v) spans fewer than kRowsTableRange ids: a
// workgroup takes a.part rows at a time (every gridDim.y-th such part).  N+(v) becomes an LDS
// table with, per 32 consecutive ids, the bits of those in N+(v) and the local
// index of the first, so one 8-byte LDS load decides an entry of N+(u_i) and
// gives its j, without the probe chains of a hash.  Each wave streams N+(u_i)
// up to the largest value of N+(v), 128 consecutive entries per step, the next
// step's loads issued before this step's lookups.  kMode: kRowsBits sets bit j
// of row i (an LDS OR) and writes the row; kRowsCount counts the triangles;
// kRowsEdges adds each triangle to its three edges' counts.
//
// Bound by the wave instructions of the lookups and, with per-edge counts, by
// the device atomics (about 3.7 ms of the 6.5 ms below).  R-MAT scale 20
// (degree-ranked; 60,395 vertices, 3.0e9 entries streamed): rows 7.0 -> 2.8 ms,
// per-edge counts 10.4 -> 6.5 ms against the LDS hash, whose probe chains
// diverge (64 lanes wait for the longest).  The span of 65,536 ids is the
// largest whose table (16 KB) still lets 32 waves share a CU; on a ranked
// graph the 60,000 vertices with d > 64 all lie within it.
enum RowsMode : int { kRowsBits = 0, kRowsCount = 1, kRowsEdges = 2 };
// Rows a workgroup takes at a time: 256, since each part builds the table anew, but
// 64 where the launch has fewer than kTableFew workgroups of 256, two per CU: a
// wave's 64 rows one after another were most of such a call.  256 and 64 rows,
// triangle / 4-clique / diamond (us): 5 vertices joined to 300 48 / 88 / 108 and 33 /
// 67 / 66; R-MAT 10 80 / 154 / 156 and 62 / 124 / 106; R-MAT 11 98 / 227 / 195 and 78
// / 195 / 135.  Above the line some gain (R-MAT 12, 1,092 workgroups: 104 / 343 / 210
// and 81 / 305 / 141) and others lose (four G(600, 0.3), 1,548: triangles 95 and 114;
// the ranked R-MAT 16, 3,124: 322 and 364)
constexpr uint32_t kTableRows = 256, kTableRowsFew = 64, kTableFew = 512;

template <int kMode>
__global__ __launch_bounds__(kThreads) void CliqueRowsTableKernel(CliqueArgs a) {
  __shared__ u64 tab[kRowsTableRange / 32];  // bits 0..31: members, 32..: index of the first
  __shared__ u64 lds_row[kMode == kRowsBits ? kWaves : 1][kRowsTableMax / 64];
  // triangles through edge (v, u_j), two 16-bit counts per word (at most one
  // per row of the part), flushed with one atomic per j
  __shared__ uint32_t lds_col[kMode == kRowsEdges ? kRowsTableMax / 2 : 1];
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t wid = threadIdx.x / kWave;
  u64* row = lds_row[kMode == kRowsBits ? wid : 0];
  uint32_t* row32 = reinterpret_cast<uint32_t*>(row);
  u64 c3 = 0;
  for (uint64_t x = blockIdx.x; x < a.nverts; x += gridDim.x) {
    const uint32_t v = a.verts[x];
    const uint64_t nb = a.up[v];
    const uint32_t d = static_cast<uint32_t>(a.rp[v + 1] - nb);
    if (blockIdx.y * a.part >= d) continue;
    const uint32_t base = a.cols[nb], vmax = a.cols[nb + d - 1];
    if (!TableTakes(d, base, vmax)) continue;
    const uint32_t range = vmax - base + 1;
    const uint32_t W = (d + 63) / 64;
    __syncthreads();  // the previous vertex's lookups are done
    for (uint32_t k = threadIdx.x; k < (range + 31) / 32; k += kThreads) tab[k] = 0;
    __syncthreads();
    for (uint32_t j = threadIdx.x; j < d; j += kThreads) {
      const uint32_t off = a.cols[nb + j] - base;
      u64 add = 1ull << (off & 31);
      if (j == 0 || (a.cols[nb + j - 1] - base) >> 5 != off >> 5) add |= static_cast<u64>(j) << 32;
      atomicOr(tab + (off >> 5), add);
    }
    u64 mine = 0;  // triangles from v found by this lane
    for (uint32_t r0 = blockIdx.y * a.part; r0 < d; r0 += gridDim.y * a.part) {
      const uint32_t r1 = r0 + a.part < d ? r0 + a.part : d;
      if (kMode == kRowsEdges)
        for (uint32_t k = threadIdx.x; k < (d + 1) / 2; k += kThreads) lds_col[k] = 0;
      __syncthreads();
      // the next row's list bounds are loaded while this row streams
      uint32_t i = r0 + wid;
      uint64_t lb_next = 0, le_next = 0;
      if (i < r1) {
        const uint32_t u = a.cols[nb + i];
        lb_next = a.up[u];
        le_next = a.rp[u + 1];
      }
      for (; i < r1; i += kWaves) {
        const uint64_t lb = lb_next;
        const uint32_t len = static_cast<uint32_t>(le_next - lb_next);
        if (i + kWaves < r1) {
          const uint32_t u = a.cols[nb + i + kWaves];
          lb_next = a.up[u];
          le_next = a.rp[u + 1];
        }
        if (kMode == kRowsBits) {
          for (uint32_t w = lane; w < W; w += kWave) row[w] = 0;
          WaveSync();
        }
        const uint32_t* list = a.cols + lb;
        const bool middle = kMode == kRowsEdges && a.middles && len && MiddleTakes(len, list[0], list[len - 1]);
        constexpr uint32_t kNone = 0xffffffffu;
        uint32_t w0 = static_cast<uint32_t>(lane) < len ? list[lane] : kNone;
        uint32_t w1 = static_cast<uint32_t>(lane) + kWave < len ? list[lane + kWave] : kNone;
        uint32_t bits = 0;
        for (uint32_t e0 = 0; e0 < len; e0 += 2 * kWave) {
          // N+(u_i) is sorted: a step starting above the largest value of N+(v)
          // ends the row (lane 0 holds the step's first entry)
          if (static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(w0))) > vmax) break;
          const uint32_t x0 = w0, x1 = w1, e = e0 + static_cast<uint32_t>(lane);
          w0 = e + 2 * kWave < len ? list[e + 2 * kWave] : kNone;
          w1 = e + 3 * kWave < len ? list[e + 3 * kWave] : kNone;
          // every entry lies above u_i, so above base
          const uint32_t o0 = x0 - base, o1 = x1 - base;
          const u64 t0 = o0 < range ? tab[o0 >> 5] : 0, t1 = o1 < range ? tab[o1 >> 5] : 0;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const uint32_t o = h ? o1 : o0;
            const u64 t = h ? t1 : t0;
            const uint32_t members = static_cast<uint32_t>(t);  // (shifts take o & 31)
            if (!((members >> (o & 31)) & 1u)) continue;
            ++bits;
            if (kMode == kRowsCount) continue;
            const uint32_t j = static_cast<uint32_t>(t >> 32) +
                               static_cast<uint32_t>(__builtin_popcount(members & ((1u << (o & 31)) - 1u)));
            if (kMode == kRowsBits) atomicOr(row32 + (j >> 5), 1u << (j & 31));
            if (kMode == kRowsEdges) {
              if (!middle) atomicAdd(a.tc + lb + e + h * kWave, 1u);  // edge (u_i, u_j)
              atomicAdd(lds_col + (j >> 1), 1u << (16 * (j & 1)));  // edge (v, u_j)
            }
          }
        }
        if (kMode == kRowsBits) {
          u64* rows = a.rows + (a.word_first[x] - a.word_first[0]);
          WaveSync();
          for (uint32_t w = lane; w < W; w += kWave) rows[static_cast<uint64_t>(w) * d + i] = row[w];
          WaveSync();
        } else if (kMode == kRowsEdges) {
          // edge (v, u_i): one triangle per bit of row i
          const u64 tot = WaveSum(bits);
          if (lane == 0) {
            if (tot) atomicAdd(a.tc + nb + i, static_cast<uint32_t>(tot));
            c3 += tot;
          }
        } else {
          mine += bits;
        }
      }
      if (kMode == kRowsEdges) {
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < d; j += kThreads) {
          const uint32_t c = (lds_col[j >> 1] >> (16 * (j & 1))) & 0xffffu;
          if (c) atomicAdd(a.tc + nb + j, c);
        }
        __syncthreads();  // before the next part clears the counts
      }
    }
    if (kMode == kRowsCount) {
      c3 += mine;
      if (a.bk.bounds) AddBucket(a.bk, v, mine, lane);
    }
  }
  if (kMode != kRowsBits) BlockAdd<kThreads>(Into{a.acc + 3, c3});
}

// Per-edge counts of the middle edges (u, w) of the triangles v < u < w whose v
// the table kernel takes: one workgroup per u keeps N+(u) as such a table and a
// count per u_j in LDS, and walks what follows u in N+(v) for its lower
// neighbours v.  Each v's list is read from its middle only, 0.4 times the
// entries of the row pass, and a triangle costs an LDS add here where it cost a
// device atomic there.  R-MAT scale 20 (degree-ranked, 4.2e8 triangles): per-edge
// counts 6.5 -> 4.0 + 2.0 ms.
__global__ __launch_bounds__(kThreads) void CliqueMiddleKernel(CliqueArgs a) {
  __shared__ u64 tab[kRowsTableRange / 32];
  __shared__ uint32_t col[kMiddleMax];
  __shared__ WalkLds walk_all[kWaves];
  __shared__ uint32_t any;
  const int lane = threadIdx.x & (kWave - 1);
  WalkLds& walk = walk_all[threadIdx.x / kWave];
  for (uint64_t y = blockIdx.x; y < a.v_end - a.v_begin; y += gridDim.x) {
    const uint32_t u = a.v_begin + static_cast<uint32_t>(y);
    const uint64_t rb = a.rp[u], nb = a.up[u];
    const uint32_t d = static_cast<uint32_t>(a.rp[u + 1] - nb);
    if (d == 0) continue;
    const uint32_t base = a.cols[nb], umax = a.cols[nb + d - 1];
    if (!MiddleTakes(d, base, umax)) continue;
    const uint32_t range = umax - base + 1;
    bool built = false;
    for (uint64_t k0 = rb; k0 < nb; k0 += kThreads) {
      const uint64_t k = k0 + threadIdx.x;
      uint64_t lb = 0;
      uint32_t len = 0;
      if (k < nb) {
        const uint32_t v = a.cols[k];
        const uint64_t vb = a.up[v], ve = a.rp[v + 1];
        const uint64_t dv = ve - vb;
        if (dv > kLocalSmall && dv <= kRowsTableMax && TableTakes(static_cast<uint32_t>(dv), a.cols[vb], a.cols[ve - 1])) {
          uint64_t lo = vb, hi = ve;  // the first entry above u
          while (lo < hi) {
            const uint64_t mid = (lo + hi) >> 1;
            if (a.cols[mid] <= u)
              lo = mid + 1;
            else
              hi = mid;
          }
          lb = lo;
          len = static_cast<uint32_t>(ve - lo);
        }
      }
      if (!built) {
        __syncthreads();  // readers of the previous u's counts and of `any` are done
        if (threadIdx.x == 0) any = 0;
        __syncthreads();
        if (len) any = 1;
        __syncthreads();
        if (!any) continue;
        built = true;
        for (uint32_t w = threadIdx.x; w < (range + 31) / 32; w += kThreads) tab[w] = 0;
        for (uint32_t j = threadIdx.x; j < d; j += kThreads) col[j] = 0;
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < d; j += kThreads) {
          const uint32_t off = a.cols[nb + j] - base;
          u64 add = 1ull << (off & 31);
          if (j == 0 || (a.cols[nb + j - 1] - base) >> 5 != off >> 5) add |= static_cast<u64>(j) << 32;
          atomicOr(tab + (off >> 5), add);
        }
        __syncthreads();
      }
      WalkLists<false>(a.cols, nullptr, lb, len, 0u, walk, lane, [&](uint32_t w, uint32_t, uint32_t) {
        const uint32_t o = w - base;  // (w < base wraps around)
        if (o >= range) return;
        const u64 t = tab[o >> 5];
        const uint32_t members = static_cast<uint32_t>(t);
        if (!((members >> (o & 31)) & 1u)) return;
        atomicAdd(col + static_cast<uint32_t>(t >> 32) +
                      static_cast<uint32_t>(__builtin_popcount(members & ((1u << (o & 31)) - 1u))),
                  1u);
      });
    }
    if (!built) continue;
    __syncthreads();
    for (uint32_t j = threadIdx.x; j < d; j += kThreads)
      if (col[j]) atomicAdd(a.tc + nb + j, col[j]);
  }
}

// One workgroup per chunk of 64 rows of one vertex v.  N+(v) goes into an LDS
// hash table (value -> local index j, at most half full); each wave then
// builds rows of the chunk by streaming N+(u_i) up to the largest value of
// N+(v), 64 consecutive entries per load, and setting bit j of the row (an
// LDS OR) for every entry found.  Every entry of N+(u_i) lies above u_i, so
// the bits set are exactly those j > i with u_j in N+(u_i).
template <int kBits>
__global__ __launch_bounds__(kThreads) void CliqueRowsHashKernel(CliqueArgs a) {
  constexpr uint32_t kSlots = 1u << kBits;
  constexpr uint32_t kEmptyKey = 0xffffffffu;
  __shared__ uint32_t lds_key[kSlots];
  __shared__ uint16_t lds_idx[kSlots];
  __shared__ u64 lds_row[kWaves][kRowsHashMax / 64];
  // per-edge counts (tc): the chunk's triangles through edge (v, u_j),
  // flushed with one atomic per j
  __shared__ uint32_t lds_col[kSlots / 2];
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = threadIdx.x / kWave;
  u64* row = lds_row[wid];
  u64 c3 = 0;
  for (uint64_t t = blockIdx.x; t < a.nchunks; t += gridDim.x) {
    const uint64_t x = ChunkVertex(a, t);
    const uint32_t v = a.verts[x];
    const uint32_t d = static_cast<uint32_t>(a.row_first[x + 1] - a.row_first[x]);
    const uint32_t W = (d + 63) / 64;
    const uint32_t r0 = static_cast<uint32_t>(t - (a.chunk_first[x] - a.chunk_first[0])) * 64;
    const uint32_t r1 = r0 + 64 < d ? r0 + 64 : d;
    const uint64_t nb = a.up[v];
    if (TableTakes(d, a.cols[nb], a.cols[nb + d - 1])) continue;
    u64* rows = a.rows + (a.word_first[x] - a.word_first[0]);
    __syncthreads();  // the previous chunk's lookups are done
    for (uint32_t k = threadIdx.x; k < kSlots; k += kThreads) lds_key[k] = kEmptyKey;
    if (a.tc)
      for (uint32_t k = threadIdx.x; k < d; k += kThreads) lds_col[k] = 0;
    __syncthreads();
    for (uint32_t j = threadIdx.x; j < d; j += kThreads) {
      const uint32_t w = a.cols[nb + j];
      uint32_t h = (w * 0x9E3779B1u) >> (32 - kBits);
      while (atomicCAS(lds_key + h, kEmptyKey, w) != kEmptyKey) h = (h + 1) & (kSlots - 1);
      lds_idx[h] = static_cast<uint16_t>(j);
    }
    __syncthreads();
    const uint32_t vmax = a.cols[nb + d - 1];
    // the next row's vertex and list bounds are loaded while this row streams
    uint32_t i = r0 + wid;
    uint64_t lb_next = 0, le_next = 0;
    if (i < r1) {
      const uint32_t u = a.cols[nb + i];
      lb_next = a.up[u];
      le_next = a.rp[u + 1];
    }
    u64 mine = 0;  // triangles from v found by this lane
    for (; i < r1; i += kWaves) {
      const uint64_t lb = lb_next, le = le_next;
      if (i + kWaves < r1) {
        const uint32_t u = a.cols[nb + i + kWaves];
        lb_next = a.up[u];
        le_next = a.rp[u + 1];
      }
      for (uint32_t w = lane; w < W; w += kWave) row[w] = 0;
      WaveSync();
      uint32_t bits = 0;
      // chunks of 64 entries, the next chunk's load issued before this
      // chunk's lookups
      uint64_t e0 = lb;
      uint32_t wcur = lb + lane < le ? a.cols[lb + lane] : kEmptyKey;
      while (e0 < le) {
        // N+(u_i) is sorted: nothing from a chunk starting above the
        // largest value of N+(v) on can be found (lane 0 holds the chunk's
        // first entry)
        if (static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(wcur))) > vmax) break;
        const uint64_t n0 = e0 + kWave;
        const uint32_t wnext = n0 + lane < le ? a.cols[n0 + lane] : kEmptyKey;
        const uint64_t e = e0 + lane;
        const uint32_t w = wcur;
        e0 = n0;
        wcur = wnext;
        if (e < le) {
          uint32_t h = (w * 0x9E3779B1u) >> (32 - kBits);
          uint32_t k;
          while ((k = lds_key[h]) != w && k != kEmptyKey) h = (h + 1) & (kSlots - 1);
          if (k == w) {
            const uint32_t j = lds_idx[h];
            if (a.rows) atomicOr(row + (j >> 6), 1ull << (j & 63));
            ++bits;
            if (a.tc) {
              atomicAdd(a.tc + e, 1u);     // edge (u_i, u_j)
              atomicAdd(lds_col + j, 1u);  // edge (v, u_j)
            }
          }
        }
      }
      WaveSync();
      if (a.rows)
        for (uint32_t w = lane; w < W; w += kWave) rows[static_cast<uint64_t>(w) * d + i] = row[w];
      if (!a.rows) {
        // edge (v, u_i): one triangle per bit of row i (with rows the count
        // kernel takes the row's popcount)
        const u64 tot = WaveSum(bits);
        if (lane == 0) {
          if (a.tc && tot) atomicAdd(a.tc + nb + i, static_cast<uint32_t>(tot));
          c3 += tot;
        }
        mine += bits;
      }
      WaveSync();
    }
    if (!a.rows && a.bk.bounds) AddBucket(a.bk, v, mine, lane);
    if (a.tc) {
      __syncthreads();
      for (uint32_t j = threadIdx.x; j < d; j += kThreads)
        if (lds_col[j]) atomicAdd(a.tc + nb + j, lds_col[j]);
    }
  }
  if (!a.rows) BlockAdd<kThreads>(Into{a.acc + 3, c3});
}

// |s & row_j| over the words of row j that can be non-zero (bits above j).
// Rows are stored word-major (word w of row j at rows[w * d + j]), so the
// lanes of a probe round, holding nearby members j, read nearby addresses.
__device__ __forceinline__ u64 Probe(const u64* s, uint32_t W, uint32_t d, const u64* rows, uint32_t j) {
  const u64* r = rows + j;
  u64 x = 0;
  for (uint32_t w = (j + 1) >> 6; w < W; ++w) x += __popcll(s[w] & r[static_cast<uint64_t>(w) * d]);
  return x;
}

// Sum over the members j of s (words [lo, W), in LDS) of |s & row_j|, as
// per-lane partial sums.  Members are queued in LDS (q: 2 x 64 entries) so
// every probe round has 64 of them, whatever the density of s.
__device__ __forceinline__ u64 LastLevel(const u64* s, uint32_t lo, uint32_t W, uint32_t d, const u64* rows, uint32_t* q,
                         int lane) {
  const u64 below = lane ? (~0ull >> (64 - lane)) : 0ull;
  u64 sum = 0;
  uint32_t qn = 0;
  for (uint32_t c = lo; c < W; ++c) {
    const u64 bits = First64(s[c]);
    if (!bits) continue;
    if ((bits >> lane) & 1) q[qn + __popcll(bits & below)] = c * 64 + static_cast<uint32_t>(lane);
    qn += __popcll(bits);
    if (qn >= static_cast<uint32_t>(kWave)) {
      WaveSync();
      sum += Probe(s, W, d, rows, q[lane]);
      const uint32_t rest = qn - kWave;
      const uint32_t carry = static_cast<uint32_t>(lane) < rest ? q[kWave + lane] : 0u;
      WaveSync();
      if (static_cast<uint32_t>(lane) < rest) q[lane] = carry;
      qn = rest;
      WaveSync();
    }
  }
  if (qn) {
    WaveSync();
    if (static_cast<uint32_t>(lane) < qn) sum += Probe(s, W, d, rows, q[lane]);
  }
  WaveSync();
  return sum;
}

struct CliqueSums {
  u64 c3 = 0, c4 = 0, c5 = 0, c6 = 0;
};

// The cliques from row i of a vertex with d upper neighbours whose rows are
// stored word-major at `rows` (device memory or LDS): s1 = row i, and for
// K >= 5 every s2 = s1 & row j (j in s1), s3 = s2 & row l, each kept in the
// wave's LDS buffers while the members below it are walked; the last set's
// members are probed by LastLevel.  Adds the level counts to *cs and
// returns this lane's share of the k-cliques.
template <int K>
__device__ __forceinline__ u64 CountRow(const u64* rows, uint32_t d, uint32_t i, u64* s1, u64* s2, u64* s3,
                                        uint32_t* q, int lane, CliqueSums* cs) {
  const uint32_t W = (d + 63) / 64;
  const u64* ri = rows + i;
  const uint32_t lo1 = (i + 1) >> 6;
  u64 vk = 0;
  WaveSync();
  for (uint32_t w = lo1 + lane; w < W; w += kWave) {
    const u64 xw = ri[static_cast<uint64_t>(w) * d];
    s1[w] = xw;
    cs->c3 += __popcll(xw);
  }
  WaveSync();
  if (K == 4) {
    const u64 y = LastLevel(s1, lo1, W, d, rows, q, lane);
    cs->c4 += y;
    return vk + y;
  }
  for (uint32_t c = lo1; c < W; ++c) {
    for (u64 m1 = First64(s1[c]); m1; m1 &= m1 - 1) {
      const uint32_t j = c * 64 + static_cast<uint32_t>(__builtin_ctzll(m1));
      const u64* rj = rows + j;
      const uint32_t lo2 = (j + 1) >> 6;
      u64 nz = 0;
      WaveSync();
      for (uint32_t w = lo2 + lane; w < W; w += kWave) {
        const u64 xw = s1[w] & rj[static_cast<uint64_t>(w) * d];
        s2[w] = xw;
        cs->c4 += __popcll(xw);
        nz |= xw;
      }
      if (!__ballot(nz != 0)) continue;
      WaveSync();
      if (K == 5) {
        const u64 y = LastLevel(s2, lo2, W, d, rows, q, lane);
        cs->c5 += y;
        vk += y;
        continue;
      }
      for (uint32_t c2 = lo2; c2 < W; ++c2) {
        for (u64 m2 = First64(s2[c2]); m2; m2 &= m2 - 1) {
          const uint32_t l = c2 * 64 + static_cast<uint32_t>(__builtin_ctzll(m2));
          const u64* rl = rows + l;
          const uint32_t lo3 = (l + 1) >> 6;
          u64 nz3 = 0;
          WaveSync();
          for (uint32_t w = lo3 + lane; w < W; w += kWave) {
            const u64 xw = s2[w] & rl[static_cast<uint64_t>(w) * d];
            s3[w] = xw;
            cs->c5 += __popcll(xw);
            nz3 |= xw;
          }
          if (!__ballot(nz3 != 0)) continue;
          WaveSync();
          const u64 y = LastLevel(s3, lo3, W, d, rows, q, lane);
          cs->c6 += y;
          vk += y;
        }
      }
    }
  }
  return vk;
}

__device__ __forceinline__ void FlushSums(unsigned long long* acc, int K, const CliqueSums& cs) {
  BlockAdd<kThreads>(Into{acc + 3, cs.c3},
                     Into{acc + 4, cs.c4},
                     Into{K >= 5 ? acc + 5 : nullptr, cs.c5},
                     Into{K >= 6 ? acc + 6 : nullptr, cs.c6});
}

// 5- and 6-cliques.  The m members of row i span W words, most of whose bits
// are not members.  Their rows are first packed to the members' columns: lane =
// member j reads the words of row j, and for each set bit of row i (the same
// for all lanes) one bit of the word moves to the next packed place.  What is
// left to count is the triangles of a graph of m vertices held as m rows of
// ceil(m / 32) words in LDS.  For 5-cliques lane = row j keeps its row in
// registers and all lanes meet the same row l at a time (an LDS broadcast, no
// bank conflicts): popcount(row_j & row_l) counts where row j has bit l.
//
// Bound by VALU issue (three quarters of the cycles in the long rows).  R-MAT
// scale 19, edge factor 32, 5-clique: 160 ms when each row j below i was
// intersected by a wave (W of 64 lanes busy) and its members probed rows in
// device memory; 92 ms packed (26 ms rows of up to 128 members, 35 up to 256,
// 30 up to 512).  Walking each lane's own bits instead of meeting rows by
// broadcast took 173 ms: the random LDS rows conflict and the lanes' bit counts
// differ.  6-cliques walk bits all the same: their inner sets differ by lane.

// Words between packed rows of NW words: 16-byte aligned from 4 words on, and
// an odd multiple of 4 so that 64 rows spread over 16 banks.
constexpr uint32_t PackStride(int nw) { return nw < 4 ? nw : nw % 8 == 4 ? nw : nw + 4; }

// Packs the rows of members r = lane + 64 g (j = mem[r], r < m), g < G, taking
// the words [w0, w1) of row i (s1), whose first set bit is packed bit `pos`.
// pack must be zero.
template <int G, int NW>
__device__ __forceinline__ void PackRows(const u64* rows, uint32_t d, const u64* s1, uint32_t w0, uint32_t w1,
                                         uint32_t pos, const uint16_t* mem, uint32_t m, uint32_t* pack, int lane) {
  if (w0 >= w1) return;
  const u64* rj[G];
  u64 next[G];
  uint32_t cur[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const uint32_t r = static_cast<uint32_t>(lane) + g * kWave;
    rj[g] = r < m ? rows + mem[r] : nullptr;
    next[g] = rj[g] ? rj[g][static_cast<uint64_t>(w0) * d] : 0;
    cur[g] = 0;
  }
  auto flush = [&](uint32_t k) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (cur[g]) atomicOr(pack + (static_cast<uint32_t>(lane) + g * kWave) * PackStride(NW) + k, cur[g]);
      cur[g] = 0;
    }
  };
  for (uint32_t w = w0; w < w1; ++w) {
    u64 x[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      x[g] = next[g];
      if (w + 1 < w1 && rj[g]) next[g] = rj[g][static_cast<uint64_t>(w + 1) * d];
    }
    const u64 mask = First64(s1[w]);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      for (uint32_t mk = static_cast<uint32_t>(mask >> (32 * h)); mk; mk &= mk - 1) {
        const uint32_t b = static_cast<uint32_t>(__builtin_ctz(mk));
#pragma unroll
        for (int g = 0; g < G; ++g)
          cur[g] |= ((static_cast<uint32_t>(x[g] >> (32 * h)) >> b) & 1u) << (pos & 31);
        if ((++pos & 31) == 0) flush((pos >> 5) - 1);
      }
    }
  }
  if (pos & 31) flush(pos >> 5);
}

// The pairs and triangles of row r of a packed graph of m rows, meeting the
// rows of the words w with w % parts == part.
template <int NW>
__device__ __forceinline__ u64 CountPacked5(const uint32_t* pack, uint32_t m, uint32_t r, uint32_t first,
                                            uint32_t parts, uint32_t part, CliqueSums* cs) {
  constexpr uint32_t S = PackStride(NW);
  uint32_t c[NW];
#pragma unroll
  for (uint32_t k = 0; k < NW; ++k) c[k] = r < m ? pack[r * S + k] : 0u;
  uint32_t pairs = 0;
  u64 x5 = 0;
#pragma unroll
  for (uint32_t w = 0; w < NW; ++w) {
    // (rows below `first`, the wave's first, have no bit in any of its rows)
    if (w * 32 >= m || w < first / 32 || (parts > 1 && w % parts != part)) continue;
    pairs += __builtin_popcount(c[w]);
    const uint32_t* pl = pack + w * 32 * S;
    const uint32_t n = m - w * 32 < 32 ? m - w * 32 : 32;
    uint32_t x = 0;
#pragma unroll 2
    for (uint32_t b = 0; b < n; ++b, pl += S) {
      uint32_t y = 0;
#pragma unroll
      for (uint32_t k = w; k < NW; ++k) y += __builtin_popcount(c[k] & pl[k]);
      x += y & (0u - ((c[w] >> b) & 1u));  // (a multiply is quarter rate)
    }
    x5 += x;
  }
  cs->c4 += pairs;
  cs->c5 += x5;
  return x5;
}

// 6-cliques: row r's pairs and triangles, and the 4-cliques below it, each
// lane walking the bits of its own row.
template <int NW>
__device__ __forceinline__ u64 CountPacked6(const uint32_t* pack, uint32_t m, uint32_t r, CliqueSums* cs) {
  constexpr uint32_t S = PackStride(NW);
  if (r >= m) return 0;
  uint32_t c[NW];
  uint32_t pairs = 0;
#pragma unroll
  for (uint32_t k = 0; k < NW; ++k) {
    c[k] = pack[r * S + k];
    pairs += __builtin_popcount(c[k]);
  }
  u64 x5 = 0, x6 = 0;
#pragma unroll
  for (uint32_t w = 0; w < NW; ++w) {
    for (uint32_t bits = c[w]; bits; bits &= bits - 1) {
      const uint32_t* pl = pack + (w * 32 + __builtin_ctz(bits)) * S;
      uint32_t t[NW];
#pragma unroll
      for (uint32_t k = 0; k < NW; ++k) {
        t[k] = k >= w ? c[k] & pl[k] : 0u;
        x5 += __builtin_popcount(t[k]);
      }
#pragma unroll
      for (uint32_t k = 0; k < NW; ++k) {
        for (uint32_t b2 = t[k]; b2; b2 &= b2 - 1) {
          const uint32_t* pq = pack + (k * 32 + __builtin_ctz(b2)) * S;
          uint32_t s6 = 0;
#pragma unroll
          for (uint32_t k2 = k; k2 < NW; ++k2) s6 += __builtin_popcount(t[k2] & pq[k2]);
          x6 += s6;
        }
      }
    }
  }
  cs->c4 += pairs;
  cs->c5 += x5;
  cs->c6 += x6;
  return x6;
}

// One row of at most 32 NW members by one wave.
template <int K, int NW>
__device__ __forceinline__ u64 CountWave(const u64* rows, uint32_t d, uint32_t i, const u64* s1, const uint16_t* mem,
                                         uint32_t m, uint32_t* pack, int lane, CliqueSums* cs) {
  constexpr int G = NW > 2 ? NW / 2 : 1;
  for (uint32_t k = lane; k < m * PackStride(NW); k += kWave) pack[k] = 0;
  WaveSync();
  PackRows<G, NW>(rows, d, s1, (i + 1) >> 6, (d + 63) / 64, 0, mem, m, pack, lane);
  WaveSync();
  u64 vk = 0;
  for (uint32_t r = 0; r < m; r += kWave)
    vk += K == 5 ? CountPacked5<NW>(pack, m, r + lane, r, 1, 0, cs) : CountPacked6<NW>(pack, m, r + lane, cs);
  return vk;
}

// 4-cliques of the vertices with d > kDenseMax: a wave takes groups of
// kRowGroup consecutive rows, one search for the group's first vertex, then a
// walk forward (a row is light next to the search).  A bucket gets one sum per group
// and vertex: with one per row 16 buckets of R-MAT 14, factor 8, took 0.88 ms, now
// 0.63.  (Held to 64 registers, without which the sum takes an eighth of the waves.)
__global__ __launch_bounds__(kThreads, 8) void CliqueCount4Kernel(CliqueArgs a) {
  __shared__ u64 lds_s[kWaves][kWordsMax];
  __shared__ uint32_t lds_q[kWaves][2 * kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = threadIdx.x / kWave;
  const uint64_t wave = (blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x) / kWave;
  const uint64_t nwaves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  CliqueSums cs;
  constexpr uint64_t kRowGroup = 16;
  const uint64_t base = a.row_first[0];
  for (uint64_t t0 = wave * kRowGroup; t0 < a.nitems; t0 += nwaves * kRowGroup) {
    const uint64_t te = t0 + kRowGroup < a.nitems ? t0 + kRowGroup : a.nitems;
    uint64_t x = ItemVertexWave(a, t0, lane), of = x;
    u64 vk = 0;  // this group's share of the 4-cliques from vertex `of`
    for (uint64_t t = t0; t < te; ++t) {
      while (a.row_first[x + 1] - base <= t) ++x;
      if (a.bk.bounds && x != of) {
        AddBucket(a.bk, a.verts[of], vk, lane);
        vk = 0;
        of = x;
      }
      const uint32_t d = static_cast<uint32_t>(a.row_first[x + 1] - a.row_first[x]);
      const uint32_t i = static_cast<uint32_t>(t - (a.row_first[x] - base));
      const u64* rows = a.rows + (a.word_first[x] - a.word_first[0]);
      vk += CountRow<4>(rows, d, i, lds_s[wid], nullptr, nullptr, lds_q[wid], lane, &cs);
    }
    if (a.bk.bounds) AddBucket(a.bk, a.verts[of], vk, lane);
  }
  FlushSums(a.acc, 4, cs);
}

// 4-cliques of the vertices with 32 (NW - 4) < d <= 32 NW: the pairs and
// triangles of the graph on N+(v), whose d rows one workgroup reads once, in
// order, into LDS.
//
// Bound by VALU issue.  R-MAT scale 20 (60,395 vertices): 1.0 ms with the few above kDenseMax; one wave
// per row, probing its members' rows in device memory, took 3.2.  Meeting every
// row, member or not, costs d^2 / 128 steps of a wave against one per 64
// members: above kDenseMax the members are few enough that probing them wins.
template <int NW>
__global__ __launch_bounds__(kThreads) void CliqueDenseKernel(CliqueArgs a) {
  constexpr uint32_t S = PackStride(NW);
  __shared__ __align__(16) uint32_t pack[32 * NW * S];
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t wid = threadIdx.x / kWave;
  CliqueSums cs;
  for (uint64_t x = blockIdx.x; x < a.nverts; x += gridDim.x) {
    const uint32_t d = static_cast<uint32_t>(a.row_first[x + 1] - a.row_first[x]);
    const uint32_t W = (d + 63) / 64;
    const u64* rows = a.rows + (a.word_first[x] - a.word_first[0]);
    __syncthreads();  // the previous vertex's readers are done
    for (uint32_t w = 0; w < NW / 2; ++w)
      for (uint32_t i = threadIdx.x; i < d; i += kThreads) {
        const u64 y = w < W ? rows[static_cast<uint64_t>(w) * d + i] : 0;
        pack[i * S + 2 * w] = static_cast<uint32_t>(y);
        pack[i * S + 2 * w + 1] = static_cast<uint32_t>(y >> 32);
      }
    __syncthreads();
    u64 vk = 0;
    for (uint32_t r = 0; r < d; r += kWave) vk += CountPacked5<NW>(pack, d, r + lane, r, kWaves, wid, &cs);
    if (a.bk.bounds) AddBucket(a.bk, a.verts[x], vk, lane);
  }
  // (pairs of the graph on N+(v) are triangles, its triangles 4-cliques)
  BlockAdd<kThreads>(Into{a.acc + 3, cs.c4}, Into{a.acc + 4, cs.c5});
}

// Row i into s1 (LDS), its members in order into mem (at most cap); returns
// their number.  All lanes of the wave.
__device__ __forceinline__ uint32_t LoadRow(const u64* rows, uint32_t d, uint32_t i, u64* s1, uint16_t* mem,
                                            uint32_t cap, int lane) {
  const uint32_t W = (d + 63) / 64, lo1 = (i + 1) >> 6;
  const u64 below = lane ? (~0ull >> (64 - lane)) : 0ull;
  WaveSync();  // readers of the previous row are done
  for (uint32_t w = lo1 + lane; w < W; w += kWave) s1[w] = rows[static_cast<uint64_t>(w) * d + i];
  WaveSync();
  uint32_t m = 0;
  for (uint32_t w = lo1; w < W; ++w) {
    const u64 bits = First64(s1[w]);
    const uint32_t at = m + static_cast<uint32_t>(__popcll(bits & below));
    if (((bits >> lane) & 1) && at < cap) mem[at] = static_cast<uint16_t>(w * 64 + lane);
    m += static_cast<uint32_t>(__popcll(bits));
  }
  WaveSync();
  return m;
}

constexpr uint32_t kPackWave = 128;  // members a wave packs

// One wave per row with at most kPackWave members.  Longer rows are left to
// CliqueLongKernel in a.long_rows: up to 256 members from the front, the others
// from the back.
template <int K>
__global__ __launch_bounds__(kThreads) void CliquePackKernel(CliqueArgs a) {
  __shared__ u64 lds_s[kWaves][kWordsMax];
  __shared__ __align__(16) uint32_t lds_pack[kWaves][PackStride(kPackWave / 32) * kPackWave];
  __shared__ uint16_t lds_mem[kWaves][kPackWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = threadIdx.x / kWave;
  u64* s1 = lds_s[wid];
  uint32_t* pack = lds_pack[wid];
  uint16_t* mem = lds_mem[wid];
  const uint64_t wave = (blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x) / kWave;
  const uint64_t nwaves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  CliqueSums cs;
  const uint64_t base = a.row_first[0];
  constexpr uint64_t kRowGroup = 4;
  for (uint64_t t0 = wave * kRowGroup; t0 < a.nitems; t0 += nwaves * kRowGroup) {
    const uint64_t te = t0 + kRowGroup < a.nitems ? t0 + kRowGroup : a.nitems;
    uint64_t x = ItemVertexWave(a, t0, lane);
    for (uint64_t t = t0; t < te; ++t) {
      while (a.row_first[x + 1] - base <= t) ++x;
      const uint32_t d = static_cast<uint32_t>(a.row_first[x + 1] - a.row_first[x]);
      const uint32_t i = static_cast<uint32_t>(t - (a.row_first[x] - base));
      const u64* rows = a.rows + (a.word_first[x] - a.word_first[0]);
      const uint32_t m = LoadRow(rows, d, i, s1, mem, kPackWave, lane);
      if (m > kPackWave) {
        if (lane == 0) {
          const bool back = K != 5 || m > 256;
          const u64 at = atomicAdd(a.nlong + (back ? 1 : 0), 1ull);
          a.long_rows[back ? a.nitems - 1 - at : at] = static_cast<uint32_t>(t);
        }
        continue;
      }
      if (lane == 0) cs.c3 += m;
      const u64 vk = m <= 32   ? CountWave<K, 1>(rows, d, i, s1, mem, m, pack, lane, &cs)
                     : m <= 64 ? CountWave<K, 2>(rows, d, i, s1, mem, m, pack, lane, &cs)
                               : CountWave<K, 4>(rows, d, i, s1, mem, m, pack, lane, &cs);
      if (a.bk.bounds) AddBucket(a.bk, a.verts[x], vk, lane);
    }
  }
  FlushSums(a.acc, K, cs);
}

// 5-cliques of the long rows with at most 32 NW members, one workgroup each,
// every wave packing a share of the columns and meeting a share of the rows.
// kBack: the rows from the back of the list (longer ones among them are left to
// CliqueUnpackedKernel).
template <int NW, bool kBack>
__global__ __launch_bounds__(kThreads) void CliqueLongKernel(CliqueArgs a) {
  constexpr uint32_t kCap = 32 * NW;
  __shared__ u64 s1[kWordsMax];
  __shared__ __align__(16) uint32_t pack[PackStride(NW) * kCap];
  __shared__ uint16_t mem[kCap];
  __shared__ uint32_t members;
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t wid = threadIdx.x / kWave;
  CliqueSums cs;
  const uint64_t base = a.row_first[0];
  const uint64_t nlong = a.nlong[kBack ? 1 : 0];
  for (uint64_t y = blockIdx.x; y < nlong; y += gridDim.x) {
    const uint64_t t = a.long_rows[kBack ? a.nitems - 1 - y : y];
    const uint64_t x = ItemVertexWave(a, t, lane);
    const uint32_t d = static_cast<uint32_t>(a.row_first[x + 1] - a.row_first[x]);
    const uint32_t i = static_cast<uint32_t>(t - (a.row_first[x] - base));
    const u64* rows = a.rows + (a.word_first[x] - a.word_first[0]);
    __syncthreads();  // the previous row's readers are done
    if (wid == 0) {
      const uint32_t m = LoadRow(rows, d, i, s1, mem, kCap, lane);
      if (lane == 0) members = m;
    }
    for (uint32_t k = threadIdx.x; k < PackStride(NW) * kCap; k += kThreads) pack[k] = 0;
    __syncthreads();
    const uint32_t m = members;
    if (m > kCap) continue;
    if (threadIdx.x == 0) cs.c3 += m;
    const uint32_t W = (d + 63) / 64, lo1 = (i + 1) >> 6;
    const uint32_t share = (W - lo1 + kWaves - 1) / kWaves;
    const uint32_t w0 = lo1 + wid * share < W ? lo1 + wid * share : W, w1 = w0 + share < W ? w0 + share : W;
    uint32_t pos = 0;
    for (uint32_t w = lo1; w < w0; ++w) pos += static_cast<uint32_t>(__popcll(First64(s1[w])));
    PackRows<(NW + 1) / 2, NW>(rows, d, s1, w0, w1, pos, mem, m, pack, lane);
    __syncthreads();
    u64 vk = 0;
    for (uint32_t r = 0; r < m; r += kWave) vk += CountPacked5<NW>(pack, m, r + lane, r, kWaves, wid, &cs);
    if (a.bk.bounds) AddBucket(a.bk, a.verts[x], vk, lane);
  }
  FlushSums(a.acc, 5, cs);
}

// The rows at the back of the list that are not packed, one wave each: 5-clique
// rows with more than kPackLong members, and all long rows of 6-cliques.
constexpr uint32_t kPackLong = 512;

template <int K>
__global__ __launch_bounds__(kThreads) void CliqueUnpackedKernel(CliqueArgs a) {
  constexpr int kBufs = K - 3;
  __shared__ u64 lds_s[kWaves][kBufs][kWordsMax];
  __shared__ uint32_t lds_q[kWaves][2 * kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = threadIdx.x / kWave;
  const uint64_t wave = (blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x) / kWave;
  const uint64_t nwaves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  CliqueSums cs;
  const uint64_t base = a.row_first[0];
  const uint64_t nlong = a.nlong[1];
  for (uint64_t y = wave; y < nlong; y += nwaves) {
    const uint64_t t = a.long_rows[a.nitems - 1 - y];
    const uint64_t x = ItemVertexWave(a, t, lane);
    const uint32_t d = static_cast<uint32_t>(a.row_first[x + 1] - a.row_first[x]);
    const uint32_t i = static_cast<uint32_t>(t - (a.row_first[x] - base));
    const u64* rows = a.rows + (a.word_first[x] - a.word_first[0]);
    if (K == 5) {
      u64 m = 0;
      for (uint32_t w = lane; w < (d + 63) / 64; w += kWave) m += __popcll(rows[static_cast<uint64_t>(w) * d + i]);
      if (First64(WaveSum(m)) <= kPackLong) continue;
    }
    const u64 vk = CountRow<K>(rows, d, i, lds_s[wid][0], lds_s[wid][kBufs > 1 ? 1 : 0], lds_s[wid][kBufs > 2 ? 2 : 0],
                               lds_q[wid], lane, &cs);
    if (a.bk.bounds) AddBucket(a.bk, a.verts[x], vk, lane);
  }
  FlushSums(a.acc, K, cs);
}

}  // namespace

void LaunchCliqueSmall(const CliqueArgs& a, hipStream_t stream) {
  if (a.v_end <= a.v_begin) return;
  // few start vertices: one per wave, so that the launch spreads over the chip
  const uint64_t nv = a.v_end - a.v_begin;
  CliqueArgs b = a;
  b.group = nv > kSmallAlone ? kSmallGroup : 1;
  const uint64_t need = Grid((nv + b.group - 1) / b.group, kWaves);
  const uint64_t most = nv > 4 * kSmallAlone ? kSmallGrid : kSmallGridFew;
  const dim3 grid(need < most ? need : most), block(kThreads);
  switch (a.k) {
    case 3: hipLaunchKernelGGL(CliqueSmallKernel<3>, grid, block, 0, stream, b); break;
    case 4: hipLaunchKernelGGL(CliqueSmallKernel<4>, grid, block, 0, stream, b); break;
    case 5: hipLaunchKernelGGL(CliqueSmallKernel<5>, grid, block, 0, stream, b); break;
    case 6: hipLaunchKernelGGL(CliqueSmallKernel<6>, grid, block, 0, stream, b); break;
  }
}

void LaunchCliqueRows(const CliqueArgs& a, hipStream_t stream) {
  if (a.nitems == 0) return;
  hipLaunchKernelGGL(CliqueRowsKernel, dim3(Grid(a.nitems, kWaves)), dim3(kThreads), 0, stream, a);
}

void LaunchCliqueRowsTable(const CliqueArgs& a, uint32_t dmax, hipStream_t stream) {
  if (a.nverts == 0) return;
  if (dmax > kRowsTableMax) dmax = kRowsTableMax;
  // parts of one vertex run side by side where the vertices alone would not
  // fill the chip several times over
  CliqueArgs b = a;
  b.part = a.nverts * ((dmax + kTableRows - 1) / kTableRows) < kTableFew ? kTableRowsFew : kTableRows;
  uint32_t parts = (dmax + b.part - 1) / b.part;
  if (a.nverts > 4096 && parts > 4) parts = 4;
  const dim3 grid(Grid(a.nverts, 1), parts), block(kThreads);
  if (a.tc)
    hipLaunchKernelGGL(CliqueRowsTableKernel<kRowsEdges>, grid, block, 0, stream, b);
  else if (a.rows)
    hipLaunchKernelGGL(CliqueRowsTableKernel<kRowsBits>, grid, block, 0, stream, b);
  else
    hipLaunchKernelGGL(CliqueRowsTableKernel<kRowsCount>, grid, block, 0, stream, b);
}

void LaunchCliqueMiddles(const CliqueArgs& a, hipStream_t stream) {
  if (a.v_end <= a.v_begin) return;
  hipLaunchKernelGGL(CliqueMiddleKernel, dim3(Grid(a.v_end - a.v_begin, 1)), dim3(kThreads), 0, stream, a);
}

void LaunchCliqueRowsHash(const CliqueArgs& a, bool small_table, hipStream_t stream) {
  if (a.nchunks == 0) return;
  const dim3 grid(Grid(a.nchunks, 1)), block(kThreads);
  if (small_table)
    hipLaunchKernelGGL(CliqueRowsHashKernel<10>, grid, block, 0, stream, a);
  else
    hipLaunchKernelGGL(CliqueRowsHashKernel<13>, grid, block, 0, stream, a);
}

void LaunchCliqueDense(const CliqueArgs& a, int words, hipStream_t stream) {
  if (a.nverts == 0) return;
  const dim3 grid(Grid(a.nverts, 1)), block(kThreads);
  switch (words) {
    case 4: hipLaunchKernelGGL(CliqueDenseKernel<4>, grid, block, 0, stream, a); break;
    case 8: hipLaunchKernelGGL(CliqueDenseKernel<8>, grid, block, 0, stream, a); break;
    case 12: hipLaunchKernelGGL(CliqueDenseKernel<12>, grid, block, 0, stream, a); break;
    case 16: hipLaunchKernelGGL(CliqueDenseKernel<16>, grid, block, 0, stream, a); break;
  }
}

void LaunchCliqueCount(const CliqueArgs& a, uint32_t dmax, hipStream_t stream) {
  if (a.nitems == 0) return;
  const dim3 grid(Grid(a.nitems, kWaves)), block(kThreads);
  const uint64_t rows = Grid(a.nitems, 1);
  const dim3 longs(rows < 2048 ? rows : 2048);
  switch (a.k) {
    case 4: hipLaunchKernelGGL(CliqueCount4Kernel, grid, block, 0, stream, a); break;
    case 5:
      // (a row has fewer members than the largest d: no launch that finds none)
      hipLaunchKernelGGL(CliquePackKernel<5>, grid, block, 0, stream, a);
      if (dmax > kPackWave) hipLaunchKernelGGL((CliqueLongKernel<8, false>), longs, block, 0, stream, a);
      if (dmax > 256) hipLaunchKernelGGL((CliqueLongKernel<16, true>), longs, block, 0, stream, a);
      if (dmax > kPackLong) hipLaunchKernelGGL(CliqueUnpackedKernel<5>, grid, block, 0, stream, a);
      break;
    case 6:
      hipLaunchKernelGGL(CliquePackKernel<6>, grid, block, 0, stream, a);
      if (dmax > kPackWave) hipLaunchKernelGGL(CliqueUnpackedKernel<6>, grid, block, 0, stream, a);
      break;
  }
}

}  // namespace sme
