// A count whose kernel writes its sums to pinned host memory: what the page
// holds before the call may not pass for this call's result.  The linker sends
// hipHostMalloc and the kernel's launcher here first (--wrap).
//   publish_test stale    the page comes filled with 1, 2, 3, ...
//   publish_test dropped  some launches do not happen
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>

#include "../../include/sme.h"
#include "kernels.h"

namespace {
unsigned long long g_fill = 0;      // value of every word of a new pinned page
bool g_stale = false;               // a launch found its call's number already published
bool g_drop = false;                // launches do not happen
}  // namespace

hipError_t RealHostMalloc(void** p, size_t n, unsigned flags) asm("__real__Z13hipHostMallocPPvmj");
hipError_t WrapHostMalloc(void** p, size_t n, unsigned flags) asm("__wrap__Z13hipHostMallocPPvmj");
hipError_t WrapHostMalloc(void** p, size_t n, unsigned flags) {
  const hipError_t e = RealHostMalloc(p, n, flags);
  for (size_t k = 0; e == hipSuccess && k < n / 8; ++k) static_cast<unsigned long long*>(*p)[k] = g_fill;
  return e;
}

void RealSmall(const sme::CliqueArgs& a, hipStream_t s) asm("__real__ZN3sme17LaunchCliqueSmallERKNS_10CliqueArgsEP9EmuStream");
void WrapSmall(const sme::CliqueArgs& a, hipStream_t s) asm("__wrap__ZN3sme17LaunchCliqueSmallERKNS_10CliqueArgsEP9EmuStream");
void WrapSmall(const sme::CliqueArgs& a, hipStream_t s) {
  if (a.publish && a.publish[sme::kCliqueMaxK + 1] == a.call) g_stale = true;
  if (!g_drop) RealSmall(a, s);
}

namespace {

// Triangles of a cycle of n with its chords (k, k + 2): n for n > 6.
int Count(sme_ctx* ctx, uint64_t n, uint64_t* count) {
  uint64_t rp[64] = {0};
  uint32_t cols[256];
  uint64_t at = 0;
  for (uint64_t v = 0; v < n; ++v) {
    for (uint64_t w = 0; w < n; ++w) {
      const uint64_t gap = (w + n - v) % n;
      if (gap == 1 || gap == 2 || gap == n - 1 || gap == n - 2) cols[at++] = static_cast<uint32_t>(w);
    }
    rp[v + 1] = at;
  }
  sme_graph* g = nullptr;
  sme_plan* plan = nullptr;
  int rc = sme_graph_upload(ctx, rp, cols, n, at, &g);
  if (rc == SME_OK) rc = sme_plan_create(SME_ALGO_LIGHT, 0, 3, 1, &plan);
  if (rc == SME_OK) rc = sme_count(ctx, g, plan, 0, static_cast<uint32_t>(n), count, nullptr, nullptr);
  sme_plan_destroy(plan);
  sme_graph_destroy(g);
  return rc;
}

int Stale() {
  for (unsigned long long fill = 1; fill <= 8; ++fill) {
    g_fill = fill;
    sme_ctx* ctx = nullptr;
    if (sme_open(0, 1 << 20, &ctx) != SME_OK) return 2;
    for (uint64_t n = 7; n < 15; ++n) {
      uint64_t got = 0;
      if (Count(ctx, n, &got) != SME_OK || got != n) {
        std::fprintf(stderr, "page of %llu, n %llu: count %llu\n", fill, static_cast<unsigned long long>(n),
                     static_cast<unsigned long long>(got));
        return 1;
      }
      if (g_stale) {
        std::fprintf(stderr, "page of %llu: call %llu is published before its launch\n", fill,
                     static_cast<unsigned long long>(n - 6));
        return 1;
      }
    }
    sme_close(ctx);
  }
  return 0;
}

// A call without its kernel is an error, and the calls after it are right.
int Dropped() {
  sme_ctx* ctx = nullptr;
  if (sme_open(0, 1 << 20, &ctx) != SME_OK) return 2;
  for (uint64_t n = 7; n < 19; ++n) {
    g_drop = n % 4 < 2;
    uint64_t got = 0;
    const int rc = Count(ctx, n, &got);
    if (rc != (g_drop ? SME_ERR_HIP : SME_OK) || (!g_drop && got != n)) {
      std::fprintf(stderr, "n %llu, launch %d: rc %d count %llu\n", static_cast<unsigned long long>(n), !g_drop, rc,
                   static_cast<unsigned long long>(got));
      return 1;
    }
  }
  sme_close(ctx);
  return 0;
}

}  // namespace

int main(int argc, char** argv) {
  const char* what = argc > 1 ? argv[1] : "";
  if (!std::strcmp(what, "stale")) return Stale();
  if (!std::strcmp(what, "dropped")) return Dropped();
  std::fprintf(stderr, "usage: %s stale|dropped\n", argv[0]);
  return 2;
}
