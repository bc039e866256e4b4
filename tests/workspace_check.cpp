// Host-side check of the sort workspace (test_sort_workspace.py builds and runs
// it without a GPU): the library's device pool is replaced by one that hands out
// addresses, and after every sequence of reservations the buffers that a
// reduce-then-scan sort of n keys uses must hold what its launches touch.
#include <cstdio>

#include "segsort.hpp"
#include "sort.hpp"

namespace sptc {
// (taken instead of the library's own: its symbols can be interposed)
void* DevicePool::alloc(size_t bytes) {
  static uintptr_t next = 1 << 20;
  next += bytes + 256;
  return reinterpret_cast<void*>(next);
}
void DevicePool::free(void*) {}
}  // namespace sptc

using namespace sptc;

static int bad = 0;

static void check(const char* what, const SortWorkspace& ws, uint64_t n, int rb) {
  const uint64_t m = ceil_div(n, sort_tile_items(rb)) << rb, nt = scan_tmp_count(m) + 1;
  const bool ok = ws.rb == rb && ws.alt_keys.size() >= n && ws.rts_cnt.size() >= m &&
                  ws.rts_off.size() >= m && ws.rts_tmp.size() >= nt;
  printf("%s: n %llu rb %d matrix %llu of %llu, scan %llu of %llu: %s\n", what,
         (unsigned long long)n, rb, (unsigned long long)ws.rts_cnt.size(), (unsigned long long)m,
         (unsigned long long)ws.rts_tmp.size(), (unsigned long long)nt, ok ? "ok" : "BAD");
  bad += !ok;
}

int main() {
  for (int rb : {8, 9, 10, 11}) {
    for (uint64_t n : {kOnesweepMax + 1, 3 * kOnesweepMax, 40 * kOnesweepMax}) {
      const uint64_t tiles = ceil_div(n, sort_tile_items(rb));
      SortWorkspace fresh;
      fresh.ensure(n, rb, nullptr);
      check("fresh", fresh, n, rb);
      for (uint64_t t : {tiles / 2, tiles, 16 * tiles}) {  // segmented sort first
        SortWorkspace ws;
        segmented_sort_reserve(ws, t, nullptr, rb);
        ws.ensure(n, rb, nullptr);
        check("segmented sort before", ws, n, rb);
      }
      SortWorkspace ws;  // operand sorts, a segmented sort, a larger sort
      ws.ensure(1000, 8, nullptr);
      ws.ensure(kOnesweepMax + 1, 8, nullptr);
      segmented_sort_reserve(ws, 4 * tiles, nullptr, rb);
      ws.ensure(n, rb, nullptr);
      check("in between", ws, n, rb);
    }
  }
  return bad != 0;
}
