// Host-side check of the row accumulator's plan over several chunks
// (test_sort_workspace.py builds and runs it without a GPU).  Launches, waits and the
// device pool are replaced by ones that only keep count: no block may go back to
// the pool, where another thread could take it for its own stream, while launches
// that may use it have not been waited for.
#include <cstdio>
#include <cstring>

#include "rowacc.hpp"

using namespace sptc;

static int in_flight = 0, bad = 0, launches = 0, frees = 0;
static U2 host[3];
static U2 kinds, counts;  // what the two scans that a count waits for report
static int waits = 0;

extern "C" hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
  ++launches;
  in_flight = 1;
  return hipSuccess;
}
extern "C" hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) {
  return hipSuccess;
}
extern "C" hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) {
  return hipSuccess;
}
extern "C" hipError_t hipStreamSynchronize(hipStream_t) {
  in_flight = 0;
  ++waits;
  return hipSuccess;
}

namespace sptc {
void* DevicePool::alloc(size_t bytes) {
  static uintptr_t next = 1 << 20;
  next += bytes + 256;
  return reinterpret_cast<void*>(next);
}
void DevicePool::free(void*) {
  ++frees;
  bad += in_flight;
}
}  // namespace sptc

int main() {
  KTimer kt;
  RowAccPlan p;
  RowAccArgs a{};
  a.K = 100000;
  a.short_max = 781;
  a.ny = 1000;
  // chunks that grow, shrink and grow: rows, short and long ones, products
  const uint64_t chunks[][3] = {{1000, 200, 50}, {5000, 3000, 10}, {10, 5, 5}, {9000, 100, 4000}};
  for (const auto& c : chunks) {
    const uint64_t rows = c[0], nshort = c[1], nlong = c[2];
    const uint64_t sp = nshort * 500, n = sp + nlong * 5000 + (rows - nshort - nlong) * 100;
    a.rows = rows;
    kinds = mk2(sp << 32 | rows, nshort << 32 | nlong);
    counts = mk2(n, (rows - nlong) << 32 | (n - nlong * 5000));
    // (the scans would write these; rowacc_count clears host[1].a and waits
    // first for the kinds, then for the counts)
    host[0] = kinds;
    host[2] = mk2(2 * nlong, 0);
    if (!rowacc_count(a, n, 4 * rows, false, &p, host, nullptr, &kt)) return 2;
    rowacc_emit(a, p, n, nullptr, nullptr, nullptr, nullptr, &kt);
    printf("chunk of %llu rows: launches %d waits %d blocks back %d, %d of them too early\n",
           (unsigned long long)rows, launches, waits, frees, bad);
  }
  hipStreamSynchronize(nullptr);
  return bad != 0 || !frees || launches < 20;
}
