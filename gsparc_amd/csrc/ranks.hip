// Column ranks (ranks.hpp).  Y's free field usually takes far fewer distinct
// values than 2^ynf; its rank among them is what the accumulators work on:
// narrow, dense and in the same order, so Y stays sorted by (contract, rank).
#include "ranks.hpp"

#include <algorithm>

namespace sptc {

namespace {

// One byte per possible free key, set by plain stores: of a skewed mode's
// entries most meet in a few words, and a bitmap's atomics there (even behind a
// look at the word) took 250 to 600 us where the stores take a tenth.
__global__ __launch_bounds__(kBlock) void k_rank_mark(const uint64_t* __restrict__ ykeys,
                                                      uint64_t ny, uint64_t fmask,
                                                      uint8_t* __restrict__ seen) {
  uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (; i < ny; i += stride) seen[ykeys[i] & fmask] = 1;
}

// Per 32 free keys: their bits and the rank of the first; the table of the keys.
struct RankWordOp {
  const uint4* seen;  // two per 32 keys
  uint32_t *words, *pre;
  uint64_t* ytab;
  uint32_t* ytab32;
  struct Aux {
    uint32_t bits;
  };
  // four bytes of 0 or 1 to four bits
  __device__ static uint32_t nibble(uint32_t b) { return (b * 0x10204080u) >> 28; }
  __device__ U2 value(uint64_t i, Aux& x) const {
    const uint4 a = seen[2 * i], b = seen[2 * i + 1];
    x.bits = nibble(a.x) | nibble(a.y) << 4 | nibble(a.z) << 8 | nibble(a.w) << 12 |
             nibble(b.x) << 16 | nibble(b.y) << 20 | nibble(b.z) << 24 | nibble(b.w) << 28;
    return mk2((uint64_t)__popc(x.bits), 0);
  }
  __device__ void emit(uint64_t i, U2 ex, U2, const Aux& x) const {
    words[i] = x.bits;
    pre[i] = (uint32_t)ex.a;
    uint64_t o = ex.a;
    for (uint32_t b = x.bits; b; b &= b - 1, ++o) {
      const uint64_t f = i * 32 + (uint64_t)__builtin_ctz(b);
      ytab[o] = f;
      if (ytab32) ytab32[o] = (uint32_t)f;
    }
  }
};

__global__ __launch_bounds__(kBlock) void k_rank_read(const uint64_t* __restrict__ ykeys,
                                                      uint64_t ny, uint64_t fmask,
                                                      const uint32_t* __restrict__ words,
                                                      const uint32_t* __restrict__ pre,
                                                      uint32_t* __restrict__ ycol,
                                                      uint32_t* __restrict__ yfree32) {
  uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (; i < ny; i += stride) {
    const uint64_t f = ykeys[i] & fmask;
    const uint32_t below = words[f >> 5] & ((1u << (f & 31)) - 1);
    ycol[i] = pre[f >> 5] + (uint32_t)__popc(below);
    if (yfree32) yfree32[i] = (uint32_t)f;
  }
}

struct RankUniqueOp {
  const uint64_t* keys;  // sorted
  uint64_t* ytab;
  uint32_t* ytab32;
  __device__ U2 value(uint64_t i) const { return mk2(i == 0 || keys[i] != keys[i - 1], 0); }
  __device__ void emit(uint64_t i, U2 ex, U2 v) const {
    if (!v.a) return;
    ytab[ex.a] = keys[i];
    if (ytab32) ytab32[ex.a] = (uint32_t)keys[i];
  }
};

__global__ __launch_bounds__(kBlock) void k_rank_search(const uint64_t* __restrict__ ykeys,
                                                        uint64_t ny, uint64_t fmask,
                                                        const uint64_t* __restrict__ ytab,
                                                        const U2* __restrict__ distinct,
                                                        uint32_t* __restrict__ ycol,
                                                        uint32_t* __restrict__ yfree32) {
  const uint64_t U = distinct->a;
  uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (; i < ny; i += stride) {
    const uint64_t f = ykeys[i] & fmask;
    uint64_t lo = 0, hi = U;
    while (lo < hi) {
      const uint64_t mid = (lo + hi) >> 1;
      if (ytab[mid] < f) lo = mid + 1; else hi = mid;
    }
    ycol[i] = (uint32_t)lo;
    if (yfree32) yfree32[i] = (uint32_t)f;
  }
}

uint32_t grid_of(uint64_t n) { return (uint32_t)std::min<uint64_t>(ceil_div(n, kBlock), 4096); }

}  // namespace

// The map costs a clear and two reads of 2^ynf bytes besides one store and one
// look-up per entry; the sort moves every key ynf / 8 times in passes of three
// launches.  Where the line lies: 24 bits and 1e6 entries 0.09 ms against 0.25,
// 25 bits and 6.4e5 entries 0.09 against 0.22; 28 bits and 1e6 entries would
// take about the sort's time and ten times its memory.
bool rank_by_map(uint64_t ny, int ynf) {
  return ynf <= 32 && rank_map_bytes(ynf) <= 64 * ny + (1ull << 22);
}

void run_rank_map(const uint64_t* ykeys, uint64_t ny, int ynf, const RankOut& o, uint8_t* map,
                  U2* tmp, U2* host, hipStream_t s) {
  const uint64_t nw = rank_words(ynf), fmask = low_mask(ynf);
  uint32_t* const words = reinterpret_cast<uint32_t*>(map + 32 * nw);
  uint32_t* const pre = words + nw;
  fill_u64(reinterpret_cast<uint64_t*>(map), 0, 4 * nw, s);
  hipLaunchKernelGGL(k_rank_mark, dim3(grid_of(ny)), dim3(kBlock), 0, s, ykeys, ny, fmask, map);
  run_scan(RankWordOp{reinterpret_cast<const uint4*>(map), words, pre, o.ytab, o.ytab32}, nw, tmp,
           s, true, host);
  hipLaunchKernelGGL(k_rank_read, dim3(grid_of(ny)), dim3(kBlock), 0, s, ykeys, ny, fmask, words,
                     pre, o.ycol, o.yfree32);
}

void run_rank_sorted(const uint64_t* sorted, const uint64_t* ykeys, uint64_t ny, int ynf,
                     const RankOut& o, U2* tmp, U2* host, hipStream_t s) {
  run_scan(RankUniqueOp{sorted, o.ytab, o.ytab32}, ny, tmp, s, true, host);
  hipLaunchKernelGGL(k_rank_search, dim3(grid_of(ny)), dim3(kBlock), 0, s, ykeys, ny,
                     low_mask(ynf), o.ytab, tmp + scan_tmp_count(ny), o.ycol, o.yfree32);
}

}  // namespace sptc
