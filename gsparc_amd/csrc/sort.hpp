// Radix sort workspace and host launchers (see sort.hip).
#pragma once
#include "common.hpp"
#include "device.hpp"
#include "ktimer.hpp"
#include "scan.hpp"

namespace sptc {

constexpr int kMaxPasses = 16;

struct LinArgs {
  const void* idx[SPTC_MAX_ORDER];
  int shift[SPTC_MAX_ORDER];
  int width[SPTC_MAX_ORDER];
  int order;
};

struct SortWorkspace {
  int rb = 8;                   // radix bits per pass
  DevBuf<uint64_t> alt_keys;
  DevBuf<float> alt_vals;
  // onesweep: [kMaxPasses][R] digit counts, kSweepHead words of tile counters,
  // [tiles][R] look-back words -- one fill clears them
  DevBuf<uint64_t> sweep;
  static constexpr uint64_t kSweepHead = 32;
  DevBuf<uint32_t> rts_cnt;     // [R][tiles] per-tile digit counts
  DevBuf<uint32_t> rts_off;     // [R][tiles] their exclusive scan
  DevBuf<U2> rts_tmp;           // scan scratch
  uint32_t epoch = 0;
  // set by a failed look-back: pinned host memory or a device word, which the
  // workspace's user clears, and reads after a wait
  uint32_t* err_word = nullptr;

  // Grows the workspace to hold `n` keys (and values) at `rb` radix bits.
  void ensure(uint64_t n, int rb, hipStream_t s, bool vals = true);
  // Gives everything back (the stream must have been waited for).
  void release() {
    alt_keys.release();
    alt_vals.release();
    sweep.release();
    rts_cnt.release();
    rts_off.release();
    rts_tmp.release();
  }
  // Clears histograms, counters and look-back words before a sort of n keys
  // (onesweep only).
  void prepare(uint64_t n, hipStream_t s);
  uint64_t* hist() const { return sweep.get(); }
  uint32_t* counters() const {
    return reinterpret_cast<uint32_t*>(sweep.get() + ((uint64_t)kMaxPasses << rb));
  }
  uint64_t* status() const { return sweep.get() + ((uint64_t)kMaxPasses << rb) + kSweepHead; }
  uint32_t* err() const { return err_word; }
  static uint64_t bytes_per_key(int rb);
};

int radix_passes(int nbits, int rb);
uint64_t sort_tile_items(int rb);
bool radix_bits_supported(int rb);
// True when n keys are sorted by one-launch passes with look-back, which need
// the digit histograms of all passes up front (ws.prepare, then a producer or
// histogram()); reduce-then-scan passes count per tile themselves.
// The line, look-back against reduce-then-scan: with 8- and 9-bit digits 0.26e6 pairs
// of 40 bits 116 us against 167, 1e6 165 against 195, 2e6 212 against 206 (24 bits
// 154 / 139, 64 bits 282 / 293), 77e6 4.5 ms against 3.8: past a few tiles per CU the
// status words cost more than the launches they save.  Wider digits have more of
// them per key, so their line lies lower: 10 bits at 0.26e6 pairs 140 us against
// 144, 0.4e6 160 / 149, 2e6 330 / 208; 11 bits at 0.1e6 146 / 148, 0.2e6 173 / 152,
// 2e6 472 / 267.
constexpr uint64_t kOnesweepMax = 1ull << 21;
constexpr uint64_t onesweep_max(int rb) {
  return rb <= 9 ? kOnesweepMax : rb == 10 ? 1ull << 18 : 1ull << 16;
}
bool sort_onesweep(uint64_t n, int rb);
// Linearizes and sorts up to one tile of nonzeros in one launch; false when there
// are more.
bool sort_linearize_small(const LinArgs& a, int idx_bytes, const float* val, uint64_t n,
                          uint64_t* keys, float* vals, hipStream_t s);
// Digit width for a sort over nbits key bits (fewest passes, digits <= 10).
int choose_radix_bits(int nbits);
void histogram(const SortWorkspace& ws, const uint64_t* keys, uint64_t n,
               int passes, hipStream_t s, int lo = 0);
// Sorts (keys, vals), stably, on bits [lo, nbits), ws.hist() holding the histograms
// of all passes for sizes that sort_onesweep.  vals NULL: the keys alone are moved;
// vsrc: the first pass reads the values there.  Returns true when the sorted data
// ended in (ws.alt_keys, ws.alt_vals) (odd pass count).
// kt (optional) times every pass under kernel class `cls`.
bool sort_after_histogram(SortWorkspace& ws, uint64_t* keys, float* vals,
                          uint64_t n, int nbits, hipStream_t s, KTimer* kt = nullptr,
                          int cls = 0, const float* vsrc = nullptr, int lo = 0);

// Device-side histogram accumulation for producers: call once per key with
// an LDS array of passes*R uint32 cleared by the block, then flush.
template <int RB>
__device__ __forceinline__ void hist_add(uint32_t* sh, uint64_t key, int passes) {
  constexpr uint32_t R = 1u << RB;
  for (int p = 0; p < passes; ++p)
    atomicAdd(&sh[p * R + ((uint32_t)(key >> (p * RB)) & (R - 1))], 1u);
}
// Wave-aggregated variant: when every valid lane of the wave has the same
// digit (typical for the high, row-index digits of product keys) one lane
// adds the whole count; otherwise each lane adds one.  All lanes of the wave
// must call it together.
template <int RB>
__device__ __forceinline__ void hist_add_wave(uint32_t* sh, uint64_t key, bool valid,
                                             int passes) {
  constexpr uint32_t R = 1u << RB;
  const uint64_t vmask = __ballot(valid);
  if (!vmask) return;
  const int first = __builtin_ctzll(vmask);
  for (int p = 0; p < passes; ++p) {
    const uint32_t d = (uint32_t)(key >> (p * RB)) & (R - 1);
    const uint32_t d0 = __shfl(d, first, 64);
    const uint64_t same = __ballot(valid && d == d0);
    if (same == vmask) {
      if ((int)__lane_id() == first) atomicAdd(&sh[p * R + d0], (uint32_t)__popcll(vmask));
    } else if (valid) {
      atomicAdd(&sh[p * R + d], 1u);
    }
  }
}

template <int RB>
__device__ __forceinline__ void hist_flush(const uint32_t* sh, uint64_t* hist,
                                           int passes) {
  constexpr int R = 1 << RB;
  for (int i = threadIdx.x; i < passes * R; i += blockDim.x)
    if (sh[i]) atomicAdd((unsigned long long*)&hist[i], (unsigned long long)sh[i]);
}

}  // namespace sptc
