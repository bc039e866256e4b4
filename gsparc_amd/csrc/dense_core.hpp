// Dense per-row accumulation core shared by the single-contraction and the
// batched dense kernels.
//
// One workgroup owns one X row.  A row of kOwnerRun products per owner or more
// is taken a wave per owner (dense_owner_runs).  The products of others -- the
// concatenation, in active-nonzero order j, of each nonzero's matched Y segment
// -- are taken in rounds of kBlock * G products: every thread loads its G
// products of the round at once (strided, so loads coalesce and G of them are in
// flight per thread) and finds their owners j by binary search over the round's
// act_prefix entries staged in LDS.  Either way each is added to its column's
// FP64 slot by an LDS atomic.  FP64 sums do not depend on the order of the adds
// (SumF64 in common.hpp says when exactly), so rows need no barrier between
// owners and the outputs equal the ESC path's.  Only the slots below the number of
// columns are cleared and read back, a wave per 64 of them, and stored by adjacent
// lanes.  (Two operands of 3001 nonzeros over some hundred rows: 35 us a thread
// per run of slots and a search per product, 20 so.)
#pragma once
#include "kernels.hpp"

namespace sptc {

constexpr int kDenseG = 4;                               // products per thread per round
constexpr uint32_t kDenseRound = kBlock * kDenseG;       // products per round

template <int EB>
struct DenseSmem {
  static constexpr int E = 1 << EB;
  static constexpr int W = E / 32;
  alignas(8) uint32_t bm[W];
  uint64_t pref[kDenseRound + 1];
  uint32_t red[kBlock / kWave];
  uint64_t jl;  // owner of the round's last product
};

// Stages the round's owner prefixes: owners of products [pb, pl] are
// entries [ja, ja + m) of [j0, j1).  Returns ja through *ja.
template <typename SM>
__device__ __forceinline__ uint32_t dense_stage_owners(const uint64_t* __restrict__ act_prefix,
                                                       uint64_t j0, uint64_t j1, uint64_t pb,
                                                       uint64_t pl, SM& sm, uint64_t* s_ja,
                                                       uint64_t* ja) {
  __syncthreads();
  // last j with act_prefix[j] <= pb (wave 0), <= pl (wave 1)
  if (threadIdx.x < 2 * kWave) {
    const uint64_t j = wave_last_le(act_prefix, j0, j1, threadIdx.x < kWave ? pb : pl);
    if (threadIdx.x == 0) *s_ja = j;
    if (threadIdx.x == kWave) sm.jl = j;
  }
  __syncthreads();
  *ja = *s_ja;
  uint64_t* pref = sm.pref;
  const uint64_t need = sm.jl - *ja + 1;
  const uint32_t m = (uint32_t)(need < kDenseRound ? need : kDenseRound);
  for (uint32_t k = threadIdx.x; k <= m; k += kBlock) pref[k] = act_prefix[*ja + k];
  __syncthreads();
  return m;
}

// Owner (index into the staged run) of product p: last k with pref[k] <= p.
__device__ __forceinline__ uint32_t dense_owner(const uint64_t* pref, uint32_t m, uint64_t p) {
  uint32_t lo = 0, hi = m;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (pref[mid] <= p) lo = mid + 1; else hi = mid;
  }
  return lo - 1;
}

// The row's products, a wave per owner: this wave takes owners w, w + nw, ...
// of [j0, j1), 256 products of a segment in flight, and calls f(rank, product) for
// each (VAL false: no product).  No searches and no barriers, but lanes idle past
// a segment's end.
template <bool VAL, class F>
__device__ __forceinline__ void dense_owner_runs(const DenseArgs& a, uint64_t j0, uint64_t j1,
                                                 uint32_t w, uint32_t nw, F&& f) {
  constexpr int G = 4;
  const uint32_t lane = lane_id();
  for (uint64_t jb = j0; jb < j1; jb += kWave) {  // 64 owners' places at once
    const uint64_t j = jb + lane < j1 ? jb + lane : jb;
    const uint64_t oy = a.act_ypos[j];
    const uint32_t on = (uint32_t)(a.act_prefix[j + 1] - a.act_prefix[j]);
    const float ox = VAL ? a.act_xval[j] : 0.f;
    const uint32_t no = (uint32_t)(j1 - jb < kWave ? j1 - jb : kWave);
    for (uint32_t k = w; k < no; k += nw) {
      const uint64_t y0 = __shfl(oy, k, kWave);
      const uint32_t len = __shfl(on, k, kWave);
      const float x = __shfl(ox, k, kWave);
      for (uint32_t b = 0; b < len; b += kWave * G) {
        uint32_t rk[G];
        float v[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const uint32_t p = b + (uint32_t)g * kWave + lane;
          const uint64_t y = y0 + (p < len ? p : len - 1);
          rk[g] = a.ycol[y];
          v[g] = VAL ? a.yvals[y] : 0.f;
        }
#pragma unroll
        for (int g = 0; g < G; ++g)
          if (b + (uint32_t)g * kWave + lane < len) f(rk[g], x * v[g]);
      }
    }
  }
}
// Products per owner from which a row is taken that way by a whole workgroup.
constexpr uint64_t kOwnerRun = 32;

// Symbolic pass: bitmap of the row's touched column ranks; returns the count
// (valid in thread 0).
template <int EB>
__device__ __forceinline__ uint32_t dense_row_count(const DenseArgs& a, uint64_t j0, uint64_t j1,
                                                    DenseSmem<EB>& sm, uint64_t* s_ja) {
  for (int i = threadIdx.x; i < DenseSmem<EB>::W; i += kBlock) sm.bm[i] = 0;
  const uint64_t p0 = j0 < j1 ? a.act_prefix[j0] : 0;
  const uint64_t p1 = j0 < j1 ? a.act_prefix[j1] : 0;
  const bool runs = p1 - p0 >= kOwnerRun * (j1 - j0);
  if (runs) {
    __syncthreads();
    dense_owner_runs<false>(a, j0, j1, threadIdx.x / kWave, kBlock / kWave, [&](uint32_t rk, float) {
      atomicOr(&sm.bm[rk >> 5], 1u << (rk & 31));
    });
  }
  for (uint64_t pb = runs ? p1 : p0; pb < p1; pb += kDenseRound) {
    uint64_t ja;
    const uint64_t pl = (pb + kDenseRound < p1 ? pb + kDenseRound : p1) - 1;
    const uint32_t m = dense_stage_owners(a.act_prefix, j0, j1, pb, pl, sm, s_ja, &ja);
#pragma unroll
    for (int g = 0; g < kDenseG; ++g) {
      const uint64_t p = pb + (uint64_t)g * kBlock + threadIdx.x;
      if (p < p1) {
        const uint32_t k = dense_owner(sm.pref, m, p);
        const uint64_t y = a.act_ypos[ja + k] + (p - sm.pref[k]);
        const uint32_t rank = a.ycol[y];
        atomicOr(&sm.bm[rank >> 5], 1u << (rank & 31));
      }
    }
  }
  __syncthreads();
  uint32_t cnt = 0;
  for (int i = threadIdx.x; i < DenseSmem<EB>::W; i += kBlock) cnt += __popc(sm.bm[i]);
  for (int off = kWave / 2; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, kWave);
  if (lane_id() == 0) sm.red[threadIdx.x / kWave] = cnt;
  __syncthreads();
  uint32_t t = 0;
  if (threadIdx.x == 0)
    for (int w = 0; w < kBlock / kWave; ++w) t += sm.red[w];
  return t;
}

// Numeric pass, then the touched slots in rank order to out_* at obase (row
// id `row`, column ytab[rank] or rank).  `acc` holds E doubles of LDS, of which
// the first `cols` are used: ranks are below it.
template <int EB>
__device__ __forceinline__ void dense_row_numeric(const DenseArgs& a, uint64_t j0, uint64_t j1,
                                                  const uint64_t* ytab, uint32_t cols,
                                                  uint32_t row, uint64_t obase, double* acc,
                                                  DenseSmem<EB>& sm, uint64_t* s_ja) {
  static_assert(DenseSmem<EB>::E >= 64 && DenseSmem<EB>::E <= 64 * kBlock, "dense row width");
  for (uint32_t i = threadIdx.x; i < cols; i += kBlock) acc[i] = 0.0;
  for (int i = threadIdx.x; i < DenseSmem<EB>::W; i += kBlock) sm.bm[i] = 0;
  const uint64_t p0 = j0 < j1 ? a.act_prefix[j0] : 0;
  const uint64_t p1 = j0 < j1 ? a.act_prefix[j1] : 0;
  double vsum = 0.0;
  const bool runs = p1 - p0 >= kOwnerRun * (j1 - j0);
  if (runs) {
    __syncthreads();
    dense_owner_runs<true>(a, j0, j1, threadIdx.x / kWave, kBlock / kWave, [&](uint32_t rk, float z) {
      vsum += (double)z;
      atomicAdd(&acc[rk], (double)z);
      atomicOr(&sm.bm[rk >> 5], 1u << (rk & 31));
    });
  }
  for (uint64_t pb = runs ? p1 : p0; pb < p1; pb += kDenseRound) {
    uint64_t ja;
    const uint64_t pl = (pb + kDenseRound < p1 ? pb + kDenseRound : p1) - 1;
    const uint32_t m = dense_stage_owners(a.act_prefix, j0, j1, pb, pl, sm, s_ja, &ja);
    uint32_t rank[kDenseG];
    float val[kDenseG];
#pragma unroll
    for (int g = 0; g < kDenseG; ++g) {
      const uint64_t p = pb + (uint64_t)g * kBlock + threadIdx.x;
      rank[g] = 0;
      val[g] = 0.f;
      if (p < p1) {
        const uint32_t k = dense_owner(sm.pref, m, p);
        const uint64_t y = a.act_ypos[ja + k] + (p - sm.pref[k]);
        rank[g] = a.ycol[y];
        val[g] = a.act_xval[ja + k] * a.yvals[y];
      }
    }
#pragma unroll
    for (int g = 0; g < kDenseG; ++g) {
      if (pb + (uint64_t)g * kBlock + threadIdx.x < p1) {
        vsum += (double)val[g];
        atomicAdd(&acc[rank[g]], (double)val[g]);
        atomicOr(&sm.bm[rank[g] >> 5], 1u << (rank[g] & 31));
      }
    }
    // (the next round's staging starts with a barrier)
  }
  __syncthreads();
  // Compaction in column order, a wave per word of 64 slots: the outputs before
  // each word, then every lane stores its slot's (adjacent lanes, adjacent outputs).
  const uint32_t words = (cols + 63) / 64;  // at most E / 64 <= kBlock
  const uint64_t* const bm64 = reinterpret_cast<const uint64_t*>(sm.bm);
  uint32_t tot;
  const uint32_t mine = threadIdx.x < words ? (uint32_t)__popcll(bm64[threadIdx.x]) : 0u;
  const uint32_t ex = block_excl_scan<uint32_t>(mine, sm.red, &tot);
  uint32_t* const wpre = reinterpret_cast<uint32_t*>(sm.pref);
  if (threadIdx.x < words) wpre[threadIdx.x] = ex;
  __syncthreads();
  for (uint32_t w = threadIdx.x / kWave; w < words; w += kBlock / kWave) {
    const uint64_t b = bm64[w];
    if (b >> lane_id() & 1) {
      const uint32_t rk = w * 64 + lane_id();
      const uint64_t o = obase + wpre[w] + popc_below(b);
      a.out_row[o] = row;
      a.out_col[o] = ytab ? ytab[rk] : rk;
      a.out_val[o] = (float)acc[rk];
    }
  }
  if (!a.vsum) return;  // batches sum their outputs instead
  for (int off = kWave / 2; off > 0; off >>= 1) vsum += __shfl_xor(vsum, off, kWave);
  if (lane_id() == 0 && vsum != 0.0) slot_add(a.vsum, vsum);
}

}  // namespace sptc
