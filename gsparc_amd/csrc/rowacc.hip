// Row accumulator: ESC's outputs without ESC's product arrays.
//
// The product sort writes every product to HBM, sorts it there and reads it
// back: about 60 bytes a product.  Its products are mostly not in disorder: a
// row's products are its owners' Y segments, each sorted by column, and a row
// has few owners with long segments (on the benchmark's shape half the
// products lie in rows of at most 22 owners with about 2000 products each).
// So the rows are taken by kind:
//   one owner   the row is that segment: its outputs are copied from Y with
//               the X value multiplied in (Y without duplicate coordinates);
//   short       up to short_max products of several owners: groups of rows
//               are expanded, sorted by (row, column) and summed in one
//               workgroup's LDS (k_ra_group);
//   long        the column ranks are cut into slabs of at most 2^16 so that a
//               (row, slab) item holds some thousand products.  k_ra_count
//               marks the item's columns in an LDS bitmap and counts them;
//               k_ra_sum marks them again, takes each column's output slot as
//               its rank in the bitmap, adds the products into FP64 slots by
//               LDS atomics, a window of slots at a time, and writes the
//               outputs in order.
// Per product: one column read twice and one value read once (from cache: Y
// is far smaller than the products), per output 16 bytes written once.
//
// Measured, 2482x2862x14036x17 with 1e6 nonzeros contracted with itself over
// its last two modes (1.67e9 products, 1.18e9 outputs): 11.3 ms of kernels
// against the product sort's 29.5, of which k_ra_sum 5.9 (1.36e9 products, 13.6
// GB written), k_ra_count 2.1, k_ra_near 1.5 (0.32e9 products, 7.7 GB moved),
// k_ra_split 0.8.  What bounds each is said beside it.
#include "rowacc.hpp"
#include "sort_core.hpp"

#include <algorithm>
#include <stdexcept>

namespace sptc {

namespace {

// live_src of a row: its first active X nonzero (one owner), its place in the
// groups' outputs (short), or long.
constexpr uint64_t kShortSrc = 1ull << 62;
constexpr uint64_t kLongSrc = 2ull << 62;

// Products an item should hold.  An item costs about 6 us of barriers and table
// making whatever it holds, more products than slots need several windows:
// k_ra_sum took 13.7 / 11.6 / 9.0 / 8.5 / 8.4 ms at 2048 / 3072 / 5120 / 7168 /
// 8192 (1e6 nonzeros as above, before its tables were packed).
constexpr uint64_t kItemProds = 7168;
// ... and products per owner of an item, below which the owner table costs
// more than the products.
constexpr uint64_t kItemRun = 4;
// An item is one workgroup's: it takes about 1.7 ns a product and 19 ns an owner
// (one row over few columns, 1e6 products of owners with 100 each 2.0 ms, with 1 each
// 21 ms), so an owner weighs as much as kOwnerWeight products.  A chunk with a heavy
// item -- long rows over few columns, or of very many owners -- goes to the product
// sort, which spreads a row over the chip.  Two lines:
//   weight above kHeavyWeight and a 64th of the chunk's products: the item alone
//     outlasts what the sort takes longer (0.13 ms and 0.03 ns a product of long
//     rows).  20 rows of owners with 100 products meet the sort at 1e5 products each
//     (385 us against 423 with 0.65e5, 504 / 453 with 1.3e5), with 5 at 0.25e5 (388 /
//     442 with 0.16e5, 744 / 559 with 0.65e5), with 1 below 0.16e5 (686 / 511); 250
//     rows of 1.3e5 products: 517 / 961;
//   products above kHeavyItem and a 1024th of the chunk's: among short rows, where
//     the sort is no slower, an item is all that differs (1.5e5 products in one row
//     beside 2e7 in short ones: 1185 us against 921).
constexpr uint64_t kHeavyItem = 1ull << 17;
constexpr uint64_t kHeavyWeight = 5ull << 14;
constexpr uint64_t kOwnerWeight = 11;

// Slab bounds follow the products: columns that occur often in Y hold most of
// a row's products (the first quarter of the benchmark's columns 61 %), so
// equal-width slabs would leave half the products in slabs of many windows.
// quant[i] is the column below which i / kQuant of the measure
// (3 columns / K + sampled share of Y) / 4 lies: a slab of 1 / S of it holds
// about 4 / S of the products at most, and K * 4/3 (1 / S + 1 / kQuant) columns.
constexpr uint32_t kQuant = 4096;

// Rows of at most kEvenProds products are cut into slabs of equal width, as
// few as hold kSlabCols columns each: whichever slab holds them, they fit its
// slots.
constexpr uint64_t kEvenProds = 12288;
__host__ __device__ __forceinline__ uint32_t even_slabs(uint32_t K) {
  return (K + kSlabCols - 1) >> kSlabBits;
}
// Least slabs of longer rows: no slab may exceed kSlabCols columns.
__host__ __device__ __forceinline__ uint32_t min_slabs(uint32_t K) {
  if (K <= kSlabCols) return 1;
  const double room = (double)(kSlabCols - 2) / (4.0 / 3.0 * K) - 1.0 / kQuant;
  return (uint32_t)(1.0 / room) + 1;
}
// Slabs of a long row of n products and `own` owners.
__device__ __forceinline__ uint32_t row_slabs(uint64_t n, uint64_t own, uint32_t K,
                                              uint32_t least) {
  if (n <= kEvenProds) return even_slabs(K);
  uint64_t s = n / kItemProds;
  const uint64_t t = n / (kItemRun * own);
  s = t < s ? t : s;
  const uint64_t hi = K >> 10;  // slabs of 1024 columns or so at least
  s = s > hi ? hi : s;
  return (uint32_t)(s > least ? s : least);
}

// quant[0 .. kQuant]: one workgroup takes kSamples Y entries, counts them by
// column in kQuant bins, adds the bins up and inverts the sum.
constexpr uint32_t kSamples = 1u << 14;
constexpr int kQuantNT = 1024;
__global__ __launch_bounds__(kQuantNT) void k_ra_quant(const uint32_t* __restrict__ ycol,
                                                       uint64_t ny, uint32_t K,
                                                       uint32_t* __restrict__ quant) {
  __shared__ uint32_t bin[kQuant];
  __shared__ uint32_t red[kQuantNT / kWave];
  constexpr uint32_t PER = kQuant / kQuantNT;
  const uint32_t tid = threadIdx.x;
  for (uint32_t i = tid; i < kQuant; i += kQuantNT) bin[i] = 0;
  __syncthreads();
  const uint32_t N = (uint32_t)(ny < kSamples ? ny : kSamples);
  for (uint32_t i = tid; i < N; i += kQuantNT) {
    const uint32_t c = ycol[(uint64_t)i * ny / N];
    atomicAdd(&bin[(uint32_t)((uint64_t)c * kQuant / K)], 1u);
  }
  __syncthreads();
  // a bin's measure: 3 kSamples for its columns, kQuant for each sample of N = kSamples
  uint32_t v[PER], sum = 0, all;
#pragma unroll
  for (uint32_t e = 0; e < PER; ++e) {
    v[e] = 3 * kSamples + (uint32_t)((uint64_t)bin[tid * PER + e] * kSamples / N) * kQuant;
    sum += v[e];
  }
  uint32_t ex = block_scan_u32<kQuantNT>(sum, red, &all);  // at most 2^28
#pragma unroll
  for (uint32_t e = 0; e < PER; ++e) {
    bin[tid * PER + e] = ex;
    ex += v[e];
  }
  __syncthreads();
  for (uint32_t i = tid; i <= kQuant; i += kQuantNT) {
    const uint32_t m = (uint32_t)((uint64_t)i * all / kQuant);
    uint32_t lo = 0, hi = kQuant;  // last bin starting at or before m
    while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) >> 1;
      if (bin[mid] <= m) lo = mid; else hi = mid;
    }
    const uint32_t w = (lo + 1 < kQuant ? bin[lo + 1] : all) - bin[lo];
    const double at = ((double)lo + (double)(m - bin[lo]) / w) * K / kQuant;
    quant[i] = i == kQuant ? K : (uint32_t)at;
  }
}

// ---- rows by kind ------------------------------------------------------------
// One scan over the chunk's rows: a = short products << 32 | live rows,
// b = short rows << 32 | long rows (a chunk holds fewer than 2^32 products).
// ACT: over its active X nonzeros instead, each row's first one standing for
// the row (rows without products are never met).
template <bool ACT>
struct RowKindOp {
  RowAccArgs a;
  uint32_t least;
  uint64_t heavy, weight;  // products, and weight, that one workgroup should not be given
  uint64_t* flag;  // pinned host memory
  uint32_t *live_row, *live_cnt;
  uint64_t* live_src;
  uint32_t *s_live, *s_prod, *l_live;
  __device__ U2 value(uint64_t i) const {
    uint64_t r = a.r0 + i;
    if (ACT) {
      r = a.act_row[a.a0 + i];
      if (i && a.act_row[a.a0 + i - 1] == r) return mk2(0, 0);
    }
    const uint64_t n = a.row_prod[r + 1] - a.row_prod[r];
    if (!n) return mk2(0, 0);
    const uint64_t own = a.row_act[r + 1] - a.row_act[r];
    if (own == 1 && !a.ydup) return mk2(1, 0);
    if (n <= a.short_max) return mk2(n << 32 | 1, 1ull << 32);
    return mk2(1, 1);
  }
  __device__ void emit(uint64_t i, U2 ex, U2 v) const {
    if (!v.a) return;
    const uint32_t k = (uint32_t)ex.a;
    const uint64_t r = ACT ? a.act_row[a.a0 + i] : a.r0 + i;
    live_row[k] = (uint32_t)(r - a.r0);
    if (v.b >> 32) {
      const uint32_t s = (uint32_t)(ex.b >> 32);
      s_live[s] = k;
      s_prod[s] = (uint32_t)(ex.a >> 32);
      live_cnt[k] = 0;  // k_ra_group's
    } else if (v.b) {
      l_live[(uint32_t)ex.b] = k;
      live_cnt[k] = 0;  // k_ra_count adds
      live_src[k] = kLongSrc;
      const uint64_t n = a.row_prod[r + 1] - a.row_prod[r];
      const uint64_t own = a.row_act[r + 1] - a.row_act[r];
      const uint64_t prods = n / row_slabs(n, own, a.K, least);
      if (prods > heavy || prods + kOwnerWeight * own > weight) *flag = 1;
    } else {
      live_cnt[k] = (uint32_t)(a.row_prod[r + 1] - a.row_prod[r]);
      live_src[k] = a.row_act[r];
    }
  }
};

// Long rows: before each, a = bitmap words (64 columns) << 32 | slabs,
// b = split entries.  (The words are only used while they fit 32 bits.)
struct SlabOp {
  RowAccArgs a;
  uint32_t least;
  const uint32_t *l_live, *live_row;
  uint64_t n;
  uint64_t *l_item, *l_split;
  uint32_t* l_word;
  __device__ U2 value(uint64_t i) const {
    const uint64_t r = a.r0 + live_row[l_live[i]];
    const uint64_t own = a.row_act[r + 1] - a.row_act[r];
    const uint64_t S = row_slabs(a.row_prod[r + 1] - a.row_prod[r], own, a.K, least);
    return mk2((S + a.K / 64 + 1) << 32 | S, own * (S + 1));
  }
  __device__ void emit(uint64_t i, U2 ex, U2 v) const {
    l_item[i] = ex.a & 0xFFFFFFFFull;
    l_word[i] = (uint32_t)(ex.a >> 32);
    l_split[i] = ex.b;
    if (i + 1 == n) l_item[n] = (ex.a + v.a) & 0xFFFFFFFFull;
  }
};

// Output offsets of the live rows; near rows (one owner or short) compacted.
// A long row keeps the near rows' outputs before it: its slabs' offsets are
// those plus the long rows' outputs before the slab (ItemOutOp).
struct alignas(8) Near {
  uint64_t off;  // first output
  uint64_t src;  // first Y entry (one owner), or kShortSrc | place in the groups' outputs
  uint32_t row;
  float x;       // the owner's X value
};
static_assert(sizeof(Near) == kNearBytes, "near row descriptor");

struct OutOp {
  RowAccArgs a;
  const uint32_t *live_cnt, *live_row;
  const uint64_t* live_src;
  uint32_t* l_near;
  uint32_t* near_pre;
  Near* near;
  __device__ U2 value(uint64_t k) const {
    const uint64_t c = live_cnt[k];
    return mk2(c, live_src[k] == kLongSrc ? 0 : 1ull << 32 | c);
  }
  __device__ void emit(uint64_t k, U2 ex, U2 v) const {
    if (!v.b) {
      l_near[k] = (uint32_t)ex.b;
      return;
    }
    const uint32_t m = (uint32_t)(ex.b >> 32);
    near_pre[m] = (uint32_t)ex.b;
    const uint64_t src = live_src[k];
    Near d;
    d.off = ex.a;
    d.src = src < kShortSrc ? a.act_ypos[src] : src;
    d.row = (uint32_t)(a.r0 + live_row[k]);
    d.x = src < kShortSrc ? a.act_xval[src] : 0.f;
    near[m] = d;
  }
};

// First index in [lo, hi) of v with v[i] >= c.
__device__ __forceinline__ uint32_t lower_bound32(const uint32_t* __restrict__ v, uint32_t lo,
                                                  uint32_t hi, uint32_t c) {
  while (lo < hi) {
    const uint32_t mid = lo + ((hi - lo) >> 1);
    if (v[mid] < c) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// An item: a slab of a long row.
struct alignas(16) Item {
  uint32_t j0, own;  // first owner, owners
  uint32_t split;    // its owners' first entries; the next slab's follow at + own
  uint32_t c0;       // first column
  uint32_t W;        // columns | unit width (log2) << 24 | last slab of its row << 31
  uint32_t live, row;
  uint32_t word;     // its bitmap words
  // columns of the slab, and words of 64 of them
  __device__ uint32_t cols() const { return W & 0xFFFFFFu; }
  __device__ uint32_t words() const { return (cols() + 63) >> 6; }
  __device__ int unit_bits() const { return (int)(W >> 24 & 0x7Fu); }
  __device__ bool last() const { return W >> 31; }
};
static_assert(sizeof(Item) == kItemBytes, "item descriptor");

struct ItemArgs {
  RowAccArgs a;
  const Item* item;
  const uint64_t* total;  // items
  uint32_t* split;
  uint64_t* words;        // the items' bitmaps (NULL: not kept)
};

// One thread per item: the long row that holds it, and what the item kernels
// need of it in one load.  Unit width: the lanes that share an owner's run of
// products (as many as the row has products per owner and slab, at most 16).
__global__ __launch_bounds__(kBlock) void k_ra_items(RowAccArgs a, const uint32_t* l_live,
                                                     const uint32_t* live_row,
                                                     const uint64_t* __restrict__ l_item,
                                                     const uint64_t* __restrict__ l_split,
                                                     const uint32_t* __restrict__ l_word,
                                                     const uint32_t* __restrict__ quant,
                                                     uint64_t nlong, Item* __restrict__ item) {
  const uint64_t total = l_item[nlong];
  for (uint64_t it = (uint64_t)blockIdx.x * kBlock + threadIdx.x; it < total;
       it += (uint64_t)gridDim.x * kBlock) {
    uint64_t lo = 0, hi = nlong;  // last row with l_item <= it
    while (hi - lo > 1) {
      const uint64_t mid = (lo + hi) >> 1;
      if (l_item[mid] <= it) lo = mid; else hi = mid;
    }
    const uint32_t q = (uint32_t)(it - l_item[lo]);
    const uint32_t S = (uint32_t)(l_item[lo + 1] - l_item[lo]);
    Item t;
    t.live = l_live[lo];
    const uint64_t r = a.r0 + live_row[t.live];
    t.row = (uint32_t)r;
    t.j0 = (uint32_t)a.row_act[r];
    t.own = (uint32_t)(a.row_act[r + 1] - a.row_act[r]);
    t.split = (uint32_t)(l_split[lo] + (uint64_t)q * t.own);
    const uint64_t n = a.row_prod[r + 1] - a.row_prod[r];
    auto bound = [&](uint32_t i) {
      return n <= kEvenProds ? (uint32_t)((uint64_t)i * a.K / S)
                             : quant[(uint64_t)i * kQuant / S];
    };
    t.c0 = bound(q);
    const uint32_t W = bound(q + 1) - t.c0;
    const uint64_t run = n / ((uint64_t)t.own * S);
    const uint32_t ub = run >= 12 ? 4 : run >= 6 ? 3 : run >= 3 ? 2 : 1;
    t.W = W | ub << 24 | (q + 1 == S ? 1u << 31 : 0u);
    t.word = l_word[lo] + t.c0 / 64 + q;  // (a slab's words never reach the next one's)
    item[it] = t;
  }
}

// Outputs of a slab start after the near outputs before its row and the
// long rows' outputs before it.
struct ItemOutOp {
  const uint32_t* item_cnt;
  const Item* item;
  const uint32_t* l_near;
  uint64_t* item_off;
  __device__ U2 value(uint64_t i) const { return mk2(item_cnt[i], 0); }
  __device__ void emit(uint64_t i, U2 ex, U2) const { item_off[i] = ex.a + l_near[item[i].live]; }
};

// Slab bounds: one wave per item finds, for every owner of its row, the first
// Y entry at or past the slab's first column (and the last slab its segment's
// end).  The searches are chains of dependent loads, so they run here, a lane
// each over the whole chip, and the item kernels read their results coalesced.
__global__ __launch_bounds__(kBlock) void k_ra_split(ItemArgs x) {
  const uint64_t total = *x.total;
  const uint64_t nw = (uint64_t)gridDim.x * (kBlock / kWave);
  const uint32_t lane = lane_id();
  for (uint64_t it = (uint64_t)blockIdx.x * (kBlock / kWave) + wave_id(); it < total; it += nw) {
    const Item t = x.item[it];
    for (uint32_t i = lane; i < t.own; i += kWave) {
      const uint64_t j = (uint64_t)t.j0 + i;
      const uint32_t y0 = (uint32_t)x.a.act_ypos[j];
      const uint32_t y1 = y0 + (uint32_t)(x.a.act_prefix[j + 1] - x.a.act_prefix[j]);
      x.split[t.split + i] = t.c0 ? lower_bound32(x.a.ycol, y0, y1, t.c0) : y0;
      if (t.last()) x.split[t.split + t.own + i] = y1;
    }
  }
}

// Orders the workgroup's LDS accesses only: __syncthreads also waits for the
// global stores before it, here an item's outputs on their way to HBM.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// ---- an item's products --------------------------------------------------------
// Owners are taken NT at a time.  An owner's run of products is cut into units
// of 2^uw lanes; a table gives each unit's owner (a search per unit, not per
// product), and every 2^uw lanes of the workgroup take units in turn, four
// units' gathers in flight.
constexpr uint32_t kUnits = 1024;

// An owner as its units see it: unit u's lane `sub` takes Y entry
// base + (u << ub) + sub while that is below end.
struct alignas(16) Owner {
  uint32_t base, end;
  float xv;
  uint32_t pad;
};
template <int NT>
struct OwnerSmem {
  Owner own[NT];
  uint32_t upre[NT + 1];  // units before each
  uint16_t utab[kUnits];
  uint32_t red[NT / kWave];
};

// Stages owners jb .. jb + NT - 1 (their entries of columns [ca, cb) when
// `cut`, else of the whole slab); returns the units.
template <int NT>
__device__ __forceinline__ uint32_t load_owners(const ItemArgs& x, const Item& t, uint32_t jb,
                                                int ub, bool cut, uint32_t ca, uint32_t cb,
                                                OwnerSmem<NT>& sm) {
  const uint32_t i = jb + threadIdx.x;
  uint32_t s = 0, e = 0;
  float xv = 0.f;
  if (i < t.own) {
    s = x.split[t.split + i];
    e = x.split[t.split + t.own + i];
    if (cut) {
      s = lower_bound32(x.a.ycol, s, e, ca);
      e = lower_bound32(x.a.ycol, s, e, cb);
    }
    xv = x.a.act_xval[(uint64_t)t.j0 + i];
  }
  const uint32_t units = (e - s + (1u << ub) - 1) >> ub;
  uint32_t tot;
  const uint32_t ex = block_scan_u32<NT>(units, sm.red, &tot);  // barriers inside
  sm.own[threadIdx.x] = Owner{s - (ex << ub), e, xv, 0};
  sm.upre[threadIdx.x] = ex;
  if (threadIdx.x == 0) sm.upre[NT] = tot;
  __syncthreads();
  return tot;
}

// Owners of batch jb.
template <int NT>
__device__ __forceinline__ uint32_t staged(const Item& t, uint32_t jb) {
  return t.own - jb < (uint32_t)NT ? t.own - jb : (uint32_t)NT;
}

// f(X values, Y entries, valid) for every four products of the `n` staged
// owners; ends with a barrier.  An invalid product's entry is 0: f loads
// without a test, since a load inside a branch is waited for there, one
// product's latency after another's.
template <int NT, class F>
__device__ __forceinline__ void for_units(OwnerSmem<NT>& sm, uint32_t n, uint32_t U, int ub,
                                          F&& f) {
  const uint32_t g = threadIdx.x >> ub, sub = threadIdx.x & ((1u << ub) - 1);
  const uint32_t G = (uint32_t)NT >> ub;
  for (uint32_t u0 = 0; u0 < U; u0 += kUnits) {
    const uint32_t m = U - u0 < kUnits ? U - u0 : kUnits;
    for (uint32_t i = threadIdx.x; i < m; i += NT) {
      uint32_t lo = 0, hi = n;  // last owner with upre <= u0 + i
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (sm.upre[mid] <= u0 + i) lo = mid; else hi = mid;
      }
      sm.utab[i] = (uint16_t)lo;
    }
    lds_barrier();
    for (uint32_t i = g; i < m; i += 4 * G) {
      uint32_t y[4];
      float xv[4];
      bool ok[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t u = i + (uint32_t)e * G;
        const Owner w = sm.own[sm.utab[u < m ? u : 0]];
        const uint32_t p = w.base + ((u0 + u) << ub) + sub;
        ok[e] = (u < m) & (p < w.end);
        y[e] = ok[e] ? p : 0;
        xv[e] = w.xv;
      }
      f(xv, y, ok);
    }
    lds_barrier();
  }
}

// ---- count -----------------------------------------------------------------------
// 8 KiB of bitmap and 7 KiB of owners at 256 threads: eight workgroups per CU.
// An item is a chain of waits (descriptor, owners, gathers, barriers), so what
// counts is how many are in flight; the next descriptor is fetched early.
// SUM (count-only runs): also the sum of the products.
constexpr int kCountNT = 256;

template <bool SUM>
__global__ __launch_bounds__(kCountNT) void k_ra_count(ItemArgs x, uint32_t* __restrict__ live_cnt,
                                                       uint32_t* __restrict__ item_cnt) {
  __shared__ alignas(16) uint32_t bm[kSlabCols / 32];
  __shared__ OwnerSmem<kCountNT> sm;
  __shared__ double s_sum[kCountNT / kWave];
  const uint32_t tid = threadIdx.x;
  const uint64_t total = *x.total;
  double vs = 0.0;
  Item nt = {};
  if (blockIdx.x < total) nt = x.item[blockIdx.x];
  for (uint64_t it = blockIdx.x; it < total; it += gridDim.x) {
    const Item t = nt;
    if (it + gridDim.x < total) nt = x.item[it + gridDim.x];
    const int ub = t.unit_bits();
    const uint32_t nw = 2 * t.words();
    for (uint32_t i = tid; i < nw; i += kCountNT) bm[i] = 0;
    for (uint32_t jb = 0; jb < t.own; jb += kCountNT) {
      const uint32_t U = load_owners<kCountNT>(x, t, jb, ub, false, 0, 0, sm);
      for_units<kCountNT>(sm, staged<kCountNT>(t, jb), U, ub,
                          [&](const float (&xv)[4], const uint32_t (&y)[4], const bool (&ok)[4]) {
        uint32_t c[4];
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          c[e] = x.a.ycol[y[e]] - t.c0;
          if (SUM) v[e] = xv[e] * x.a.yvals[y[e]];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (ok[e]) atomicOr(&bm[c[e] >> 5], 1u << (c[e] & 31));
          if (SUM) vs += ok[e] ? (double)v[e] : 0.0;
        }
      });
    }
    uint32_t c = 0;
    uint32_t* words = SUM || !x.words ? nullptr : reinterpret_cast<uint32_t*>(x.words + t.word);
    for (uint32_t i = tid; i < nw; i += kCountNT) {
      const uint32_t b = bm[i];
      c += (uint32_t)__popc(b);
      if (words) words[i] = b;
    }
    uint32_t tot;
    block_scan_u32<kCountNT>(c, sm.red, &tot);
    if (tid == 0) {
      item_cnt[it] = tot;
      if (tot) atomicAdd(&live_cnt[t.live], tot);
    }
  }
  if (SUM) {
    for (int off = kWave / 2; off > 0; off >>= 1) vs += __shfl_xor(vs, off, kWave);
    if (lane_id() == 0) s_sum[wave_id()] = vs;
    __syncthreads();
    if (tid == 0) {
      double u = 0.0;
      for (int w = 0; w < kCountNT / kWave; ++w) u += s_sum[w];
      slot_add(x.a.vsum, u);
    }
  }
}

// ---- sum ---------------------------------------------------------------------------
// 79 KiB of LDS at 512 threads (bitmap 8, ranks 4, slots 44, slot columns 11,
// owners 12): two workgroups, 16 waves, per CU.  The bitmap is the count's
// (WORDS) or is marked again.  Of 5.9 ms (1.36e9 products in 3.4e5 items), the
// products take about 1.5 and the stores 1.9, the rest is the items' own.
constexpr int kSumNT = 512;
constexpr uint32_t kSlots = 5632;  // 3072 (and items to match): 10.4 against 9.0 ms
constexpr uint32_t kSumPer = kSlabCols / 64 / kSumNT;  // bitmap words per thread

struct SumSmem {
  alignas(16) uint32_t bm[kSlabCols / 32];
  uint32_t pre[kSlabCols / 64 + 1];  // columns marked before each 64
  double slot[kSlots];
  uint16_t col[kSlots];
  OwnerSmem<kSumNT> own;
  uint64_t red[kSumNT / kWave];
  uint32_t we;
};
typedef uint64_t u64_alias __attribute__((__may_alias__));

// Adds the products of the staged owners to the slots of columns ranked r0 on,
// and notes the slots' columns.
__device__ __forceinline__ void add_units(const ItemArgs& x, SumSmem& sm, uint32_t c0, uint32_t r0,
                                          const float (&xv)[4], const uint32_t (&y)[4],
                                          const bool (&ok)[4], double& vs) {
  const u64_alias* bm64 = reinterpret_cast<const u64_alias*>(sm.bm);
  uint32_t c[4], sl[4];
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    c[e] = x.a.ycol[y[e]];
    v[e] = x.a.yvals[y[e]];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    c[e] = ok[e] ? c[e] - c0 : 0;
    v[e] = ok[e] ? xv[e] * v[e] : 0.f;
    const uint32_t w = c[e] >> 6;
    const uint64_t below = bm64[w] & ((1ull << (c[e] & 63)) - 1);
    sl[e] = sm.pre[w] - r0 + (uint32_t)__popcll(below);
    vs += (double)v[e];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (ok[e]) {
      atomicAdd(&sm.slot[sl[e]], (double)v[e]);
      sm.col[sl[e]] = (uint16_t)c[e];
    }
}

// Writes slots [0, m) at output ob: streaming stores of whole 128-byte lines
// but at the run's ends (lanes are counted from the 32-output boundary below
// its start).
__device__ __forceinline__ void store_slots(const ItemArgs& x, const SumSmem& sm, uint32_t row,
                                            uint32_t c0, uint32_t m, uint64_t ob,
                                            uint32_t* __restrict__ out_row,
                                            uint64_t* __restrict__ out_col,
                                            float* __restrict__ out_val) {
  const uint64_t al = ob & ~31ull;
  const uint32_t lead = (uint32_t)(ob - al);
  for (uint32_t j0 = 0; j0 < lead + m; j0 += 4 * kSumNT) {
    uint64_t c[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {  // four gathers in flight
      const uint32_t i = j0 + (uint32_t)e * kSumNT + threadIdx.x - lead;
      const uint32_t rk = c0 + sm.col[i < m ? i : 0];
      c[e] = x.a.ytab32 ? (uint64_t)x.a.ytab32[rk] : x.a.ytab ? x.a.ytab[rk] : rk;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t jj = j0 + (uint32_t)e * kSumNT + threadIdx.x;
      const uint32_t i = jj - lead;  // wraps below lead
      if (i >= m) continue;
      __builtin_nontemporal_store(row, &out_row[al + jj]);
      __builtin_nontemporal_store(c[e], &out_col[al + jj]);
      __builtin_nontemporal_store((float)sm.slot[i], &out_val[al + jj]);
    }
  }
}

// An item of at most kSlots outputs and kSumNT owners with its bitmap kept --
// nearly all -- takes five barriers, and everything it needs before its
// gathers (descriptor, bitmap, owners) was loaded during the item before it:
// per-item waits, not its products, were its time.  Others go window by
// window of at most kSlots outputs (take_windows).
struct Ahead {
  uint64_t wd[kSumPer];
  uint32_t s, e;
  float xv;
};

__device__ __forceinline__ void load_ahead(const ItemArgs& x, const Item& t, Ahead& p) {
  const uint32_t nw = t.words(), i = threadIdx.x;
#pragma unroll
  for (uint32_t e = 0; e < kSumPer; ++e) {
    const uint32_t w = i * kSumPer + e;
    p.wd[e] = x.words[t.word + (w < nw ? w : 0)];
  }
  const uint32_t k = i < t.own ? i : 0;
  p.s = x.split[t.split + k];
  p.e = x.split[t.split + t.own + k];
  p.xv = x.a.act_xval[(uint64_t)t.j0 + k];
}

template <bool WORDS>
__device__ __forceinline__ void take_windows(const ItemArgs& x, const Item& t, uint64_t obase,
                                             SumSmem& sm, double& vs,
                                             uint32_t* __restrict__ out_row,
                                             uint64_t* __restrict__ out_col,
                                             float* __restrict__ out_val) {
  const uint32_t tid = threadIdx.x;
  const int ub = t.unit_bits();
  const uint32_t nw = t.words();
  u64_alias* bm64 = reinterpret_cast<u64_alias*>(sm.bm);
  __syncthreads();
  if (WORDS) {
    for (uint32_t w = tid; w < nw; w += kSumNT) bm64[w] = x.words[t.word + w];
  } else {
    for (uint32_t i = tid; i < 2 * nw; i += kSumNT) sm.bm[i] = 0;
    for (uint32_t jb = 0; jb < t.own; jb += kSumNT) {
      const uint32_t U = load_owners<kSumNT>(x, t, jb, ub, false, 0, 0, sm.own);
      for_units<kSumNT>(sm.own, staged<kSumNT>(t, jb), U, ub,
                        [&](const float (&)[4], const uint32_t (&y)[4], const bool (&ok)[4]) {
        uint32_t c[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) c[e] = x.a.ycol[y[e]] - t.c0;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (ok[e]) atomicOr(&sm.bm[c[e] >> 5], 1u << (c[e] & 31));
      });
    }
  }
  __syncthreads();
  uint32_t pc[kSumPer], sum = 0, all;
#pragma unroll
  for (uint32_t e = 0; e < kSumPer; ++e) {
    const uint32_t w = tid * kSumPer + e;
    pc[e] = w < nw ? (uint32_t)__popcll(bm64[w]) : 0;
    sum += pc[e];
  }
  uint32_t ex = block_scan_u32<kSumNT>(sum, sm.own.red, &all);
#pragma unroll
  for (uint32_t e = 0; e < kSumPer; ++e) {
    const uint32_t w = tid * kSumPer + e;
    if (w < nw) sm.pre[w] = ex;
    ex += pc[e];
  }
  if (tid == 0) sm.pre[nw] = all;
  __syncthreads();
  const bool whole = all <= kSlots;  // one window: no cut
  for (uint32_t ws = 0; ws < nw;) {
    // the window: whole words of the bitmap with at most kSlots columns
    const uint32_t r0 = sm.pre[ws];
    uint32_t we = nw;
    if (!whole) {
      if (tid == 0) sm.we = ws + 1;
      __syncthreads();
      for (uint32_t w = ws + 1 + tid; w < nw; w += kSumNT)
        if (sm.pre[w + 1] - r0 <= kSlots) atomicMax(&sm.we, w + 1);
      __syncthreads();
      we = sm.we;
    }
    const uint32_t m = sm.pre[we] - r0;
    for (uint32_t i = tid; i < m; i += kSumNT) sm.slot[i] = 0.0;
    __syncthreads();
    if (m) {
      for (uint32_t jb = 0; jb < t.own; jb += kSumNT) {
        const uint32_t U =
            load_owners<kSumNT>(x, t, jb, ub, !whole, t.c0 + ws * 64, t.c0 + we * 64, sm.own);
        for_units<kSumNT>(sm.own, staged<kSumNT>(t, jb), U, ub,
                          [&](const float (&xv)[4], const uint32_t (&y)[4],
                              const bool (&ok)[4]) { add_units(x, sm, t.c0, r0, xv, y, ok, vs); });
      }
      store_slots(x, sm, t.row, t.c0, m, obase + r0, out_row, out_col, out_val);
    }
    __syncthreads();
    ws = we;
  }
}

__device__ __forceinline__ Item uniform(const Item& t) {
  Item u;
  u.j0 = __builtin_amdgcn_readfirstlane(t.j0);
  u.own = __builtin_amdgcn_readfirstlane(t.own);
  u.split = __builtin_amdgcn_readfirstlane(t.split);
  u.c0 = __builtin_amdgcn_readfirstlane(t.c0);
  u.W = __builtin_amdgcn_readfirstlane(t.W);
  u.live = __builtin_amdgcn_readfirstlane(t.live);
  u.row = __builtin_amdgcn_readfirstlane(t.row);
  u.word = __builtin_amdgcn_readfirstlane(t.word);
  return u;
}

template <bool WORDS>
__global__ __launch_bounds__(kSumNT) void k_ra_sum(ItemArgs x, uint64_t nitems,
                                                   const uint32_t* __restrict__ item_cnt,
                                                   const uint64_t* __restrict__ item_off,
                                                   uint32_t* __restrict__ out_row,
                                                   uint64_t* __restrict__ out_col,
                                                   float* __restrict__ out_val) {
  __shared__ SumSmem sm;
  __shared__ double s_sum[kSumNT / kWave];
  const uint32_t tid = threadIdx.x, lane = lane_id(), wave = wave_id();
  u64_alias* bm64 = reinterpret_cast<u64_alias*>(sm.bm);
  double vs = 0.0;
  // descriptors two items ahead, bitmap and owners one ahead
  const uint64_t last = nitems - 1, G = gridDim.x;
  auto at = [&](uint64_t i) { return i < last ? i : last; };
  Item d1 = x.item[at(blockIdx.x)], d2 = x.item[at(blockIdx.x + G)];
  uint32_t n1 = item_cnt[at(blockIdx.x)], n2 = item_cnt[at(blockIdx.x + G)];
  uint64_t o1 = item_off[at(blockIdx.x)], o2 = item_off[at(blockIdx.x + G)];
  Ahead p1;
  if (WORDS) load_ahead(x, d1, p1);
  for (uint64_t it = blockIdx.x; it < nitems; it += G) {
    const Item t = uniform(d1);
    const uint32_t outs = __builtin_amdgcn_readfirstlane(n1);
    const uint64_t obase = o1;
    const Ahead p = p1;
    d1 = d2;
    n1 = n2;
    o1 = o2;
    if (WORDS) load_ahead(x, d1, p1);
    d2 = x.item[at(it + 2 * G)];
    n2 = item_cnt[at(it + 2 * G)];
    o2 = item_off[at(it + 2 * G)];
    if (!outs) continue;
    if (!WORDS || outs > kSlots || t.own > (uint32_t)kSumNT) {
      take_windows<WORDS>(x, t, obase, sm, vs, out_row, out_col, out_val);
      continue;
    }
    const int ub = t.unit_bits();
    const uint32_t nw = t.words();
    // ranks of the bitmap's words and units of the owners in one scan
    uint32_t marked = 0;
#pragma unroll
    for (uint32_t e = 0; e < kSumPer; ++e)
      marked += tid * kSumPer + e < nw ? (uint32_t)__popcll(p.wd[e]) : 0;
    const uint32_t cnt = tid < t.own ? p.e - p.s : 0;
    const uint32_t units = (cnt + (1u << ub) - 1) >> ub;
    const uint64_t both = (uint64_t)marked << 32 | units;
    const uint64_t inc = wave_incl_scan(both);
    lds_barrier();  // the item before has been stored
    if (lane == kWave - 1) sm.red[wave] = inc;
    lds_barrier();
    uint64_t ex = inc - both, all = 0;
#pragma unroll
    for (uint32_t w = 0; w < kSumNT / kWave; ++w) {
      const uint64_t r = sm.red[w];
      ex += w < wave ? r : 0;
      all += r;
    }
    uint32_t rank = (uint32_t)(ex >> 32);
#pragma unroll
    for (uint32_t e = 0; e < kSumPer; ++e) {
      const uint32_t w = tid * kSumPer + e;
      if (w < nw) {
        bm64[w] = p.wd[e];
        sm.pre[w] = rank;
        rank += (uint32_t)__popcll(p.wd[e]);
      }
    }
    sm.own.own[tid] = Owner{p.s - ((uint32_t)ex << ub), tid < t.own ? p.e : 0u, p.xv, 0};
    sm.own.upre[tid] = (uint32_t)ex;
    const uint32_t U = (uint32_t)all;
    for (uint32_t i = tid; i < outs; i += kSumNT) sm.slot[i] = 0.0;
    lds_barrier();
    for_units<kSumNT>(sm.own, t.own, U, ub,
                      [&](const float (&xv)[4], const uint32_t (&y)[4], const bool (&ok)[4]) {
      add_units(x, sm, t.c0, 0, xv, y, ok, vs);
    });
    store_slots(x, sm, t.row, t.c0, outs, obase, out_row, out_col, out_val);
  }
  for (int off = kWave / 2; off > 0; off >>= 1) vs += __shfl_xor(vs, off, kWave);
  if (lane == 0) s_sum[wave] = vs;
  __syncthreads();
  if (tid == 0) {
    double u = 0.0;
    for (int w = 0; w < kSumNT / kWave; ++w) u += s_sum[w];
    slot_add(x.a.vsum, u);
  }
}

// ---- short rows --------------------------------------------------------------------
// First index of v[0 .. n) with v[i] >= c, by a whole wave (64-way rounds).
__device__ __forceinline__ uint32_t wave_lower_bound32(const uint32_t* __restrict__ v, uint32_t n,
                                                       uint64_t c) {
  const uint32_t lane = lane_id();
  uint32_t lo = 0, hi = n;  // answer in [lo, hi]
  while (hi - lo > (uint32_t)kWave) {
    const uint32_t step = (hi - lo + kWave - 1) / kWave;
    const uint64_t i = (uint64_t)lo + (uint64_t)lane * step;
    const uint32_t k = (uint32_t)__popcll(__ballot(i < hi && v[i] < c));  // a prefix of the lanes
    if (!k) return lo;
    const uint64_t nh = (uint64_t)lo + (uint64_t)k * step;
    lo = lo + (k - 1) * step + 1;
    hi = nh < hi ? (uint32_t)nh : hi;
  }
  const uint32_t i = lo + lane;
  return lo + (uint32_t)__popcll(__ballot(i < hi && v[i] < c));
}

struct GroupArgs {
  RowAccArgs a;
  const uint32_t *live_row, *s_live, *s_prod;
  uint32_t nshort, prods;
  uint32_t* live_cnt;
  uint64_t* live_src;
  uint32_t* tcol;  // NULL: counts and the value sum only
  float* tval;
};

struct GroupOwners {          // while the products are made
  uint32_t y[kGroupTile];     // first Y entry minus the owner's first product
  float x[kGroupTile];
  uint16_t first[kGroupTile]; // first product in the group
  uint16_t row[kGroupTile];
};
template <typename KT>
struct GroupSort {            // while they are sorted
  TileSmem<10, kGroupIPT, kGroupNT, KT> t;
  float v[kGroupTile];
};
constexpr uint32_t kGroupRows = kGroupHalf + 1;  // rows hold a product at least

// One workgroup per group of short rows: their owners are staged (a lane
// each), every product finds its owner by an LDS search, makes its key (row
// in the group, column) and value, and the group is sorted on the bits that
// vary by stable LDS passes of 10 bits.  Runs of equal keys are summed by the
// lane at their head; the outputs go to (tcol, tval) from the group's first
// product on, compacted, with each row's count and place.
// KT: 32 bits hold the key while the column has at most kGroupBits.  (8e6 x 3e6
// nonzeros, 0.23e6 products in short rows over 2^22 columns, 7.4e6 rows: call 2970
// us by the product sort, of which 590 in its row tables, 1753 here.)
constexpr int kGroupBits = 21;  // and a row of the group 11
template <typename KT>
__global__ __launch_bounds__(kGroupNT) void k_ra_group(GroupArgs g) {
  __shared__ union {
    GroupOwners own;
    GroupSort<KT> sort;
  } sm;
  __shared__ uint32_t s_live[kGroupRows], s_j0[kGroupRows];
  __shared__ uint16_t s_first[kGroupRows + 1], s_own[kGroupRows + 1];
  __shared__ uint32_t s_k[2], red[kGroupNT / kWave], s_or[kGroupNT / kWave];
  __shared__ double s_sum[kGroupNT / kWave];
  constexpr int IPT = kGroupIPT, NT = kGroupNT, RB = 10, R = 1 << RB;
  const uint32_t tid = threadIdx.x, lane = lane_id(), wave = wave_id();
  if (tid < 2 * kWave) {
    const uint64_t c = ((uint64_t)blockIdx.x + wave) * kGroupHalf;
    const uint32_t k = c >= g.prods ? g.nshort : wave_lower_bound32(g.s_prod, g.nshort, c);
    if (lane == 0) s_k[wave] = k;
  }
  __syncthreads();
  const uint32_t k0 = s_k[0], nr = s_k[1] - s_k[0];
  if (!nr) return;
  const uint32_t base = g.s_prod[k0];
  const uint32_t n = (k0 + nr < g.nshort ? g.s_prod[k0 + nr] : g.prods) - base;
  uint32_t no = 0;
  for (uint32_t b = 0; b < nr; b += NT) {
    const uint32_t i = b + tid;
    uint32_t own = 0;
    if (i < nr) {
      const uint32_t k = g.s_live[k0 + i];
      const uint64_t r = g.a.r0 + g.live_row[k];
      const uint64_t j0 = g.a.row_act[r];
      own = (uint32_t)(g.a.row_act[r + 1] - j0);
      s_live[i] = k;
      s_j0[i] = (uint32_t)j0;
      s_first[i] = (uint16_t)(g.s_prod[k0 + i] - base);
    }
    uint32_t tot;
    const uint32_t ex = block_scan_u32<NT>(own, red, &tot);
    if (i < nr) s_own[i] = (uint16_t)(no + ex);
    no += tot;
  }
  __syncthreads();
  for (uint32_t o = tid; o < no; o += NT) {
    uint32_t lo = 0, hi = nr;  // last row whose owners start at or before o
    while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) >> 1;
      if (s_own[mid] <= o) lo = mid; else hi = mid;
    }
    const uint64_t j = (uint64_t)s_j0[lo] + (o - s_own[lo]);
    const uint32_t first =
        s_first[lo] + (uint32_t)(g.a.act_prefix[j] - g.a.act_prefix[s_j0[lo]]);
    sm.own.y[o] = (uint32_t)g.a.act_ypos[j] - first;
    sm.own.x[o] = g.a.act_xval[j];
    sm.own.first[o] = (uint16_t)first;
    sm.own.row[o] = (uint16_t)lo;
  }
  __syncthreads();
  const uint32_t wbase = wave * (kWave * IPT);
  KT k[IPT];
  uint32_t rr[IPT], ow[IPT], pos[IPT];
  float v[IPT];
  double vs = 0.0;
  uint32_t cor = 0;
#pragma unroll
  for (int i = 0; i < IPT; ++i) {
    const uint32_t p = wbase + (uint32_t)i * kWave + lane;
    uint32_t lo = 0, hi = no;  // last owner whose products start at or before p
    while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) >> 1;
      if (sm.own.first[mid] <= p) lo = mid; else hi = mid;
    }
    rr[i] = sm.own.row[lo];
    ow[i] = lo;
    pos[i] = p < n ? sm.own.y[lo] + p : 0;
  }
#pragma unroll
  for (int i = 0; i < IPT; ++i) {  // all the gathers in flight
    k[i] = g.a.ycol[pos[i]];
    v[i] = g.a.yvals[pos[i]];
  }
#pragma unroll
  for (int i = 0; i < IPT; ++i) {
    const bool ok = wbase + (uint32_t)i * kWave + lane < n;
    k[i] = ok ? k[i] : 0;
    v[i] = ok ? sm.own.x[ow[i]] * v[i] : 0.f;
    vs += (double)v[i];
    cor |= (uint32_t)k[i];
  }
  for (int off = kWave / 2; off > 0; off >>= 1) cor |= __shfl_xor(cor, off, kWave);
  for (int off = kWave / 2; off > 0; off >>= 1) vs += __shfl_xor(vs, off, kWave);
  if (lane == 0) {
    s_or[wave] = cor;
    s_sum[wave] = vs;
  }
  __syncthreads();  // (the owners are read: their LDS is the sort's from here on)
  cor = 0;
  for (int w = 0; w < NT / kWave; ++w) cor |= s_or[w];
  if (tid == 0) {
    double u = 0.0;
    for (int w = 0; w < NT / kWave; ++w) u += s_sum[w];
    slot_add(g.a.vsum, u);
  }
  // the row goes right above the bits the group's columns use
  const int cb = cor ? 32 - __builtin_clz(cor) : 0;
  const int rbits = nr > 1 ? 32 - __builtin_clz(nr - 1) : 0;
#pragma unroll
  for (int i = 0; i < IPT; ++i) k[i] |= (KT)rr[i] << cb;
  const int passes = (cb + rbits + RB - 1) / RB;
  auto& sb = sm.sort;
  if (!passes) {  // one column of one row
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
      const uint32_t p = wbase + (uint32_t)i * kWave + lane;
      sb.t.buf[p] = 0;
      sb.v[p] = v[i];
    }
    __syncthreads();
  }
  for (int ps = 0; ps < passes; ++ps) {
    const int shift = ps * RB;
    for (int i = tid; i < (NT / kWave) * R; i += NT) (&sb.t.cnt[0][0])[i] = 0;
    __syncthreads();
    tile_rank<false, RB, IPT, NT>(sb.t, n, shift, k, pos);
    __syncthreads();
    tile_prefix_fold<RB, IPT, NT>(sb.t);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
      const uint32_t p = wbase + (uint32_t)i * kWave + lane;
      if (p < n) {
        const uint32_t q = pos[i] + (uint32_t)sb.t.cnt[wave][(uint32_t)(k[i] >> shift) & (R - 1)];
        sb.t.buf[q] = k[i];
        sb.v[q] = v[i];
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
      const uint32_t p = wbase + (uint32_t)i * kWave + lane;
      if (p < n) {
        k[i] = sb.t.buf[p];
        v[i] = sb.v[p];
      }
    }
    __syncthreads();
  }
  // heads in sorted order: (wave, item, lane) is the sorted order
  uint32_t hm = 0, run = 0;
#pragma unroll
  for (int i = 0; i < IPT; ++i) {
    const uint32_t p = wbase + (uint32_t)i * kWave + lane;
    const bool head = p < n && (p == 0 || sb.t.buf[p - 1] != k[i]);
    const uint64_t b = __ballot(head);
    pos[i] = run + popc_below(b);
    run += (uint32_t)__popcll(b);
    hm |= (uint32_t)head << i;
  }
  if (lane == 0) red[wave] = run;
  __syncthreads();
  uint32_t before = 0, T = 0;
  for (uint32_t w = 0; w < NT / kWave; ++w) {
    before += w < wave ? red[w] : 0;
    T += red[w];
  }
  const uint32_t cmask = (uint32_t)low_mask(cb);
  constexpr int kBits = (int)sizeof(KT) * 8;
#pragma unroll
  for (int i = 0; i < IPT; ++i) {
    if (!((hm >> i) & 1u)) continue;
    const uint32_t p = wbase + (uint32_t)i * kWave + lane;
    const uint32_t o = before + pos[i];
    const uint32_t row = cb < kBits ? (uint32_t)(k[i] >> cb) : 0;
    if (p == 0 || (cb < kBits ? (uint32_t)(sb.t.buf[p - 1] >> cb) : 0) != row) s_first[row] = (uint16_t)o;
    if (g.tcol) {
      SumF64 s;
      s.add(v[i]);
      for (uint32_t q = p + 1; q < n && sb.t.buf[q] == k[i]; ++q) s.add(sb.v[q]);
      g.tcol[base + o] = (uint32_t)k[i] & cmask;
      g.tval[base + o] = s.value();
    }
  }
  __syncthreads();
  for (uint32_t i = tid; i < nr; i += NT) {
    const uint32_t f = s_first[i];
    g.live_cnt[s_live[i]] = (i + 1 < nr ? (uint32_t)s_first[i + 1] : T) - f;
    g.live_src[s_live[i]] = kShortSrc | (base + f);
  }
}

// ---- near rows: outputs ----------------------------------------------------------------
// Tiles of 2048 outputs of the one-owner and short rows (every such row has
// one at least, so a tile meets at most 2048 rows); an output finds its row by
// an LDS search from its previous one's.  Bound by the 16 bytes stored per
// output and the 8 read.  OUT = false (count-only): the one-owner rows' value
// sum alone.
constexpr int kNearItems = 8;
constexpr uint32_t kNearTile = kBlock * kNearItems;

struct NearArgs {
  RowAccArgs a;
  const uint32_t* near_pre;
  const Near* near;
  uint32_t near_rows, near_outs;
  const uint32_t* tcol;
  const float* tval;
  uint32_t* out_row;
  uint64_t* out_col;
  float* out_val;
};

template <bool OUT>
__global__ __launch_bounds__(kBlock) void k_ra_near(NearArgs g, uint32_t ntiles) {
  __shared__ uint32_t s_pre[kNearTile + 1];
  __shared__ uint32_t s_m[2];
  __shared__ double s_sum[kBlock / kWave];
  const uint32_t tid = threadIdx.x;
  double vs = 0.0;
  for (uint32_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const uint32_t ob = tile * kNearTile;
    const uint32_t oe = g.near_outs - ob < kNearTile ? g.near_outs : ob + kNearTile;
    __syncthreads();
    if (tid < 2 * kWave) {  // rows of the first and the last output
      const uint64_t o = tid < kWave ? ob : oe - 1;
      const uint32_t m = wave_lower_bound32(g.near_pre, g.near_rows, o + 1) - 1;
      if (lane_id() == 0) s_m[wave_id()] = m;
    }
    __syncthreads();
    const uint32_t m0 = s_m[0], nm = s_m[1] - m0 + 1;
    for (uint32_t i = tid; i < nm; i += kBlock) s_pre[i] = g.near_pre[m0 + i];
    __syncthreads();
    // an output's row: its place and Y entry (or the groups' output), looked
    // up when the row changes; then all the thread's loads, then its stores
    uint32_t cur = 0, kc = ~0u, row = 0;
    uint64_t off = 0, y0 = 0;
    float xv = 0.f;
    bool is_one = false;
    uint64_t y[kNearItems], at[kNearItems];
    float x[kNearItems];
    uint32_t rw[kNearItems], one = 0;
#pragma unroll
    for (int e = 0; e < kNearItems; ++e) {
      const uint32_t o = ob + (uint32_t)e * kBlock + tid;
      y[e] = at[e] = 0;
      x[e] = 0.f;
      rw[e] = 0;
      if (o < oe) {
        uint32_t i = cur;
        if (i + 1 < nm && s_pre[i + 1] <= o) {
          uint32_t lo = i + 1, hi = nm;
          while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (s_pre[mid] <= o) lo = mid; else hi = mid;
          }
          i = lo;
        }
        cur = i;
        if (i != kc) {
          kc = i;
          const Near d = g.near[m0 + i];
          off = d.off - s_pre[i];
          y0 = (d.src & ~kShortSrc) - s_pre[i];
          row = d.row;
          xv = d.x;
          is_one = d.src < kShortSrc;
        }
        y[e] = y0 + o;
        at[e] = off + o;
        x[e] = xv;
        rw[e] = row;
        one |= (uint32_t)is_one << e;
      }
    }
    const uint32_t valid = [&] {
      uint32_t v = 0;
#pragma unroll
      for (int e = 0; e < kNearItems; ++e)
        v |= (uint32_t)(ob + (uint32_t)e * kBlock + tid < oe) << e;
      return v;
    }();
    const uint32_t grp = valid & ~one;
    float v[kNearItems];
    uint64_t c[kNearItems];
#pragma unroll
    for (int e = 0; e < kNearItems; ++e) {
      const uint64_t i = (one >> e & 1) ? y[e] : 0;
      v[e] = g.a.yvals[i];
      if (OUT) c[e] = g.a.yfree32 ? (uint64_t)g.a.yfree32[i] : g.a.ykeys[i] & g.a.yfmask;
    }
#pragma unroll
    for (int e = 0; e < kNearItems; ++e) {
      v[e] = x[e] * v[e];
      vs += (one >> e & 1) ? (double)v[e] : 0.0;
      v[e] += 0.f;  // a sum of one product: no negative zero
    }
    if (OUT && __ballot(grp != 0)) {
      uint32_t rk[kNearItems];
#pragma unroll
      for (int e = 0; e < kNearItems; ++e) {
        const bool is = grp >> e & 1;
        rk[e] = is ? g.tcol[y[e]] : 0;
        v[e] = is ? g.tval[y[e]] : v[e];
      }
#pragma unroll
      for (int e = 0; e < kNearItems; ++e)
        if (grp >> e & 1)
          c[e] = g.a.ytab32 ? (uint64_t)g.a.ytab32[rk[e]] : g.a.ytab ? g.a.ytab[rk[e]] : rk[e];
    }
    if (OUT) {
#pragma unroll
      for (int e = 0; e < kNearItems; ++e) {
        if (!(valid >> e & 1)) continue;
        g.out_row[at[e]] = rw[e];
        g.out_col[at[e]] = c[e];
        g.out_val[at[e]] = v[e];
      }
    }
  }
  for (int off = kWave / 2; off > 0; off >>= 1) vs += __shfl_xor(vs, off, kWave);
  if (lane_id() == 0) s_sum[wave_id()] = vs;
  __syncthreads();
  if (tid == 0) {
    double u = 0.0;
    for (int w = 0; w < kBlock / kWave; ++w) u += s_sum[w];
    if (u != 0.0) slot_add(g.a.vsum, u);
  }
}

uint32_t grid_of(uint64_t n, uint64_t cap) {
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(n, cap));
}

ItemArgs item_args(const RowAccArgs& a, const RowAccPlan& p) {
  return ItemArgs{a, reinterpret_cast<const Item*>(p.item.get()), p.l_item.get() + p.nlong,
                  p.split.get(), p.keep_words ? p.words.get() : nullptr};
}

NearArgs near_args(const RowAccArgs& a, const RowAccPlan& p) {
  NearArgs g{};
  g.a = a;
  g.near_pre = p.near_pre.get();
  g.near = reinterpret_cast<const Near*>(p.near.get());
  g.near_rows = (uint32_t)p.near_rows;
  g.near_outs = (uint32_t)p.near_outs;
  g.tcol = p.tcol.get();
  g.tval = p.tval.get();
  return g;
}

// A buffer that grows goes back to the pool, where another thread may take it for
// its own stream: no launch may be under way.
template <class T>
void room(DevBuf<T>& b, uint64_t n) {
  if (b.size() < n) b.reset(n);
}

}  // namespace

// Upper bound of what a chunk's plan holds.
uint64_t rowacc_bytes(uint64_t rows, uint64_t owners, uint64_t nprod, uint64_t K) {
  const uint64_t live = std::min(rows, owners);
  const uint64_t least = K <= 1ull << kRowAccMaxBits ? min_slabs((uint32_t)K) : 1;
  const uint64_t items = nprod / 256 * least + nprod / kItemProds;  // long rows: 256 products
  const uint64_t b = live * (28 + 4 + 4 + kNearBytes) + 8 * nprod + items * (kItemBytes + 4 + 8) +
                     4 * (owners * (least + 1) + nprod / kItemRun) + 4 * nprod + (2ull << 20);
  return b + b / 8;  // the pool rounds large blocks up by as much
}

bool rowacc_count(const RowAccArgs& a, uint64_t nprod, uint64_t owners, bool count_only,
                  RowAccPlan* p, U2* host, hipStream_t s, KTimer* kt) {
  // every live row has an active X nonzero: the fewer of both are scanned
  const bool by_act = owners < a.rows;
  const uint64_t rows = by_act ? owners : a.rows;
  if (nprod >= (1ull << 32)) throw std::length_error("row accumulator chunk");
  // (column spaces too wide to cut into slabs take no long rows)
  const bool slabs = a.K <= 1u << kRowAccMaxBits;
  const uint32_t least = slabs ? min_slabs(a.K) : 1;
  // (items: long rows hold more than 256 products)
  const uint64_t ntmp =
      scan_tmp_count(std::max(rows, nprod / 256 * least + nprod / kItemProds)) + 1;
  if (p->live_row.size() < rows || p->tmp.size() < ntmp) {
    // the chunk before may still use them; with this chunk's sizes the largest
    // (the engine says so) this happens once
    if (p->tmp.size()) SPTC_HIP(hipStreamSynchronize(s));
    const uint64_t r = std::max(rows, p->rows_at_most);
    room(p->live_row, r);
    room(p->live_cnt, r);
    room(p->live_src, r);
    room(p->s_live, r);
    room(p->s_prod, r);
    room(p->l_live, r);
    room(p->tmp, std::max(ntmp, scan_tmp_count(std::max(r, p->prods_at_most / 256 * least +
                                                               p->prods_at_most / kItemProds)) +
                                    1));
  }
  const uint64_t heavy = std::max(kHeavyItem, nprod >> 10);
  const uint64_t weight = kHeavyWeight + (nprod >> 6);
  host[1].a = 0;
  auto kinds = [&](auto op) {
    op = {a, least, heavy, weight, &host[1].a, p->live_row.get(), p->live_cnt.get(),
          p->live_src.get(), p->s_live.get(), p->s_prod.get(), p->l_live.get()};
    run_scan(op, rows, p->tmp.get(), s, true, host);
  };
  if (by_act) kinds(RowKindOp<true>{});
  else kinds(RowKindOp<false>{});
  SPTC_HIP(hipStreamSynchronize(s));
  if (host[1].a || (!slabs && (host->b & 0xFFFFFFFFull))) return false;
  p->live = host->a & 0xFFFFFFFFull;
  p->short_prods = host->a >> 32;
  p->nshort = host->b >> 32;
  p->nlong = host->b & 0xFFFFFFFFull;
  p->items = 0;
  p->outs = p->near_outs = p->near_rows = 0;
  if (!p->live) return true;
  // slabs and split entries of the long rows: at most n / kItemProds slabs, and
  // owners * slabs at most n / kItemRun, past the least a row is cut into
  const uint64_t max_items = p->nlong * least + nprod / kItemProds;
  const uint64_t max_split = owners * (least + 1) + nprod / kItemRun;
  if (max_split >= (1ull << 32)) return false;  // 32-bit places in the descriptors
  // the bitmaps are kept from the count to the sum while they take no more
  // than a few bytes per product (one write and one read of K / 8 bytes per
  // row against another gather and LDS atomic per product)
  const uint64_t max_words = p->nlong * (a.K / 64 + 1) + max_items;
  p->keep_words = !count_only && max_words * 8 <= 4 * nprod + (1ull << 20);
  // (all tables, while nothing runs)
  if (!count_only) {
    room(p->tcol, p->short_prods);
    room(p->tval, p->short_prods);
  }
  if (p->nlong) {
    room(p->l_item, p->nlong + 1);
    room(p->l_split, p->nlong);
    room(p->l_word, p->nlong);
    room(p->item, max_items * (kItemBytes / 4));
    room(p->item_cnt, max_items);
    room(p->split, max_split);
    if (p->keep_words) room(p->words, max_words);
  }
  const bool new_quant = p->nlong && !p->quant.size();
  if (new_quant) p->quant.reset(kQuant + 1);
  room(p->l_near, p->live);
  room(p->near_pre, p->live);
  room(p->near, p->live * (kNearBytes / 8));
  if (p->nshort) {
    GroupArgs g{a,
                p->live_row.get(),
                p->s_live.get(),
                p->s_prod.get(),
                (uint32_t)p->nshort,
                (uint32_t)p->short_prods,
                p->live_cnt.get(),
                p->live_src.get(),
                count_only ? nullptr : p->tcol.get(),
                count_only ? nullptr : p->tval.get()};
    const int tok = kt->begin(s);
    const dim3 gg((uint32_t)ceil_div(p->short_prods, kGroupHalf)), gt(kGroupNT);
    if (a.K <= 1u << kGroupBits)
      hipLaunchKernelGGL(k_ra_group<uint32_t>, gg, gt, 0, s, g);
    else
      hipLaunchKernelGGL(k_ra_group<uint64_t>, gg, gt, 0, s, g);
    kt->end(tok, SPTC_K_SORT_LOCAL, (count_only ? 8.0 : 16.0) * (double)p->short_prods, s);
  }
  if (p->nlong) {
    SlabOp slab{a, least, p->l_live.get(), p->live_row.get(), p->nlong, p->l_item.get(),
                p->l_split.get(), p->l_word.get()};
    run_scan(slab, p->nlong, p->tmp.get(), s, true, host + 2);
    if (new_quant)
      hipLaunchKernelGGL(k_ra_quant, dim3(1), dim3(kQuantNT), 0, s, a.ycol, a.ny, a.K,
                         p->quant.get());
    hipLaunchKernelGGL(k_ra_items, dim3(grid_of(ceil_div(max_items, kBlock), 2048)), dim3(kBlock),
                       0, s, a, p->l_live.get(), p->live_row.get(), p->l_item.get(),
                       p->l_split.get(), p->l_word.get(), p->quant.get(), p->nlong,
                       reinterpret_cast<Item*>(p->item.get()));
    const ItemArgs x = item_args(a, *p);
    const int tok = kt->begin(s);
    hipLaunchKernelGGL(k_ra_split, dim3(grid_of(ceil_div(max_items, kBlock / kWave), 4096)),
                       dim3(kBlock), 0, s, x);
    const dim3 g(grid_of(max_items, 256 * 8 * 4));
    if (count_only)
      hipLaunchKernelGGL(k_ra_count<true>, g, dim3(kCountNT), 0, s, x, p->live_cnt.get(),
                         p->item_cnt.get());
    else
      hipLaunchKernelGGL(k_ra_count<false>, g, dim3(kCountNT), 0, s, x, p->live_cnt.get(),
                         p->item_cnt.get());
    kt->end(tok, SPTC_K_REDUCE, (count_only ? 8.0 : 4.0) * (double)(nprod - p->short_prods), s);
  }
  OutOp out{a,
            p->live_cnt.get(),
            p->live_row.get(),
            p->live_src.get(),
            p->l_near.get(),
            p->near_pre.get(),
            reinterpret_cast<Near*>(p->near.get())};
  run_scan(out, p->live, p->tmp.get(), s, true, host);
  SPTC_HIP(hipStreamSynchronize(s));
  p->outs = host[0].a;
  p->near_rows = host[0].b >> 32;
  p->near_outs = host[0].b & 0xFFFFFFFFull;
  if (p->nlong) p->items = host[2].a & 0xFFFFFFFFull;
  if (!count_only) room(p->item_off, p->items);
  if (count_only && p->near_outs) {
    const uint32_t nt = (uint32_t)ceil_div(p->near_outs, kNearTile);
    const int tok = kt->begin(s);
    hipLaunchKernelGGL(k_ra_near<false>, dim3(grid_of(nt, 8192)), dim3(kBlock), 0, s,
                       near_args(a, *p), nt);
    kt->end(tok, SPTC_K_EXPAND, 4.0 * (double)p->near_outs, s);
  }
  return true;
}

void rowacc_emit(const RowAccArgs& a, RowAccPlan& p, uint64_t nprod, uint32_t* out_row,
                 uint64_t* out_col, float* out_val, hipStream_t s, KTimer* kt) {
  if (p.near_outs) {
    NearArgs g = near_args(a, p);
    g.out_row = out_row;
    g.out_col = out_col;
    g.out_val = out_val;
    const uint32_t nt = (uint32_t)ceil_div(p.near_outs, kNearTile);
    const int tok = kt->begin(s);
    hipLaunchKernelGGL(k_ra_near<true>, dim3(grid_of(nt, 8192)), dim3(kBlock), 0, s, g, nt);
    kt->end(tok, SPTC_K_EXPAND, 24.0 * (double)p.near_outs, s);
  }
  if (p.items) {
    const int tok = kt->begin(s);
    ItemOutOp op{p.item_cnt.get(), reinterpret_cast<const Item*>(p.item.get()), p.l_near.get(),
                 p.item_off.get()};
    run_scan(op, p.items, p.tmp.get(), s);
    const dim3 g(grid_of(p.items, 256 * 3 * 8));
    const ItemArgs x = item_args(a, p);
    if (p.keep_words)
      hipLaunchKernelGGL(k_ra_sum<true>, g, dim3(kSumNT), 0, s, x, p.items, p.item_cnt.get(),
                         p.item_off.get(), out_row, out_col, out_val);
    else
      hipLaunchKernelGGL(k_ra_sum<false>, g, dim3(kSumNT), 0, s, x, p.items, p.item_cnt.get(),
                         p.item_off.get(), out_row, out_col, out_val);
    kt->end(tok, SPTC_K_REDUCE,
            12.0 * (double)(nprod - p.short_prods) + 16.0 * (double)(p.outs - p.near_outs), s);
  }
}

}  // namespace sptc
