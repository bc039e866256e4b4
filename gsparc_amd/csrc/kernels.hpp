// Host launchers and argument structs of the SpTC phase kernels.
#pragma once
#include "common.hpp"
#include "scan.hpp"
#include "sort.hpp"

namespace sptc {

constexpr int kMaxFusedPasses = 8;  // producers fuse histograms up to this many passes

// Packed key of a group of contracted coordinates, above the previous
// group's rank: key = prev << prev_shift | OR_j (idx_j & (2^w_j-1)) << s_j.
struct TupleArgs {
  const void* idx[SPTC_MAX_ORDER];
  int shift[SPTC_MAX_ORDER];
  int width[SPTC_MAX_ORDER];
  int n;
  int bytes;               // 4 or 8 (index arrays)
  const uint64_t* prev;    // NULL for the first group
  int prev_shift;
};

// Y's entries by the top bits of their contract value c: tab[c >> sh] =
// {first, end} among the sorted keys.  sh == 0: one contract value per entry.
struct YTable {
  const U2* tab;
  const uint64_t* ykeys;
  uint64_t ny;
  int sh, ynf;
};
// Entries of the table (a power of two) for ny keys of ncbits contract bits:
// one per contract value while that is at most 4 per key (or 2^14 in all, which
// one short fill clears), else up to one per key -- so that a table takes no more
// than 64 bytes per key, and a small Y under a wide field no long fill.
inline int ytable_bits(int ncbits, uint64_t ny, int exact_max = 22) {
  const int fl = ny ? 63 - __builtin_clzll(ny) : 0;
  if (ncbits <= 14 || (ncbits <= exact_max && ncbits <= fl + 2)) return ncbits;
  return ncbits < fl ? ncbits : fl;
}

struct MatchOut {
  // engine form (compacted active X nonzeros and X rows)
  uint64_t* act_prefix;
  uint64_t* act_ypos;
  float* act_xval;
  uint32_t* act_row;
  uint64_t* row_key;
  uint64_t* row_prod;
  uint64_t* row_act;
  // per-phase API form
  uint64_t* mpos;
  uint64_t* mcnt;
  uint64_t* prefix;
};

struct ExpandArgs {
  const uint64_t* act_prefix;
  const uint64_t* act_ypos;
  const float* act_xval;
  const uint32_t* act_row;
  uint64_t A0, A1, P0, P1;
  uint32_t r0;
  const uint64_t* ykeys;
  const float* yvals;
  int ynf;
  uint64_t fmask;
  uint64_t* out_keys;
  float* out_vals;
  // row-segmented sort (launch_expand_items, narrow form): products go out
  // as 32-bit columns, to (big_col, big_val) for big-row tiles and to
  // (out_col32, out_vals) for small-row groups; launch_expand writes 64-bit
  // keys to out_keys
  uint32_t* big_col;
  float* big_val;
  uint32_t* out_col32;
  // column field of every Y key as 32 bits (NULL: taken from ykeys & fmask)
  const uint32_t* ycol;
  uint64_t* hist;
  int passes;
  double* vsum;  // [kSumSlots]
  uint32_t remap;  // XCD-contiguous tile order (set by launch_expand)
  // big-row tiles count the first pass's digits at this column shift
  // (set by launch_expand_items from the plan)
  int dshift = 0;
};

struct DenseArgs {
  const uint64_t* act_prefix;  // [A+1], act_prefix[A] = ir
  const uint64_t* act_ypos;
  const float* act_xval;
  const uint64_t* row_act;     // [R+1]
  uint64_t r0;                 // first row of the chunk
  const uint32_t* ycol;        // [ny] column rank of each Y entry
  const float* yvals;
  const uint64_t* ytab;        // rank -> Y free key (NULL: field is the key)
  uint32_t cols;               // ranks below it
  uint32_t* row_cnt;           // [rows] symbolic counts
  const uint64_t* out_off;     // [rows] output offsets
  uint32_t* out_row;
  uint64_t* out_col;
  float* out_val;
  double* vsum;                // [kSumSlots] sum of the products (may be NULL)
};

constexpr int kDenseMaxBits = 13;  // dense LDS rows up to 8192 slots
// Products per active X nonzero below which ESC is taken.  5e4 rows of 5 owners over
// 1000 columns, dense against ESC: 491 us / 299 with 4 products per owner, 348 / 327
// with 8, 372 / 385 with 16, 400 / 485 with 32.  (5e3 rows: 208 / 250 with 4.)
constexpr uint64_t kDenseMinRun = 16;
// Owners (active X nonzeros) per row up to which dense is chosen.  The line was drawn
// for a pass that added owner by owner, and is not where the two meet now: the same
// rows with 16 products per owner take 372 us / 385 with 5 owners, 416 / 455 with 8,
// 546 / 661 with 16; eight batched instances of 2000 rows with 32 products per owner
// 276 / 243 with 1, 325 / 341 with 5, 588 / 1172 with 64.  Nor does it know the
// columns: over 8000 of them, 2 owners of 400 products, 500 rows take 206 us / 255,
// 5e3 355 / 387, 5e4 1464 / 815.
constexpr uint64_t kDenseMaxOwnersPerRow = 5;
// The automatic choice (single and batched planners alike): dense when its
// rows are dense enough for the slots (ir * 32 >= rows * slots), the Y
// segments long enough and the owners per row few enough.
inline bool dense_pays(uint64_t ir, uint64_t rows, uint64_t active, uint64_t slots) {
  return ir * 32 >= rows * slots && ir >= kDenseMinRun * active &&
         active <= kDenseMaxOwnersPerRow * rows;
}

void launch_dense_count(const DenseArgs& a, int eb, uint64_t rows, hipStream_t s);
void launch_dense_numeric(const DenseArgs& a, int eb, uint64_t rows, hipStream_t s);
// *out (device or pinned host memory) = sum of the kSumSlots slots, added in a
// fixed order.
void launch_fold_sums(const double* slots, double* out, hipStream_t s);
void run_row_count_scan(const uint32_t* cnt, uint64_t* off, uint64_t n, U2* tmp, hipStream_t s,
                        U2* host = nullptr);

void launch_linearize(const LinArgs& a, int idx_bytes, uint64_t n, uint64_t* keys,
                      uint64_t* hist, int passes, int rb, hipStream_t s, int lo = 0);
// Fills and builds the table in tab[0 .. 2^bits - 1] (bits from ytable_bits).  hdup
// (pinned host memory, cleared by the caller; may be NULL) is set when two Y keys are
// equal.
YTable build_ytable(U2* tab, int bits, const uint64_t* ykeys, uint64_t ny, int ncbits, int ynf,
                    hipStream_t s, uint64_t* hdup = nullptr);
// look (may be NULL): scratch of 2 * nx words for what the lookups find; without
// it they run twice.  The per-phase form (api) keeps them in mpos and mcnt.
void run_match(const uint64_t* xkeys, const float* xvals, uint64_t nx, int ncbits,
               const YTable& t, const MatchOut& o, int api, U2* tmp, hipStream_t s,
               U2* host = nullptr, uint64_t* look = nullptr);
// Reduce half of run_match: tmp[scan_tmp_count(nx)] = {ir, A << 32 | R}.
void run_match_count(const uint64_t* xkeys, uint64_t nx, int ncbits, const YTable& t, U2* tmp,
                     hipStream_t s);
void run_exclusive_scan(const uint64_t* in, uint64_t* out, uint64_t n, U2* tmp,
                        hipStream_t s);
void launch_chunk_end(const uint64_t* row_prod, const uint64_t* row_act, uint64_t R,
                      uint64_t r0, uint64_t rmax, uint64_t cap, uint64_t* out,
                      hipStream_t s);
void launch_max_row(const uint64_t* row_prod, uint64_t R, uint64_t* out, hipStream_t s);
void launch_expand(const ExpandArgs& a, int rb, hipStream_t s);
// Reduce counts: tmp holds reduce_tmp_count(n) entries (tile sums, total,
// block partials); the scanned tile sums are the emit's tile offsets.
void run_reduce_count(const uint64_t* keys, uint64_t n, U2* tmp, hipStream_t s);
void run_reduce_emit(const uint64_t* keys, const float* vals, uint64_t n, uint32_t* out_row,
                     uint64_t* out_col, float* out_val, uint64_t r0, int ynf,
                     uint64_t fmask, const uint64_t* ytab, const U2* tmp, hipStream_t s);
// NarrowRows::tile_row for a chunk of rstart[nrows] products: 2 entries per
// wave tile, 2 * (narrow_tile_count(n) + 1) in all.
void launch_tile_rows(const uint64_t* rstart, uint64_t nrows, uint64_t n, uint32_t* tile_row,
                      hipStream_t s);
// Narrow-form count and emit (outputs' rows are r0 + chunk-local row): tmp
// holds narrow_tmp_count(n) entries, the total at tmp[narrow_tile_count(n)];
// columns and values 16-byte aligned.
// scan = false leaves the per-tile counts in tmp unscanned (more counts are
// added to them before scan_narrow_tiles).
void run_reduce_count_narrow(const NarrowRows& nr, uint64_t n, U2* tmp, hipStream_t s,
                             bool scan = true);
void scan_narrow_tiles(uint64_t n, U2* tmp, hipStream_t s);
// ytab32 (may be NULL): the same table as 32-bit words, used when set.
void run_reduce_emit_narrow(const NarrowRows& nr, const float* vals, uint64_t n,
                            uint32_t* out_row, uint64_t* out_col, float* out_val, uint64_t r0,
                            const uint64_t* ytab, const uint32_t* ytab32, const U2* tmp,
                            hipStream_t s);
void launch_yfree_extract(const uint64_t* ykeys, uint64_t ny, uint64_t fmask, uint64_t* out,
                          hipStream_t s);
void run_unique(const uint64_t* sorted, uint64_t n, uint64_t* out, U2* tmp, hipStream_t s,
                U2* host = nullptr);
void launch_tuple_key(const TupleArgs& a, uint64_t n, uint64_t* out, hipStream_t s);
// *out = max(*out, largest of the n indices); *out cleared by the caller.
void launch_mode_max(const void* idx, int bytes, uint64_t n, uint64_t* out, hipStream_t s);
// ycol[i] = ykeys[i] & fmask (a column field of at most 32 bits).
void launch_ycol(const uint64_t* ykeys, uint64_t ny, uint64_t fmask, uint32_t* ycol,
                 hipStream_t s);
void launch_yrank(const uint64_t* ykeys, uint64_t ny, int ynf, uint64_t fmask,
                  const uint64_t* ytab, uint64_t U, int yrb, uint64_t* out, hipStream_t s);
void launch_pack_keys(const uint32_t* row, const uint64_t* col, const uint64_t* row_key,
                      uint64_t n, int ynf, uint64_t* out, hipStream_t s);
void launch_gather_rowkey(const uint32_t* row, const uint64_t* row_key, uint64_t n,
                          uint64_t* out, hipStream_t s);

}  // namespace sptc
