// Row accumulator (rowacc.hip): the products of a chunk of X rows summed into
// its outputs without ever being written to HBM.
#pragma once
#include "kernels.hpp"

namespace sptc {

// Column ranks per slab of a long row: the slab's LDS bitmap is 8 KiB and a
// column's offset in it fits 16 bits.
constexpr int kSlabBits = 16;
constexpr uint32_t kSlabCols = 1u << kSlabBits;
// Column spaces up to this many bits (16 slabs) are cut into slabs; over wider
// ones the row accumulator takes chunks without long rows, and the product sort,
// whose cost does not grow with the columns, the others.
constexpr int kRowAccMaxBits = 20;

// Products of a group of short rows (one workgroup's LDS sort) and the most
// a short row may hold: a group starts at the first row past a multiple of
// half a tile.
constexpr int kGroupNT = 512;
constexpr int kGroupIPT = 6;
constexpr uint32_t kGroupTile = kGroupNT * kGroupIPT;
constexpr uint32_t kGroupHalf = kGroupTile / 2;

// A chunk's operands and tables.  Rows are the global X rows [r0, r0 + rows).
struct RowAccArgs {
  const uint64_t* act_prefix;  // [A + 1]
  const uint64_t* act_ypos;    // [A]
  const float* act_xval;       // [A]
  const uint64_t* row_prod;    // [R + 1]
  const uint64_t* row_act;     // [R + 1]
  const uint32_t* act_row;     // [A]
  uint64_t a0;                 // the chunk's first active X nonzero
  uint64_t r0, rows;
  uint64_t ny;
  const uint32_t* ycol;        // [ny] column rank of each Y entry
  const float* yvals;          // [ny]
  const uint64_t* ykeys;       // [ny] Y keys, free field in the low bits
  uint64_t yfmask;             // its mask
  const uint32_t* yfree32;     // [ny] the free field as 32 bits (NULL: wider)
  const uint64_t* ytab;        // rank -> Y free key (NULL: the rank is the key)
  const uint32_t* ytab32;      // the same as 32 bits (NULL: wider)
  uint32_t K;                  // column ranks below K
  uint32_t short_max;          // rows of several owners up to this many products are short
  bool ydup;                   // Y holds duplicate coordinates
  double* vsum;                // [kSumSlots]
};

// The chunk's rows by kind and its output offsets.  Every row with products is
// "live" (k counts them); a row of one owner is copied from its Y segment, a
// short row of several owners is sorted in a group, the others ("long") are
// summed slab by slab.
constexpr uint64_t kItemBytes = 32, kNearBytes = 24;
struct RowAccPlan {
  // most rows with products and most products of the call's chunks (0: unknown)
  uint64_t rows_at_most = 0, prods_at_most = 0;
  uint64_t live = 0, nshort = 0, nlong = 0;  // rows
  uint64_t short_prods = 0;
  uint64_t items = 0;                        // long rows' slabs (after count)
  uint64_t outs = 0, near_outs = 0;          // outputs, and those of rows that are not long
  uint64_t near_rows = 0;
  DevBuf<uint32_t> live_row, live_cnt;       // [live] chunk-local row, outputs
  DevBuf<uint64_t> live_src;                 // [live] where its outputs come from
  DevBuf<uint32_t> s_live, s_prod;           // [nshort] live index; products before
  DevBuf<uint32_t> l_live;                   // [nlong] live index
  DevBuf<uint32_t> l_near;                   // [live] near outputs before a long row
  DevBuf<uint64_t> l_item, l_split;          // [nlong + 1], [nlong] slabs, split entries before
  DevBuf<uint32_t> quant;                    // slab bounds (of the call's Y)
  DevBuf<uint32_t> l_word;                   // [nlong] bitmap words before
  DevBuf<uint32_t> item;                     // [items] descriptors of kItemBytes
  DevBuf<uint32_t> item_cnt;                 // [items] outputs
  DevBuf<uint64_t> item_off;                 // [items] first output
  DevBuf<uint64_t> words;                    // the items' bitmaps, when kept
  bool keep_words = false;
  DevBuf<uint32_t> split;                    // slab bounds of every owner of a long row
  DevBuf<uint32_t> near_pre;                 // [near_rows] outputs of near rows before
  DevBuf<uint64_t> near;                     // [near_rows] descriptors of kNearBytes
  DevBuf<uint32_t> tcol;                     // [short_prods] a group's outputs, compacted
  DevBuf<float> tval;
  DevBuf<U2> tmp;
};

// Classifies the rows and counts every row's outputs (plan->outs); host
// receives three U2 of pinned memory.  One wait for the row kinds, one for the
// counts.  count_only: the groups' outputs are not kept and the value sum is
// taken here.  nprod and owners: the chunk's products and active X nonzeros.
// False, with nothing done, when a row is too heavy for one workgroup an item
// or a long row meets a column space wider than kRowAccMaxBits.
bool rowacc_count(const RowAccArgs& a, uint64_t nprod, uint64_t owners, bool count_only,
                  RowAccPlan* plan, U2* host, hipStream_t s, KTimer* kt);
// Bytes a plan holds at most, for K column ranks.
uint64_t rowacc_bytes(uint64_t rows, uint64_t owners, uint64_t nprod, uint64_t K);
// Writes the outputs (plan->outs entries, in (row, column) order).
void rowacc_emit(const RowAccArgs& a, RowAccPlan& plan, uint64_t nprod, uint32_t* out_row,
                 uint64_t* out_col, float* out_val, hipStream_t s, KTimer* kt);

}  // namespace sptc
