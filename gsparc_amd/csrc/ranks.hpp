// Column ranks: Y's free keys replaced by their rank among the distinct ones
// (ranks.hip).
#pragma once
#include "kernels.hpp"

namespace sptc {

// Outputs of a rank compression of ny Y keys with free fields of ynf bits.
struct RankOut {
  uint64_t* ytab;     // [distinct] rank -> free key
  uint32_t* ytab32;   // the same as 32-bit words (NULL: ynf > 32)
  uint32_t* ycol;     // [ny] rank of each Y entry
  uint32_t* yfree32;  // [ny] its free key as 32 bits (NULL: ynf > 32)
};

// True when the ranks are taken from a map of the free field (a byte for each of
// its 2^ynf values) rather than from a sort of the free keys.
bool rank_by_map(uint64_t ny, int ynf);
inline uint64_t rank_words(int ynf) { return ynf <= 5 ? 1 : 1ull << (ynf - 5); }
// Bytes of scratch: the map, its bits and their ranks.
inline uint64_t rank_map_bytes(int ynf) { return 40 * rank_words(ynf); }
// map: rank_map_bytes(ynf) bytes, 16-byte aligned; tmp as for a scan of
// rank_words(ynf) items.  *host (pinned) receives the distinct count.
void run_rank_map(const uint64_t* ykeys, uint64_t ny, int ynf, const RankOut& o, uint8_t* map,
                  U2* tmp, U2* host, hipStream_t s);
// From the sorted free keys: distinct ones (tmp as for a scan of ny items; the
// count stays on the device, *host receives it too), then a search per entry.
void run_rank_sorted(const uint64_t* sorted, const uint64_t* ykeys, uint64_t ny, int ynf,
                     const RankOut& o, U2* tmp, U2* host, hipStream_t s);

}  // namespace sptc
