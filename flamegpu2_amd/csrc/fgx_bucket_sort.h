// Stable bin sort through LDS (fgx_bucket_sort.hip): used by the message-list build, the
// bucket index and the agent sort where bucket_plan() accepts the sizes.
#pragma once

#include "fgx_keys.h"

namespace fgx {

struct BucketPlan {
    uint32_t one_block;   // the whole list is sorted by one block
    uint32_t threads;     // 256 or 1024 per block
    uint32_t items;       // list elements per thread of a tile
    uint32_t shift;       // bucket = key >> shift
    uint32_t buckets;
    uint32_t tiles;
    uint32_t piece_log;   // elements of a piece of an oversize bucket: 1 << piece_log
    uint32_t rows;        // words of bin counts of such pieces
};

// Whether n_cap elements over `bins` keys (of which about `used` occur) take this sort, and
// how it is split.  Depends on the sizes only.
bool bucket_plan(uint32_t n_cap, uint32_t bins, uint64_t used, BucketPlan* p);

// The sort.  `words_a`, `words_b`, `words_c`: n_cap words of scratch each.  start_out: the
// bins + 1 bin starts, or NULL when nobody reads them.
int bucket_sort(const BucketPlan& p, const KeyArgs& ka, uint32_t bins, const uint32_t* d_n, uint32_t n_cap, const float* x,
                const float* y, const float* z, const VarTable& vt, uint32_t* start_out, uint32_t* words_a,
                uint32_t* words_b, uint32_t* words_c, hipStream_t st);

}  // namespace fgx
