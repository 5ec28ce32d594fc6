// Token positions named by Top-K block ids.
#pragma once

#include "ekv_fastdiv.h"   // EKV_HD

#include <cstdint>

namespace ekv {

// Position of token `offset` of block `id`, and whether it lies below `bound`
// (at most `cols`, the positions of the table; cols, block_size and offset
// are below 2^31). An int64 id is compared with `cols` before it is
// multiplied: a block starts at or past its own id, so one that is not below
// cols names no position, and id * block_size of a large one (INT64_MAX as
// padding) would wrap to a position that looks valid. int32 ids cannot wrap.
// `position` is below 2^62 and, where the result is true, in [0, bound).
template <typename Id>
EKV_HD inline bool token_position(Id id, uint32_t block_size, uint32_t offset, int64_t cols, int64_t bound,
                                  int64_t& position) {
    if (sizeof(Id) == 4) {
        position = static_cast<int64_t>(id) * block_size + offset;
        return id >= 0 && position < bound;
    }
    const bool inside = static_cast<uint64_t>(id) < static_cast<uint64_t>(cols);
    position = static_cast<int64_t>(inside ? id : 0) * block_size + offset;
    return inside && position < bound;
}

}  // namespace ekv
