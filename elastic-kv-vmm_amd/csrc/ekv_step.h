// Launches that the one-call decode step shares with the entry points it is made of.
#pragma once

#include "../../include/ekv_kernels.h"

namespace ekv {

// The step's lookup and swap-in in one launch (swap_in.hip); false, with nothing launched, when the tensors' layouts
// need the separate kernels. The arguments are those both entry points have accepted (checked by the caller).
bool lookup_swap_in(const ekv_step_args& s, const ekv_tensor& misses, const ekv_tensor& counts, const ekv_tensor& src,
                    const ekv_tensor& dst, void* stream);

// ekv_move_kv over the lists of the batch rows that `selected` names (gather.hip): entries outside the batch move
// nothing, and the counts of rows it does not name are not read.
void move_selected(const ekv_planes* src, const ekv_tensor* src_rows, const ekv_planes* dst, const ekv_tensor* dst_rows,
                   const ekv_tensor* counts, const ekv_tensor* selected, int64_t zero_below, void* stream);

}  // namespace ekv
