// Prefill launches whose items are split over the kv range (prefill_split.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace pa {

struct PrefillParams;

// Workspace bytes of a split launch of this shape at head size 128; 0: the
// shape is not one that splits.  span: tokens a block-table row can hold.
size_t prefill_split_bytes(int32_t batch, int32_t n_qtiles, int32_t num_kv_heads, int64_t span);

// Whether a launch of `p` (head size 128) has few enough, long enough items for
// a split to pay.
bool prefill_splits(const PrefillParams& p);

// Split launch of `p` (head size 128, bf16 pages) with a workspace of
// prefill_split_bytes, zero rows included.  Returns a PA_* code.
int prefill_split_launch(const char* name, const PrefillParams& p, int paging, void* workspace, hipStream_t s);

}  // namespace pa
