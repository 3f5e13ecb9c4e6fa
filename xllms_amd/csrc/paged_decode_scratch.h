// Fixed device scratch of nxt_paged_attention_noalloc (paged_decode_scratch.hip).
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>

namespace xhip {

// Bytes of split-K partials and unit prefix that a plan may need, 66 MiB.
// Every automatic plan fits on a 256-CU MI355X: the MFMA path's 2048
// wavefronts need at most 64 MiB of partials (2 slots x 32 heads x 128 dims x
// 4 B each; head tiles of 16 half of that, with 1024 wavefronts for rows of
// more than 256 bytes, and 16 MiB for the 4096 at head_size 32) plus 1 MiB of
// (m, l) pairs and the unit prefix; the VALU path's head tiles of up to 8
// heads run at most 2048 wavefronts for 8 heads (32 MiB at 256 dims), 4096
// for 4 and 8192 for fewer.  A plan that needs more (an explicit
// partition_tokens, or a larger device) is refused.
constexpr size_t kNoAllocScratchBytes = (size_t)66 << 20;

// What the kernels keep behind a plan's unit prefix (its units per
// wavefront): in the array, beside the plan's bytes.
constexpr size_t kNoAllocScratchTail = 256;

// This device's scratch address (looked up once per device, with it
// current) and size.  Allocates nothing.
hipError_t noalloc_scratch(int device, void **ptr, size_t *bytes);

}  // namespace xhip
