// Compiled for its assertions only (tests/test_tile_lds_order.py): the LDS of
// the cascade's partition launch, whose in-kernel plan needs two workgroups
// on a CU's 160 KB.
#include "paged_decode_cascade_attn.h"

namespace xhip {

// dynamic LDS left to the plan of either of two workgroups
template <int KV, int D, int RS> constexpr long long plan_room() {
    return (160 * 1024) / 2 - (long long)sizeof(MfmaLdsPair<KV, D, RS>) -
           (long long)sizeof(int) * kMfmaWavesPerGroup * (1 + 2 * kMfmaHeads);
}

// 1024 sequences of a group of 64 query heads (one prefix-batch sequence per
// member), 1500 of a group of 32, in 16 groups; 1024 of a group of 16 in 256
constexpr long long plan_bytes(long long B, long long group, long long NG) {
    return 4 * inplan_lds_ints(B, (B * group + 63) / 64 + NG, NG);
}
template <int KV, int D> constexpr bool fits() {
    return plan_bytes(1024, 64, 16) <= plan_room<KV, D, 2>() &&
           plan_bytes(1500, 32, 16) <= plan_room<KV, D, 2>() &&
           plan_bytes(1024, 16, 256) <= plan_room<KV, D, 1>();
}
static_assert(fits<KV_F16, 128>() && fits<KV_BF16, 128>(), "head_size 128");
static_assert(fits<KV_F16, 96>() && fits<KV_BF16, 96>(), "head_size 96");
static_assert(fits<KV_F16, 64>() && fits<KV_F16, 32>(), "head_sizes 64 and 32");

}  // namespace xhip
