// Compiled to LLVM IR only (tests/test_tile_lds_order.py): the LDS exchanges
// between the lanes of one wavefront in the matrix tile path, twice over, so
// that both directions (a tile's words written then read by other lanes, and
// read before the next tile's are written) are in the listing.
#include "paged_decode_mfma.h"

namespace xhip {

template <int KV, int D> __device__ __forceinline__ void v_tiles(const u32x4 *in, u32x4 *out) {
    using G = MfmaGeometry<KV, D>;
    static_assert(G::kVStaged, "a head size whose V tile passes through LDS");
    __shared__ MfmaVLds<KV, D> vs;
    const int lane = threadIdx.x;
#pragma unroll
    for (int t = 0; t < 2; t++) {
        MfmaTileRegs<KV, D> r;
#pragma unroll
        for (int c = 0; c < G::kVLoads; c++) r.v[c] = in[(t * G::kVLoads + c) * 64 + lane];
        vs.put(r, lane);
        for_groups<KV, D>([&](auto b) {
            constexpr int B = decltype(b)::value;
            u32x4 v[4];
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = vs.template chunk<B>(r, lane, i);
#pragma unroll
            for (int i = 0; i < 4; i++) out[((t * 4 + B) * 4 + i) * 64 + lane] = v[i];
        });
    }
}

#define V_TILES(KV, D)                                                                    \
    extern "C" __global__ void __launch_bounds__(64)                                      \
        v_tiles_##KV##_##D(const u32x4 *__restrict__ in, u32x4 *__restrict__ out) {       \
        v_tiles<KV, D>(in, out);                                                          \
    }
V_TILES(KV_F16, 32)
V_TILES(KV_F16, 64)
V_TILES(KV_F16, 80)
V_TILES(KV_BF16, 96)
V_TILES(KV_BF16, 112)
V_TILES(KV_F32, 32)

// The members of a prefix piece's query rows (mfma_load_q, kSrcPrefix).
extern "C" __global__ void __launch_bounds__(64)
    prefix_members(const DecodeParams p, const MfmaPiece a, const MfmaPiece b,
                   const CascadeLdsPlan plan, u32x4 *out) {
    __shared__ int win[2 * kMfmaHeads];
    CascadeLdsPlan cp = plan;
    cp.win = win;
    u32x4 q[2][MfmaGeometry<KV_F16, 32>::kQkSteps];
    for (int t = 0; t < 2; t++) {
        mfma_load_q<KV_F16, 32, 2, kSrcPrefix>(p, t ? b : a, threadIdx.x, q, &cp);
        out[(2 * t) * 64 + threadIdx.x] = q[0][0];
        out[(2 * t + 1) * 64 + threadIdx.x] = q[1][0];
    }
}

}  // namespace xhip
