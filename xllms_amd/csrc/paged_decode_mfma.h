// MFMA tile path of the paged-decode attention (block_size >= 16; fp16 / bf16
// K/V at head sizes that are multiples of 32, and in automatic plans at 80 and
// 112 and fp32 up to head_size 128).  One wavefront serves R row blocks of 16
// query heads of one kv head (R = 1, or 2 for groups of 17-32 heads at
// head_size <= 128): every K/V tile it loads is used by all 16R heads.
// Below, one row block; with R = 2 the QK^T MFMAs run once per block on the
// same K registers, and each V^T operand feeds both blocks' PV MFMAs.
//
// Per 16-token tile (one page when block_size = 16), with g = lane/16 and
// j = lane%16 (v_mfma_f32_16x16x{32,16} operand layouts, checked on gfx950):
//   QK^T  S[token][head] = sum_d K[token][d] Q[head][d]
//         D/32 x v_mfma_f32_16x16x32: A = K rows (lane: row j, dims
//         32c+8g..+7, a 16-byte load straight from the page), B = Q of the 16
//         heads (lane: head j, same dims).  C: lane holds rows 4g+r of head j.
//         Row 4g+r is token tile_token(g, r) = 4r+g.
//   softmax per head j: the 16 scores of head j sit in lanes j, j+16, j+32,
//         j+48 (4 each): in-lane max, two xor shuffles, exp2, running sum.
//   PV    O^T[dim][head] += sum_t V[t][dim] P[head][t]
//         v_mfma_f32_16x16x16 per dim block (twice: P = P_hi + P_lo in the
//         16-bit type, so the product keeps ~22 bits of P over fp16 and ~16
//         over bf16, of a result with 11 and 8): B = P, which is
//         exactly the C layout of the QK^T step (lane: head j, rows
//         4g..4g+3); A = V^T (lane: one dim per block, the same four tokens).
//         Which dim a lane holds in which block is free, so lane (g, j) loads
//         chunk j of each of its own four token rows (16 bytes at
//         head_size 128; the row in 16 equal chunks below that, and in groups
//         of 16 above), and the dims of a chunk become row j of as many
//         blocks.  V goes from the load registers to the MFMA with two
//         v_perm_b32 per block (one half of each of four rows), and C (lane:
//         O^T rows 4g+r of head j) holds a chunk's consecutive dims over the
//         blocks of its group: whole output chunks.
//         A trip of the tile through LDS instead (row-major write, 32
//         two-byte reads a lane to gather V^T) was 40 LDS instructions and a
//         write-to-read wait in every tile's chain; fp16, head_size 128,
//         16 x 1024 tokens, 32 / 8 heads: 21.3 -> 20.7 us a step.
// fp32: v_mfma_f32_16x16x4 for both products, 16-byte chunks of 4 dims on
// either side: QK^T step (c, i) multiplies element i of the K and Q chunks at
// byte 64c + 16g, PV step r element e of the chunk of row 4g + r with P's row
// 4g + r, so neither operand needs a permutation.
// fp16 / bf16 at head sizes 80 and 112 (kP32): PV as for fp32, on V's elements
// converted as they leave the chunk.
// Loads are buffer loads: a token past the end of the range, or in a page
// with a negative id, gets an out-of-range offset and reads as zero without
// touching memory; its score is masked to -inf.  The next tile's K/V loads
// are issued before the current tile is computed.
#pragma once

#include <type_traits>

#include "paged_decode_kernels.h"
#include "wg_trace.h"

namespace xhip {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));

constexpr uint32_t kOobOffset = 0x80000000u;

template <int KV, int D> struct MfmaGeometry {
    static constexpr int kTile = 16;  // tokens per tile
    static constexpr int kElemBytes = KvTraits<KV>::kBytes;
    static constexpr int kRowBytes = kElemBytes * D;
    static constexpr int kQkSteps = (kRowBytes + 63) / 64;  // 16-byte K loads per lane
    // V rows: groups of 16 chunks, a lane holding one chunk of each group (of
    // its four token rows); full groups have kDims dims (16 bytes) per chunk,
    // the last one as many as the row still has.  An odd count of 16-bit dims
    // (head sizes 80, 112) is padded: whole chunks, of which the last lanes'
    // lie past the row (kPadded; their rows of the blocks are never used).
    static constexpr int kDims = 16 / kElemBytes;
    static constexpr int kVGroups = (D + 16 * kDims - 1) / (16 * kDims);
    static constexpr int group_dims(int b) {
        const int r = (D - 16 * kDims * b) / 16;
        return r >= kDims || (kElemBytes == 2 && r % 2) ? kDims : r;
    }
    static constexpr bool kPadded = kElemBytes == 2 && (D / 16) % 2 != 0;
    // P in fp32 (v_mfma_f32_16x16x4 for PV): fp32 K/V, and the 16-bit head
    // sizes whose explicit plans run the VALU tiles (80, 112), where P is fp32
    // too: two 16-bit parts are ~22 bits of P for fp16, 16 for bf16, and a V
    // of infinity times a part that is 0 is NaN.
    static constexpr bool kP32 = KV == KV_F32 || kPadded;
    // Its MFMAs of four tokens per chain of a tile's sum.  fp32 results hold
    // the rounding of that sum, and chains of 16 tokens left short contexts
    // further from 64 bits than the VALU tiles, which add up 4 to 8 rows' sums
    // (16 tokens: head_size 64 1.18e-7 against 1.13e-7, 128 1.23e-7 against
    // 1.19e-7).  Two chains of 8: 1.09e-7 and 1.15e-7, and 1.86e-7 against
    // 2.05e-7 at 2000 tokens, for 0.7% of the step of 32 sequences of up to
    // 2048 tokens at 32 / 8 heads, 1-3% at more heads.  Four of 4 (3% more)
    // where the VALU tiles add up the most rows, head_size 32: 1.09e-7 against
    // 1.11e-7; chains of 16 had 1.19e-7.  16-bit results show none of this.
    static constexpr int kPvChain = KV != KV_F32 ? 4 : kRowBytes < 256 ? 1 : 2;
    static constexpr int group_words(int b) { return group_dims(b) * kElemBytes / 4; }
    static constexpr int kDimBlocks = kDims * (kVGroups - 1) + group_dims(kVGroups - 1);
    // Rows of fewer than 16 chunks of 16 bytes: the tile is loaded in whole
    // 16-byte lanes and dealt to the lane chunks through LDS (4- to 12-byte
    // loads, one per token row, are slower: head_size 32, bf16, 64 sequences
    // of 256-4096 tokens, 32 / 8 heads 39.4 us a step).
    static constexpr bool kVStaged = kRowBytes < 256;
    static constexpr int kVLoads = kVStaged ? (kRowBytes + 63) / 64 : 4 * kVGroups;
    static_assert(D % 16 == 0 && (!kPadded || kVStaged), "head sizes of the MFMA path");
};

// First of the group_dims(b) dims of chunk i of V group b: element e of the
// chunk is row i of dim block kDims * b + e.
template <int KV, int D> __device__ __forceinline__ int mfma_dim(int b, int i) {
    using G = MfmaGeometry<KV, D>;
    return 16 * G::kDims * b + G::group_dims(b) * i;
}

template <int KV> __device__ __forceinline__ f32x4 mfma_qk(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (KV == KV_F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                      __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

template <int KV> __device__ __forceinline__ f32x4 mfma_pv(u32x2 a, u32x2 b, f32x4 c) {
    if constexpr (KV == KV_F16)
        return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a),
                                                     __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(i16x4, a),
                                                         __builtin_bit_cast(i16x4, b), c, 0, 0, 0);
}

// 16x16x4 (A lane: row j, k = g; B lane: column j, k = g).
__device__ __forceinline__ f32x4 mfma_f32(uint32_t a, uint32_t b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, a),
                                                __builtin_bit_cast(float, b), c, 0, 0, 0);
}

// Element e of a chunk, in fp32.
template <int KV> __device__ __forceinline__ uint32_t chunk_elem(u32x4 v, int e) {
    if constexpr (KV == KV_F32) {
        return lane_word(v, e);
    } else {
        const f32x2 x = unpack16<KV>(lane_word(v, e / 2));
        return __builtin_bit_cast(uint32_t, e & 1 ? x.y : x.x);
    }
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const char *base) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, 0x7FFFFFFF, 0x00020000);
}

// K/V pages are streamed once per launch: nontemporal loads (cache policy
// `nt`).  On MI355X they raise the read rate of this access pattern (random
// 4 KB runs, 16-byte lane loads) from ~5.9 to ~6.6 TB/s.
constexpr int kStreamPolicy = 2;

// A chunk of W words (1 to 4; the rest of the vector is unspecified).
template <int W, int POLICY>
__device__ __forceinline__ u32x4 buf_load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    u32x4 x;
    if constexpr (W == 4) {
        x = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, POLICY);
    } else if constexpr (W == 3) {
        const u32x3 y = __builtin_amdgcn_raw_buffer_load_b96(r, (int)off, 0, POLICY);
        x = __builtin_shufflevector(y, y, 0, 1, 2, -1);
    } else if constexpr (W == 2) {
        const u32x2 y = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, POLICY);
        x = __builtin_shufflevector(y, y, 0, 1, -1, -1);
    } else {
        x.x = __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, POLICY);
    }
    return x;
}

// fn(std::integral_constant<int, b>) for every V group b (their widths differ).
template <int KV, int D, typename Fn> __device__ __forceinline__ void for_groups(Fn &&fn) {
    constexpr int N = MfmaGeometry<KV, D>::kVGroups;
    static_assert(N >= 1 && N <= 4, "V groups of a row");
    fn(std::integral_constant<int, 0>{});
    if constexpr (N > 1) fn(std::integral_constant<int, 1>{});
    if constexpr (N > 2) fn(std::integral_constant<int, 2>{});
    if constexpr (N > 3) fn(std::integral_constant<int, 3>{});
}

template <int KV, int D> struct MfmaTileRegs {
    u32x4 k[MfmaGeometry<KV, D>::kQkSteps];     // score row j, 16 bytes at 64c + 16g of the K row
    u32x4 v[MfmaGeometry<KV, D>::kVLoads];      // 4b + r: score row 4g + r, chunk j of V group b;
                                                // staged: bytes 1024c + 16 * lane of the V tile
};

// Token, within its tile, of score row 4g + r.  Lane group g holds V rows
// tile_token(g, 0..3), one per load, so a load covers the four neighbouring
// rows 4r..4r+3.  (With rows 4g + r, 4 apart in a load, the pieces of a row
// that is not whole 128-byte lines were fetched twice: head_size 96, 24
// sequences of 100-2000 tokens, 32 / 32 heads 60.1 us against 57.)
__device__ __forceinline__ int tile_token(int g, int r) { return 4 * r + g; }

template <int KV, int D, int POLICY>
__device__ __forceinline__ void mfma_issue_loads(__amdgpu_buffer_rsrc_t rk,
                                                 __amdgpu_buffer_rsrc_t rv, int n, int lane,
                                                 MfmaTileRegs<KV, D> &r) {
    using G = MfmaGeometry<KV, D>;
    constexpr int RB = G::kRowBytes;
    const int j = lane & 15, g = lane >> 4;
    const int kt = tile_token(j >> 2, j & 3);
    const bool krow_ok = kt < n;
#pragma unroll
    for (int c = 0; c < G::kQkSteps; c++)
        r.k[c] = buf_load<4, POLICY>(rk, krow_ok && (RB % 64 == 0 || 64 * c + 16 * g < RB)
                                             ? (uint32_t)(kt * RB + 64 * c + 16 * g)
                                             : kOobOffset);
    if constexpr (G::kVStaged) {
#pragma unroll
        for (int c = 0; c < G::kVLoads; c++) {
            const int at = 1024 * c + 16 * lane;
            r.v[c] = buf_load<4, POLICY>(rv, at < min(n, G::kTile) * RB ? (uint32_t)at : kOobOffset);
        }
    } else {
        for_groups<KV, D>([&](auto b) {
            constexpr int B = decltype(b)::value;
            constexpr int W = G::group_words(B);
#pragma unroll
            for (int i = 0; i < 4; i++)
                r.v[4 * B + i] = buf_load<W, POLICY>(
                    rv, tile_token(g, i) < n
                            ? (uint32_t)(tile_token(g, i) * RB + 256 * B + 4 * W * j)
                            : kOobOffset);
        });
    }
}

// Issue the K and V loads of the tile starting at token t0 (block id blk):
// rows past t_end or in a negative page read as zero.
template <int KV, int D>
__device__ __forceinline__ void mfma_load_tile(const DecodeParams &p, const char *kb,
                                               const char *vb, int t0, int t_end, int blk,
                                               int lane, bool cached, MfmaTileRegs<KV, D> &r) {
    constexpr int EB = MfmaGeometry<KV, D>::kElemBytes;
    const int bmask = p.block_size - 1;
    const long long page = (long long)blk * p.kv_block_stride + (long long)(t0 & bmask) * D;
    const __amdgpu_buffer_rsrc_t rk = tile_rsrc(kb + page * EB);
    const __amdgpu_buffer_rsrc_t rv = tile_rsrc(vb + page * EB);
    const int n = blk >= 0 ? t_end - t0 : 0;  // tokens of the tile
    if (cached)
        mfma_issue_loads<KV, D, 0>(rk, rv, n, lane, r);
    else
        mfma_issue_loads<KV, D, kStreamPolicy>(rk, rv, n, lane, r);
}

// Running state of one wavefront over one segment: lane (g, j) owns head j.
template <int KV, int D> struct MfmaState {
    f32x4 o[MfmaGeometry<KV, D>::kDimBlocks];  // block kDims*b + e, row 4g + r of
                                               // head j: dim mfma_dim(b, 4g + r) + e
    float m;                               // running max of head j (log2 units)
    float l;                               // this lane's part of the running sum
};

// A piece's query rows (MFMA B layout): in registers, or, where R = 2 states
// leave no room for them beside two tiles of K/V (head_size 128: 10 VGPRs
// spilled, and 64 / 2 heads over 64 sequences of 512-8192 tokens took 76.7 us
// against 67.0), parked by each lane in LDS and read back every tile.  At
// head_size 96 they fit, and LDS is the slower place (64 / 2 heads, 32
// sequences of 650-2592 tokens 25.5 us against 22.3).
template <int KV, int D, int R> constexpr bool mfma_q_in_lds() {
    return R == 2 && MfmaGeometry<KV, D>::kRowBytes > 192;
}
template <int KV, int D, int R, bool LDS = mfma_q_in_lds<KV, D, R>()> struct MfmaQLds {};
template <int KV, int D, int R> struct MfmaQLds<KV, D, R, true> {
    u32x4 q[R][MfmaGeometry<KV, D>::kQkSteps][64];
};

// Between LDS accesses of different lanes of one wavefront.  The wavefront's
// LDS accesses complete in order, so there is nothing to wait for; but the
// compiler orders two accesses only where one lane's addresses may meet, and
// a word that another lane wrote never does.  (No instruction at this scope.)
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
}

// The V tile of a wavefront where it is staged (MfmaGeometry::kVStaged), row-major.
template <int KV, int D, bool STAGED = MfmaGeometry<KV, D>::kVStaged> struct MfmaVLds {
    __device__ __forceinline__ void put(const MfmaTileRegs<KV, D> &, int) {}
    // chunk j of V group B of the lane's score row 4g + i
    template <int B>
    __device__ __forceinline__ u32x4 chunk(const MfmaTileRegs<KV, D> &r, int, int i) const {
        return r.v[4 * B + i];
    }
};
template <int KV, int D> struct MfmaVLds<KV, D, true> {
    u32x4 t[64 * MfmaGeometry<KV, D>::kVLoads];
    __device__ __forceinline__ void put(const MfmaTileRegs<KV, D> &r, int lane) {
        wave_lds_fence();  // after the last tile's chunks
#pragma unroll
        for (int c = 0; c < MfmaGeometry<KV, D>::kVLoads; c++) t[64 * c + lane] = r.v[c];
        wave_lds_fence();  // before this tile's
    }
    template <int B>
    __device__ __forceinline__ u32x4 chunk(const MfmaTileRegs<KV, D> &, int lane, int i) const {
        using G = MfmaGeometry<KV, D>;
        constexpr int W = G::group_words(B);
        const uint32_t *src = (const uint32_t *)t +
                              tile_token(lane >> 4, i) * (G::kRowBytes / 4) + W * (lane & 15);
        u32x4 x;
        if constexpr (W == 4) {
            x = *(const u32x4 *)src;
        } else if constexpr (W == 2) {
            const u32x2 y = *(const u32x2 *)src;
            x = __builtin_shufflevector(y, y, 0, 1, -1, -1);
        } else {
#pragma unroll
            for (int w = 0; w < W; w++) x[w] = src[w];
        }
        return x;
    }
};

template <int KV, int D, int R, bool LDS = mfma_q_in_lds<KV, D, R>()> struct MfmaQuery {
    u32x4 q[R][MfmaGeometry<KV, D>::kQkSteps];
    __device__ __forceinline__ void put(MfmaQLds<KV, D, R> &, int,
                                        const u32x4 (&x)[R][MfmaGeometry<KV, D>::kQkSteps]) {
#pragma unroll
        for (int b = 0; b < R; b++)
#pragma unroll
            for (int c = 0; c < MfmaGeometry<KV, D>::kQkSteps; c++) q[b][c] = x[b][c];
    }
    __device__ __forceinline__ u32x4 get(const MfmaQLds<KV, D, R> &, int, int b, int c) const {
        return q[b][c];
    }
};
template <int KV, int D, int R> struct MfmaQuery<KV, D, R, true> {
    __device__ __forceinline__ void put(MfmaQLds<KV, D, R> &s, int lane,
                                        const u32x4 (&x)[R][MfmaGeometry<KV, D>::kQkSteps]) {
#pragma unroll
        for (int b = 0; b < R; b++)
#pragma unroll
            for (int c = 0; c < MfmaGeometry<KV, D>::kQkSteps; c++) s.q[b][c][lane] = x[b][c];
    }
    __device__ __forceinline__ u32x4 get(const MfmaQLds<KV, D, R> &s, int lane, int b, int c) const {
        return s.q[b][c][lane];
    }
};

template <int KV, int D, int R>
__device__ __forceinline__ void mfma_tile(const DecodeParams &p, const MfmaQuery<KV, D, R> &q,
                                          int t0, int t_end, bool page_ok, int lane,
                                          const MfmaQLds<KV, D, R> &qs, MfmaVLds<KV, D> &vs,
                                          const MfmaTileRegs<KV, D> &r, MfmaState<KV, D> (&st)[R]) {
    using G = MfmaGeometry<KV, D>;
    const int g = lane >> 4;
    vs.put(r, lane);

    // S = K Q^T for 16 tokens x 16 heads, per row block.
    f32x4 s[R];
    if constexpr (KV == KV_F32) {
        // A sum per chunk and element of a chunk (four products), added up as a
        // tree: chains of D / 16 MFMAs carried more rounding into the scores
        // than the VALU tile's sums over lanes do (error against 64 bits,
        // 64 / 8 heads, head_size 128: VALU 2.2e-7, sums of two chunks 1.9e-7,
        // of one 1.8e-7 with the exponent below).  The matrix cores wait for HBM
        // here: the adds cost little (the 32-sequence batch of 256-2048 tokens,
        // 32 / 8 heads: 56.9-57.4 us a step before, 57.3-58.0 after; VALU 63.4).
        static_assert(R == 1, "fp32 tiles have one row block");
        f32x4 part[G::kQkSteps];
#pragma unroll
        for (int c = 0; c < G::kQkSteps; c++) {
            const u32x4 qc = q.get(qs, lane, 0, c);
            f32x4 x[4];
#pragma unroll
            for (int i = 0; i < 4; i++)
                x[i] = mfma_f32(lane_word(r.k[c], i), lane_word(qc, i), f32x4{0.0f, 0.0f, 0.0f, 0.0f});
            part[c] = (x[0] + x[1]) + (x[2] + x[3]);
        }
#pragma unroll
        for (int w = 1; w < G::kQkSteps; w <<= 1)
#pragma unroll
            for (int c = 0; c + w < G::kQkSteps; c += 2 * w) part[c] += part[c + w];
        s[0] = part[0];
    } else {
#pragma unroll
        for (int b = 0; b < R; b++) s[b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < G::kQkSteps; c++)
#pragma unroll
            for (int b = 0; b < R; b++) s[b] = mfma_qk<KV>(r.k[c], q.get(qs, lane, b, c), s[b]);
    }

    bool ok[4];
#pragma unroll
    for (int i = 0; i < 4; i++) ok[i] = page_ok && (t0 + tile_token(g, i) < t_end);

    // Online softmax of head j over the four tokens of this lane; P in the
    // 16-bit type as hi + lo parts (B operand of the PV MFMA).
    u32x2 p_hi[R], p_lo[R];
    float p32[4], alpha32 = 1.0f;  // kP32: P itself, and the rescale of the running output
#pragma unroll
    for (int b = 0; b < R; b++) {
        float sc[4];
#pragma unroll
        for (int i = 0; i < 4; i++) sc[i] = ok[i] ? s[b][i] * p.scale_log2 : -INFINITY;
        float mx = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float m_new = fmaxf(st[b].m, mx);
        const float ms = (m_new == -INFINITY) ? 0.0f : m_new;
        const float alpha = fast_exp2(st[b].m - ms);
        float pe[4];
        float psum = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float x = sc[i] - ms;
            // fp32: the scaled score's own rounding stays out of the exponent.
            // From 2^23 on half a unit of the maximum's last place is no
            // longer small (at 2^33 it is 2^9: a weight of exp2(512), or of 0
            // for the largest score), and the difference of the rounded
            // scores, at most 0, is kept; so is an infinite maximum's (NaN).
            if constexpr (KV == KV_F32)
                x = ok[i] && fabsf(ms) < 8388608.0f ? fmaf(s[b][i], p.scale_log2, -ms) : x;
            pe[i] = fast_exp2(x);
            psum += pe[i];
        }
        st[b].l = st[b].l * alpha + psum;
        st[b].m = m_new;
        if constexpr (G::kP32) {
            static_assert(R == 1, "fp32 P: one row block");
            alpha32 = alpha;
#pragma unroll
            for (int i = 0; i < 4; i++) p32[i] = pe[i];
            continue;
        }
        // P = hi + lo in the 16-bit type (lo = the exact fp32 remainder of hi)
        const uint32_t h01 = pack16<KV>(pe[0], pe[1]), h23 = pack16<KV>(pe[2], pe[3]);
        const f32x2 r01 = unpack16<KV>(h01), r23 = unpack16<KV>(h23);
        p_hi[b] = u32x2{h01, h23};
        p_lo[b] = u32x2{pack16<KV>(pe[0] - r01.x, pe[1] - r01.y),
                        pack16<KV>(pe[2] - r23.x, pe[3] - r23.y)};
        // Rescale only when some head's running max moved: alpha is then
        // exactly 1 in every lane, and x * 1 == x, so skipping is exact (past
        // the first few hundred tokens most tiles skip).
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int n = 0; n < G::kDimBlocks; n++) st[b].o[n] *= alpha;
        }
    }

    // O^T += V^T P for every dim block: the block's dim of the lane's four
    // token rows, a 16-bit half of one word of each row's chunk.  kP32: the
    // element in fp32, one 16x16x4 per row; the tile's sum starts from zero
    // and is then added to the rescaled running output, one rounding per tile
    // in the long sum instead of 16.
    for_groups<KV, D>([&](auto vb) {
        constexpr int B = decltype(vb)::value;
        u32x4 v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = vs.template chunk<B>(r, lane, i);
#pragma unroll
        for (int e = 0; e < G::group_dims(B); e++) {
            if constexpr (G::kP32) {
                f32x4 &o = st[0].o[G::kDims * B + e];
                f32x4 t[4];
#pragma unroll
                for (int i = 0; i < 4; i++)
                    t[i] = mfma_f32(chunk_elem<KV>(v[i], e), __builtin_bit_cast(uint32_t, p32[i]),
                                    i % G::kPvChain == 0 ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : t[i - 1]);
                if constexpr (G::kPvChain == 4) o = o * alpha32 + t[3];
                else if constexpr (G::kPvChain == 2) o = o * alpha32 + (t[1] + t[3]);
                else o = o * alpha32 + ((t[0] + t[1]) + (t[2] + t[3]));
                continue;
            }
            const int n = G::kDims * B + e, w = e / 2;
            const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
            const u32x2 a = {__builtin_amdgcn_perm(lane_word(v[1], w), lane_word(v[0], w), sel),
                             __builtin_amdgcn_perm(lane_word(v[3], w), lane_word(v[2], w), sel)};
#pragma unroll
            for (int b = 0; b < R; b++) {
                st[b].o[n] = mfma_pv<KV>(a, p_hi[b], st[b].o[n]);
                st[b].o[n] = mfma_pv<KV>(a, p_lo[b], st[b].o[n]);
            }
        }
    });
}

// The lane's dims of row i = 4g + r of V group B (consecutive ones from
// mfma_dim(B, i)), gathered from the blocks of a state.
template <int KV, int D, int B>
__device__ __forceinline__ void state_dims(const MfmaState<KV, D> &st, int r,
                                           float (&f)[MfmaGeometry<KV, D>::group_dims(B)]) {
    using G = MfmaGeometry<KV, D>;
#pragma unroll
    for (int e = 0; e < G::group_dims(B); e++) f[e] = st.o[G::kDims * B + e][r];
}

// N consecutive floats of a row whose first one is at a multiple of N (N = 4
// or 8: 16-byte aligned; else of the largest power of two in N).
template <int N> constexpr int float_step() { return N % 4 == 0 ? 4 : N % 2 == 0 ? 2 : 1; }

template <int N> __device__ __forceinline__ void store_floats(float *dst, const float (&f)[N]) {
    constexpr int S = float_step<N>();
#pragma unroll
    for (int e = 0; e < N; e += S) {
        if constexpr (S == 4) *(f32x4 *)(dst + e) = f32x4{f[e], f[e + 1], f[e + 2], f[e + 3]};
        else if constexpr (S == 2) *(f32x2 *)(dst + e) = f32x2{f[e], f[e + 1]};
        else dst[e] = f[e];
    }
}

template <int N> __device__ __forceinline__ void load_floats(const float *src, float (&f)[N]) {
    constexpr int S = float_step<N>();
#pragma unroll
    for (int e = 0; e < N; e += S) {
        if constexpr (S == 4) {
            const f32x4 x = *(const f32x4 *)(src + e);
#pragma unroll
            for (int k = 0; k < 4; k++) f[e + k] = x[k];
        } else if constexpr (S == 2) {
            const f32x2 x = *(const f32x2 *)(src + e);
            f[e] = x.x;
            f[e + 1] = x.y;
        } else {
            f[e] = src[e];
        }
    }
}

// N consecutive values of the element type at element d of a row (d a
// multiple of N), rounded to nearest even.
template <int KV, int N>
__device__ __forceinline__ void store_elems(char *row, int d, const float (&f)[N]) {
    if constexpr (KV == KV_F32) {
        store_floats((float *)row + d, f);
    } else {
        static_assert(N % 2 == 0, "16-bit elements go in pairs");
        uint32_t w[N / 2];
#pragma unroll
        for (int e = 0; e < N / 2; e++) w[e] = pack16<KV>(f[2 * e], f[2 * e + 1]);
        uint32_t *dst = (uint32_t *)(row + (size_t)d * 2);
        if constexpr (N == 8) *(u32x4 *)dst = u32x4{w[0], w[1], w[2], w[3]};
        else if constexpr (N == 4) *(u32x2 *)dst = u32x2{w[0], w[1]};
        else
#pragma unroll
            for (int e = 0; e < N / 2; e++) dst[e] = w[e];
    }
}

// Where the partition body finds a sequence's length, block table and query
// rows.  kSrcBatch: the batch's own arrays (DecodeParams and the lens /
// tables kernel arguments).  The cascade's in-kernel plan
// (paged_decode_cascade_attn.h) keeps the per-sequence data of its two
// batches in LDS (CascadeLdsPlan) and reads the caller's block tables and
// query rows in place: kSrcSuffix, the suffix of each caller sequence (its
// length past the shared prefix, its pages from its first private one);
// kSrcPrefix, the prefix-batch sequences (a group's shared pages, from its
// lowest member's table row, and query rows gathered from its members).
enum { kSrcBatch = 0, kSrcSuffix = 1, kSrcPrefix = 2 };

struct CascadeLdsPlan {
    const int *slen;    // [num_seqs] suffix length of caller sequence s
    const int *soff;    // [num_seqs] its shared prefix pages (the suffix's first page)
    const int *vlen;    // [v_max] length of prefix-batch sequence v (0: unused)
    const int *vrow;    // [v_max] block-table row of v's pages (its group's lowest member)
    const int *vdesc;   // [v_max][4] v's group: its first prefix-batch sequence, its
                        // members, -, the group id (-1: v unused)
    const int *grp;     // [num_seqs] group of caller sequence s (-1: none)
    int *win;           // [waves per workgroup][32] each wavefront's members of a piece
    int *p_row;         // [num_seqs] (global) a member's first row in the prefix batch
    const char *q;      // caller's query rows: [num_seqs][num_heads][head_size]
    const char *const *q_rows;  // or, when set, sequence s's rows at q_rows[s]
    int num_heads;      // caller's query heads
    int group;          // caller's query heads per kv head
    int rows;           // query rows per kv head of a prefix-batch sequence
    int num_seqs;       // caller's sequences
};

// Clamped length of sequence s of the batch under source SRC.
template <int SRC>
__device__ __forceinline__ int src_len(const DecodeParams &p, const int *__restrict__ lens, int s,
                                       const CascadeLdsPlan *cp) {
    if constexpr (SRC == kSrcBatch)
        return p.nt_fold ? p.nt_len - 1 : min(max(lens[s], 0), p.max_ctx);
    else if constexpr (SRC == kSrcSuffix) return __builtin_amdgcn_readfirstlane(cp->slen[s]);
    else return __builtin_amdgcn_readfirstlane(cp->vlen[s]);
}

// Block table of sequence s of the batch under source SRC.
template <int SRC>
__device__ __forceinline__ const int *src_table(const DecodeParams &p,
                                                const int *__restrict__ tables, int s,
                                                const CascadeLdsPlan *cp) {
    if constexpr (SRC == kSrcBatch) return tables + (size_t)s * p.max_blocks;
    else if constexpr (SRC == kSrcSuffix)
        return tables + (size_t)s * p.max_blocks + __builtin_amdgcn_readfirstlane(cp->soff[s]);
    else return tables + (size_t)__builtin_amdgcn_readfirstlane(cp->vrow[s]) * p.max_blocks;
}

// One piece of a wavefront's stream-K range: tokens [t_begin, t_end) of the
// segment (sequence s, kv head kvh, head tile ht).  `whole`: the piece is the
// entire segment (the output is written directly); else its partial goes to
// `slot`.  All fields are wavefront-uniform.
struct MfmaPiece {
    int s, kvh, ht, t_begin, t_end, L, whole, slot;
};

// Cursor over the pieces of one wavefront's range [g, g_end) of the batch's
// split units; s is the sequence holding unit g, w the wavefront (its
// partial slots), ht its head tile under paired head tiles (else -1).
struct RangeCursor {
    int g, g_end, s, first, w, ht;
};

// The next piece of the range (false at its end).  Same decomposition as
// stream_k_walk, one piece at a time, so the kernel can look one piece ahead.
// A range that ends inside a segment's start-up units makes no piece of it.
template <int TT, int SRC = kSrcBatch>
__device__ __forceinline__ bool next_piece(const DecodeParams &p, const int *__restrict__ lens,
                                           const int *pre, RangeCursor &c, MfmaPiece &pc,
                                           const CascadeLdsPlan *cp = nullptr) {
    const int segs = seq_segments(p);
    while (c.g < c.g_end) {
        const int L = src_len<SRC>(p, lens, c.s, cp);
        const int Ts = (L + TT - 1) / TT;
        const int Cs = segment_units(p, Ts);
        const int base = __builtin_amdgcn_readfirstlane(pre[c.s]);
        const int local = c.g - base;
        const int seg = local / Cs;
        const int u0 = local - seg * Cs;
        const int u1 = min(Cs, u0 + (c.g_end - c.g));
        const int t0 = max(u0 - p.seg_cost, 0), t1 = max(u1 - p.seg_cost, 0);
        c.g += u1 - u0;
        const int cur_s = c.s;
        if (c.g - base >= Cs * segs) {  // sequence done: next one with tiles
            int s = c.s + 1;
            while (s < p.num_seqs - 1 && pre[s + 1] == pre[s]) s++;
            c.s = __builtin_amdgcn_readfirstlane(s);
        }
        if (t1 <= t0) continue;  // only start-up units of this segment (the range's end)
        pc.s = cur_s;
        if (c.ht >= 0) {  // paired head tiles: a segment per kv head
            pc.kvh = seg;
            pc.ht = c.ht;
        } else {
            pc.kvh = seg / p.head_tiles;
            pc.ht = seg - pc.kvh * p.head_tiles;
        }
        pc.t_begin = t0 * TT;
        pc.t_end = min(L, t1 * TT);
        pc.L = L;
        pc.whole = t0 == 0 && t1 == Ts;
        pc.slot = c.w * 2 + (c.first ? 0 : 1);
        c.first = 0;
        return true;
    }
    return false;
}

// Q rows of the piece's (up to) 16R query heads in the MFMA B layout (row
// block b, lane: head 16b + j, dims 32c+8g..+7); heads past the group read
// as zero.  kSrcPrefix: with the group's rows laid end to end (rows per
// prefix-batch sequence), row k is query head k % G (of the kv head's G) of
// the group's member of rank k / G, members ranked in sequence order; rows
// past the last member read as zero.  The wavefront finds the (at most 16R)
// members of its rows with one ballot per 64 caller sequences, and the piece
// that starts its sequence's kv head 0 stores each member's first row
// (p_row).
template <int KV, int D, int R, int SRC = kSrcBatch>
__device__ __forceinline__ void mfma_load_q(const DecodeParams &p, const MfmaPiece &pc, int lane,
                                            u32x4 (&q)[R][MfmaGeometry<KV, D>::kQkSteps],
                                            const CascadeLdsPlan *cp = nullptr) {
    const int j = lane & 15, g = lane >> 4;
    const int g0 = pc.ht * kMfmaHeads * R;
    auto q_chunk_ok = [](int c, int gr) {
        constexpr int RBQ = MfmaGeometry<KV, D>::kRowBytes;
        return RBQ % 64 == 0 || 64 * c + 16 * gr < RBQ;
    };
    if constexpr (SRC == kSrcPrefix) {
        const int *d = cp->vdesc + 4 * pc.s;
        const int vbase = __builtin_amdgcn_readfirstlane(d[0]);
        const int count = __builtin_amdgcn_readfirstlane(d[1]);
        const int gid = __builtin_amdgcn_readfirstlane(d[3]);
        const int G = cp->group;
        const int row0 = (pc.s - vbase) * cp->rows + g0;
        const int r_lo = row0 / G, r_hi = min((row0 + 16 * R - 1) / G, count - 1);
        int *win = cp->win + (threadIdx.x >> 6) * (16 * R);
        int acc = 0;
        wave_lds_fence();  // after the last piece's lookups
        for (int c0 = 0; c0 < cp->num_seqs && acc <= r_hi; c0 += 64) {
            const int s = c0 + lane;
            const bool in = s < cp->num_seqs && cp->grp[s] == gid;
            const unsigned long long m = __ballot(in);
            const int rk = acc + (int)__builtin_amdgcn_mbcnt_hi(
                                     (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
            if (in && rk >= r_lo && rk <= r_hi) win[rk - r_lo] = s;
            acc += __popcll(m);
        }
        wave_lds_fence();
        __builtin_amdgcn_wave_barrier();
        const size_t row_bytes = MfmaGeometry<KV, D>::kRowBytes;
        const bool first = pc.kvh == 0 && pc.t_begin == 0;
#pragma unroll
        for (int b = 0; b < R; b++) {
            const int rig = row0 + 16 * b + j;
            const int r = rig / G, gq = rig - r * G;
            const char *src = nullptr;
            if (r < count) {
                const int s = win[r - r_lo];
                const size_t h = (size_t)pc.kvh * G + gq;
                src = cp->q_rows ? cp->q_rows[s] + h * row_bytes
                                 : cp->q + ((size_t)s * cp->num_heads + h) * row_bytes;
                if (first && gq == 0 && g == 0) cp->p_row[s] = vbase * cp->rows + r * G;
            }
#pragma unroll
            for (int c = 0; c < MfmaGeometry<KV, D>::kQkSteps; c++)
                q[b][c] = src && q_chunk_ok(c, g) ? load16(src + 64 * c + 16 * g) : u32x4{0, 0, 0, 0};
        }
        return;
    }
    const int nh = min(kMfmaHeads * R, p.group - g0);
    constexpr int RB = MfmaGeometry<KV, D>::kRowBytes;
    const char *q0 = q_row(p, pc.s, pc.kvh * p.group + g0, D, MfmaGeometry<KV, D>::kElemBytes);
#pragma unroll
    for (int b = 0; b < R; b++)
#pragma unroll
        for (int c = 0; c < MfmaGeometry<KV, D>::kQkSteps; c++)
            q[b][c] = (16 * b + j < nh && q_chunk_ok(c, g))
                          ? load16(q0 + (size_t)(16 * b + j) * RB + 64 * c + 16 * g)
                          : u32x4{0, 0, 0, 0};
}

// Prefix fold (DecodeParams::fold_row) of a piece that starts its segment:
// the prefix pass's result for each head, (m = lse, l = 1, O^T = the
// normalized prefix row), is merged into the piece's state after its last
// tile, like one more partial.  Its loads are issued when the piece begins
// (R = 1), so their latency hides behind the piece's tiles; with R = 2 the 32
// extra registers would not fit, and they are loaded at the end.
template <int KV, int D, int R> struct MfmaFold {
    f32x4 o[R][MfmaGeometry<KV, D>::kDimBlocks];
    float m[R];
    int base;  // the sequence's fold base, < 0: no fold
};

template <int KV, int D, int R>
__device__ __forceinline__ void mfma_fold_load(const DecodeParams &p, const MfmaPiece &pc,
                                               int lane, MfmaFold<KV, D, R> &f) {
    using G = MfmaGeometry<KV, D>;
    const int j = lane & 15, g = lane >> 4;
    const int g0 = pc.ht * kMfmaHeads * R;
    const int nh = min(kMfmaHeads * R, p.group - g0);
#pragma unroll
    for (int b = 0; b < R; b++) {
        // heads past the group read head g0 (valid) and are never written
        const size_t r = fold_state_row(p, f.base, pc.kvh, g0 + (16 * b + j < nh ? 16 * b + j : 0));
        f.m[b] = p.fold_lse[r];
        for_groups<KV, D>([&](auto vb) {
            constexpr int B = decltype(vb)::value, N = G::group_dims(B);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int d = mfma_dim<KV, D>(B, 4 * g + i);
                float x[N] = {};
                if (!G::kPadded || d < D) load_floats(p.fold_out + r * D + d, x);
#pragma unroll
                for (int e = 0; e < N; e++) f.o[b][G::kDims * B + e][i] = x[e];
            }
        });
    }
}

template <int KV, int D, int R>
__device__ __forceinline__ void mfma_fold_apply(const MfmaFold<KV, D, R> &f, int lane,
                                                MfmaState<KV, D> (&st)[R]) {
    const int g = lane >> 4;
#pragma unroll
    for (int b = 0; b < R; b++) {
        const float M = fmaxf(st[b].m, f.m[b]);
        const float Ms = (M == -INFINITY) ? 0.0f : M;
        const float a = fast_exp2(st[b].m - Ms), w = fast_exp2(f.m[b] - Ms);
        st[b].l = st[b].l * a + (g == 0 ? w : 0.0f);  // l is summed over the 4 lane groups
#pragma unroll
        for (int n = 0; n < MfmaGeometry<KV, D>::kDimBlocks; n++)
            st[b].o[n] = st[b].o[n] * a + f.o[b][n] * w;
        st[b].m = M;
    }
}

// Block ids of the piece's tiles first .. first+63, lane i holding tile
// first+i (clamped to the piece's last tile).
template <int SRC = kSrcBatch>
__device__ __forceinline__ int mfma_load_ids(const DecodeParams &p, const int *__restrict__ tables,
                                             const MfmaPiece &pc, int first, int lane,
                                             const CascadeLdsPlan *cp = nullptr) {
    const int *bt = src_table<SRC>(p, tables, pc.s, cp);
    const int ti = pc.t_begin + 16 * (first + lane);
    return bt[(ti < pc.t_end ? ti : pc.t_end - 1) >> p.bs_shift];
}

}  // namespace xhip

namespace xhip {

// Where a finished segment's rows go: its output rows (element type), or in
// partial-output mode its fp32 rows and log-sum-exp.  st holds unreduced
// per-lane sums (lane group g of head j); they are reduced here.
template <int KV, int D, int R, bool HS = false>
__device__ __forceinline__ void mfma_write_rows(const DecodeParams &p, const MfmaPiece &pc,
                                                int lane, const MfmaState<KV, D> (&st)[R]) {
    using G = MfmaGeometry<KV, D>;
    constexpr int GT = kMfmaHeads * R;
    const int j = lane & 15, gq = lane >> 4;
    const int g0 = pc.ht * GT;
    const int nh = min(GT, p.group - g0);
    const size_t qrow0 = ((size_t)pc.s * p.num_heads + (size_t)pc.kvh * p.group + g0) * D;
#pragma unroll
    for (int b = 0; b < R; b++) {
        float l = st[b].l;
        l += __shfl_xor(l, 16);
        l += __shfl_xor(l, 32);
        const int hj = 16 * b + j;  // head of this lane in the tile
        if (hj >= nh) continue;
        const float inv = l > 0.0f ? 1.0f / l : 0.0f;
        const size_t row = qrow0 + (size_t)hj * D;  // element index
        char *orow = HS          ? (char *)p.out_h + row * 2
                     : p.out_f32 ? (char *)(p.out_f32 + row)
                                 : o_row(p, pc.s, pc.kvh * p.group + g0 + hj, D, G::kElemBytes);
        for_groups<KV, D>([&](auto vb) {
            constexpr int B = decltype(vb)::value, N = G::group_dims(B);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int d = mfma_dim<KV, D>(B, 4 * gq + i);
                if (G::kPadded && d >= D) continue;
                float f[N];
                state_dims<KV, D, B>(st[b], i, f);
#pragma unroll
                for (int e = 0; e < N; e++) f[e] *= inv;
                if constexpr (HS) store_elems<KV_F16>(orow, d, f);
                else if (p.out_f32) store_floats((float *)orow + d, f);
                else store_elems<KV>(orow, d, f);
            }
        });
        if ((HS || p.out_f32) && gq == 0)
            p.out_lse[qrow0 / D + hj] = l > 0.0f ? st[b].m + log2f(l) : -INFINITY;
    }
}

// The partial of a cut segment's piece, in the piece's slot of the split-K
// workspace: fp32 (m, l, unnormalized o), or HS: an fp16 state
// (DecodeParams::ws_h) (m + log2 l, 1, o / l in fp16).
template <int KV, int D, int R, bool HS = false>
__device__ __forceinline__ void mfma_write_partial(const DecodeParams &p, const MfmaPiece &pc,
                                                   int lane, const MfmaState<KV, D> (&st)[R]) {
    using G = MfmaGeometry<KV, D>;
    constexpr int GT = kMfmaHeads * R;
    const int j = lane & 15, gq = lane >> 4;
    const int nh = min(GT, p.group - pc.ht * GT);
#pragma unroll
    for (int b = 0; b < R; b++) {
        float l = st[b].l;
        l += __shfl_xor(l, 16);
        l += __shfl_xor(l, 32);
        const int hj = 16 * b + j;
        if (hj >= nh) continue;
        const float inv = !HS ? 1.0f : l > 0.0f ? 1.0f / l : 0.0f;
        const size_t row = ((size_t)pc.slot * GT + hj) * D;
        for_groups<KV, D>([&](auto vb) {
            constexpr int B = decltype(vb)::value, N = G::group_dims(B);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int d = mfma_dim<KV, D>(B, 4 * gq + i);
                if (G::kPadded && d >= D) continue;
                float f[N];
                state_dims<KV, D, B>(st[b], i, f);
                if constexpr (HS) {
#pragma unroll
                    for (int e = 0; e < N; e++) f[e] *= inv;
                    store_elems<KV_F16>((char *)p.ws_h + row * 2, d, f);
                } else {
                    store_floats(p.ws_o + row + d, f);
                }
            }
        });
        if (gq == 0) {
            float *ml = p.ws_ml + ((size_t)pc.slot * GT + hj) * 2;
            ml[0] = !HS ? st[b].m : l > 0.0f ? st[b].m + log2f(l) : -INFINITY;
            ml[1] = !HS ? l : l > 0.0f ? 1.0f : 0.0f;
        }
    }
}

// LDS slot of one wavefront for the workgroup-level combine (mfma_wg_fixup):
// a state in the lane layout of MfmaState (per-lane o, m and unreduced l),
// so two states merge lane by lane.
template <int KV, int D> struct MfmaFixSlot {
    f32x4 o[MfmaGeometry<KV, D>::kDimBlocks][64];
    float m[64], l[64];
    int ends;  // the state reaches the end of its segment
};

template <int KV, int D>
__device__ __forceinline__ void fix_store(MfmaFixSlot<KV, D> &slot, int lane, const MfmaState<KV, D> &st) {
#pragma unroll
    for (int n = 0; n < MfmaGeometry<KV, D>::kDimBlocks; n++) slot.o[n][lane] = st.o[n];
    slot.m[lane] = st.m;
    slot.l[lane] = st.l;
}

template <int KV, int D>
__device__ __forceinline__ void fix_load(const MfmaFixSlot<KV, D> &slot, int lane, MfmaState<KV, D> &st) {
#pragma unroll
    for (int n = 0; n < MfmaGeometry<KV, D>::kDimBlocks; n++) st.o[n] = slot.o[n][lane];
    st.m = slot.m[lane];
    st.l = slot.l[lane];
}

// st <- st (+) the state in slot (online log-sum-exp, per lane).
template <int KV, int D>
__device__ __forceinline__ void fix_absorb(const MfmaFixSlot<KV, D> &slot, int lane, MfmaState<KV, D> &st) {
    const float mo = slot.m[lane];
    const float M = fmaxf(st.m, mo);
    const float Ms = (M == -INFINITY) ? 0.0f : M;
    const float a = fast_exp2(st.m - Ms), b = fast_exp2(mo - Ms);
    st.l = st.l * a + slot.l[lane] * b;
#pragma unroll
    for (int n = 0; n < MfmaGeometry<KV, D>::kDimBlocks; n++) st.o[n] = st.o[n] * a + slot.o[n][lane] * b;
    st.m = M;
}

// The workgroup's relay slot of the mode-2 combine: one state of R row
// blocks in the lane layout.
template <int KV, int D, int R> struct MfmaRelaySlot {
    f32x4 o[R][MfmaGeometry<KV, D>::kDimBlocks][64];
    float m[R][64], l[R][64];
};

// LDS of one workgroup of the partition kernel: the query rows of each
// wavefront's piece (mfma_q_in_lds), its V tile (short rows), and the slots of
// the workgroup-level combine (by mode).  Mode 2: the relay slot takes the
// query rows' place, which no wavefront reads past the combine's first
// barrier, and beside it, per wavefront, whether it relayed its state and
// whether that state reaches the end of its segment.  (With a place of its
// own the slot left the cascade's in-kernel plan 30 KB for two workgroups per
// CU, not 46: 64 / 1 heads, 720 sequences in 16 groups went to the plan
// kernels, 143 us a step for 131.)
template <int KV, int D, int R, int FIX = mfma_wg_fixup(kMfmaHeads * R, D)> struct MfmaLds {
    MfmaQLds<KV, D, R> qs[kMfmaWavesPerGroup];
    MfmaVLds<KV, D> vs[kMfmaWavesPerGroup];
};
template <int KV, int D, int R> struct MfmaLds<KV, D, R, 1> {
    MfmaQLds<KV, D, R> qs[kMfmaWavesPerGroup];
    MfmaVLds<KV, D> vs[kMfmaWavesPerGroup];
    MfmaFixSlot<KV, D> fix[kMfmaWavesPerGroup];
};
template <int KV, int D, int R> struct MfmaLds<KV, D, R, 2> {
    union {
        MfmaQLds<KV, D, R> qs[kMfmaWavesPerGroup];
        MfmaRelaySlot<KV, D, R> relay;
    };
    MfmaVLds<KV, D> vs[kMfmaWavesPerGroup];
    int relayed[kMfmaWavesPerGroup];
    int ends[kMfmaWavesPerGroup];
};

// st <- st (+) the partial in workspace slot `slot` (its l is the reduced
// sum: lane group 0 takes it; fp32, or HS: an fp16 state).  Rows past the group
// were never written; they are left alone.
template <int KV, int D, int R, bool HS = false>
__device__ __forceinline__ void absorb_partial(const DecodeParams &p, int slot, int ht, int lane,
                                               MfmaState<KV, D> (&st)[R]) {
    using G = MfmaGeometry<KV, D>;
    constexpr int GT = kMfmaHeads * R;
    const int j = lane & 15, gq = lane >> 4;
    const int nh = min(GT, p.group - ht * GT);
#pragma unroll
    for (int b = 0; b < R; b++) {
        const int hj = 16 * b + j;
        if (hj >= nh) continue;
        const size_t row = ((size_t)slot * GT + hj) * D;
        const float mo = p.ws_ml[((size_t)slot * GT + hj) * 2];
        const float lo = gq == 0 ? p.ws_ml[((size_t)slot * GT + hj) * 2 + 1] : 0.0f;
        const float M = fmaxf(st[b].m, mo);
        const float Ms = (M == -INFINITY) ? 0.0f : M;
        const float a = fast_exp2(st[b].m - Ms), w = fast_exp2(mo - Ms);
        st[b].l = st[b].l * a + lo * w;
        for_groups<KV, D>([&](auto vb) {
            constexpr int B = decltype(vb)::value, N = G::group_dims(B);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int d = mfma_dim<KV, D>(B, 4 * gq + i);
                if (G::kPadded && d >= D) continue;
                const size_t at = row + d;
                float x[N];
                if constexpr (HS) {
#pragma unroll
                    for (int e = 0; e < N; e += 2) {
                        const f32x2 h =
                            unpack16<KV_F16>(*(const uint32_t *)((const char *)p.ws_h + (at + e) * 2));
                        x[e] = h.x;
                        x[e + 1] = h.y;
                    }
                } else {
                    load_floats(p.ws_o + at, x);
                }
#pragma unroll
                for (int e = 0; e < N; e++) {
                    f32x4 &o = st[b].o[G::kDims * B + e];
                    o[i] = o[i] * a + x[e] * w;
                }
            }
        });
        st[b].m = M;
    }
}

// Partition kernel, MFMA tile path (head tile of 16R query heads).
//
// A wavefront walks the pieces of its stream-K range (usually one or two
// segments) as one pipeline: while the last tile of a piece is computed, the
// next piece's first K/V tile is already in flight, and its block ids were
// requested when the current piece began.  Without this look-ahead a
// wavefront whose range crosses a segment boundary waited on a chain of
// dependent loads (block ids, then the first tile) at the crossing, and those
// wavefronts finished the launch last (measured on MI355X: 3 us later on
// average at config 2).  Q is loaded when its piece begins: requesting the
// next piece's Q a piece early as well gained ~1% at configs 2-4 but cost 5%
// (cascade) to 10% (plain decode) at config 5 (measured, same box).
//
// Cut segments (mfma_wg_fixup instantiations).  A piece that is not a whole
// segment is cut at the start (it continues the previous wavefront's range),
// at the end (the next wavefront continues it), or both.  Writing each such
// piece's fp32 partial to memory put ~16-20 MB of stores at config 4b into
// the wavefronts' critical paths (a cut first piece's stores delay the next
// piece's loads, which share the memory counter; every wavefront ends with
// one), measured at 8.6 us of a 76 us kernel.  Instead: a cut first piece
// followed by more pieces goes to the wavefront's LDS slot; the last piece's
// state stays in registers; at the end, a last piece that continues the
// left neighbour's goes to the slot too, and after one workgroup barrier
// the leftmost holder of each segment in the workgroup absorbs the slots of
// the neighbours its piece continues into and writes it: finished rows when
// the whole segment lay in the workgroup, else one partial.  (A sweep from
// the last wavefront down to the first, one barrier per wavefront, kept the
// workgroup ~1.8 us past its last tile, measured on MI355X.)  The first
// wavefront's cut first piece (its left neighbour is in another workgroup)
// is written as a partial after its range, from its slot.
// Mode 2 (two row blocks) keeps one relay slot per workgroup: cut first
// pieces followed by more pieces are written as partials by every
// wavefront, and a left neighbour absorbs such a partial from memory (the
// workgroup barrier orders it) instead of from the relay slot.
//
// The body runs one workgroup's four ranges: logical workgroup `wg` of a
// plan of `waves` wavefronts over the batch of p, whose split-unit prefix
// `pre` is in LDS.  PAIR: the batch's head tiles are paired
// (DecodeParams::pair_tiles): the workgroup's two pairs of wavefronts walk
// two ranges, one head tile per wavefront, and every cut piece leaves its
// own partial (no workgroup combine).  SRC: where the batch's per-sequence
// data is (kSrcBatch: lens / tables and p; else the in-kernel cascade plan
// cp).  HS: partial-output rows and partials are fp16 states
// (DecodeParams::out_h, ws_h).
template <int KV, int D, int R, bool PAIR = false, int SRC = kSrcBatch, bool HS = false>
__device__ __forceinline__ void mfma_partition_body(
    const DecodeParams &p, const int *__restrict__ lens, const int *__restrict__ tables,
    const int *pre, int wg, int waves,
    MfmaLds<KV, D, R, PAIR ? 0 : mfma_wg_fixup(kMfmaHeads * R, D)> &sm,
    const CascadeLdsPlan *cp = nullptr) {
    using G = MfmaGeometry<KV, D>;
    constexpr int EB = G::kElemBytes;
    constexpr int FIX = PAIR ? 0 : mfma_wg_fixup(kMfmaHeads * R, D);
    constexpr bool kFoldAhead = R == 1 && KV != KV_F32;  // (registers for it)
    constexpr int NW = kMfmaWavesPerGroup;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if constexpr (FIX == 2) {
        // ordered before any read by the sweep's first barrier
        if (lane == 0) sm.relayed[wave] = 0;
    }

    const int B = p.num_seqs;
    const int total = pre[B];
    const int w = wg * NW + wave;
    const int wr = PAIR ? w >> 1 : w;  // this wavefront's range
    const int tpw = tiles_per_wave(total, PAIR ? waves >> 1 : waves, p.min_tiles_per_wave);
    const long long g_lo = (long long)wr * tpw;

    MfmaState<KV, D> st[R];   // the state of the piece being computed; after the loop, the last one's
    MfmaPiece pc;         // the piece being computed; after the loop, the last one
    bool have_last = false;  // FIX: the last piece is cut (its state is kept for the sweep)
    MfmaPiece pc_first;      // FIX == 1, first wavefront: its cut first piece, saved in its slot
    bool first_saved = false;
#if XHIP_TRACING
    int n_tiles = 0, n_pieces = 0;
#endif
    RangeCursor cur;
    cur.g = (int)g_lo;
    cur.g_end = g_lo < total ? min(total, cur.g + tpw) : cur.g;
    cur.first = 1;
    cur.w = w;
    cur.ht = PAIR ? (w & 1) : -1;
    {
        // the sequence holding unit g: the last s with pre[s] <= g (empty
        // sequences share their successor's prefix, so this lands on one
        // with tiles)
        int lo = 0, hi = B - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (pre[mid] <= cur.g) lo = mid; else hi = mid - 1;
        }
        cur.s = __builtin_amdgcn_readfirstlane(lo);
    }

    // A range inside one segment's start-up units holds no tile (only when
    // tpw <= seg_cost); the segment's tiles belong to the next wavefront.
    if (g_lo < total && next_piece<16, SRC>(p, lens, pre, cur, pc, cp)) {
        u32x4 ql[R][G::kQkSteps];
        MfmaQuery<KV, D, R> q;
        int ids;
        if constexpr (SRC == kSrcPrefix) {
            // (the block ids' round trip overlaps the members' lookup)
            ids = mfma_load_ids<SRC>(p, tables, pc, 0, lane, cp);
            mfma_load_q<KV, D, R, SRC>(p, pc, lane, ql, cp);
        } else {
            mfma_load_q<KV, D, R, SRC>(p, pc, lane, ql, cp);
            ids = mfma_load_ids<SRC>(p, tables, pc, 0, lane, cp);
        }
        q.put(sm.qs[wave], lane, ql);
        // fold base of the current piece (requested a piece ahead from here on)
        int fold_base = (p.fold_row && pc.t_begin == 0) ? p.fold_row[pc.s] : -1;
        MfmaTileRegs<KV, D> ra, rb;
        int blk_a = __builtin_amdgcn_readlane(ids, 0);
        XHIP_WAVE_STAMP(p, wave, 0);
        {
            const char *kb = (const char *)p.k + (size_t)pc.kvh * (size_t)p.kv_head_stride * EB;
            const char *vb = (const char *)p.v + (size_t)pc.kvh * (size_t)p.kv_head_stride * EB;
            mfma_load_tile<KV, D>(p, kb, vb, pc.t_begin, pc.t_end, blk_a, lane, pc.s < p.cached_seqs,
                              ra);
        }

        while (true) {
            MfmaPiece pn = pc;
            const bool has_next = next_piece<16, SRC>(p, lens, pre, cur, pn, cp);
            // Issued whether or not there is a next piece (pn is then the
            // current one again), so every path through the loop below has
            // the same loads in flight and the compiler's wait counts stay
            // exact.
            const int ids_n = mfma_load_ids<SRC>(p, tables, pn, 0, lane, cp);
            const int fold_base_n =
                (p.fold_row && has_next && pn.t_begin == 0) ? p.fold_row[pn.s] : -1;
            const char *kb = (const char *)p.k + (size_t)pc.kvh * (size_t)p.kv_head_stride * EB;
            const char *vb = (const char *)p.v + (size_t)pc.kvh * (size_t)p.kv_head_stride * EB;
            const char *kb_n = (const char *)p.k + (size_t)pn.kvh * (size_t)p.kv_head_stride * EB;
            const char *vb_n = (const char *)p.v + (size_t)pn.kvh * (size_t)p.kv_head_stride * EB;
            const bool cached = pc.s < p.cached_seqs;
            const bool cached_n = has_next && pn.s < p.cached_seqs;
            const int *bt = src_table<SRC>(p, tables, pc.s, cp);

#pragma unroll
            for (int b = 0; b < R; b++) {
#pragma unroll
                for (int n = 0; n < G::kDimBlocks; n++) st[b].o[n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                st[b].m = -INFINITY;
                st[b].l = 0.0f;
            }
            MfmaFold<KV, D, R> fold;
            fold.base = fold_base;
            if (kFoldAhead && fold.base >= 0) mfma_fold_load<KV, D, R>(p, pc, lane, fold);
            const int ntiles = (pc.t_end - pc.t_begin + 15) >> 4;
#if XHIP_TRACING
            n_tiles += ntiles;
            n_pieces++;
#endif
            for (int i = 0; i < ntiles; i++) {
                if (i > 0 && (i & 63) == 0) ids = mfma_load_ids<SRC>(p, tables, pc, i, lane, cp);
                const int t0 = pc.t_begin + 16 * i;
                // The next tile: this piece's, else the next piece's first (all
                // rows out of range when there is none).
                const int nl = (i + 1) & 63;
                const bool in_piece = i + 1 < ntiles;
                int blk_b;
                if (in_piece)
                    blk_b = nl != 0 ? __builtin_amdgcn_readlane(ids, nl) : bt[(t0 + 16) >> p.bs_shift];
                else
                    blk_b = has_next ? __builtin_amdgcn_readlane(ids_n, 0) : -1;
                mfma_load_tile<KV, D>(p, in_piece ? kb : kb_n, in_piece ? vb : vb_n,
                                  in_piece ? t0 + 16 : pn.t_begin,
                                  in_piece ? pc.t_end : (has_next ? pn.t_end : 0), blk_b, lane,
                                  in_piece ? cached : cached_n, rb);
                mfma_tile<KV, D, R>(p, q, t0, pc.t_end, blk_a >= 0, lane, sm.qs[wave], sm.vs[wave], ra, st);
                ra = rb;
                blk_a = blk_b;
            }

            if (fold.base >= 0) {
                if (!kFoldAhead) mfma_fold_load<KV, D, R>(p, pc, lane, fold);
                mfma_fold_apply<KV, D, R>(fold, lane, st);
            }
            if (pc.whole) {
                mfma_write_rows<KV, D, R, HS>(p, pc, lane, st);
            } else if constexpr (FIX == 1) {
                if (has_next) {
                    // a cut piece with more pieces after it: the wavefront's
                    // first piece, a continuation that ends its segment here.
                    // It goes to the wavefront's slot; the first wavefront's
                    // (whose left neighbour is in another workgroup) is
                    // written as a partial after the range, so that its
                    // stores do not sit in front of the next piece's loads.
                    fix_store<KV, D>(sm.fix[wave], lane, st[0]);
                    if (lane == 0) sm.fix[wave].ends = 1;
                    if (wave == 0) {
                        pc_first = pc;
                        first_saved = true;
                    }
                } else {
                    have_last = true;  // the sweep below decides where it goes
                }
            } else if constexpr (FIX == 2) {
                if (has_next)
                    mfma_write_partial<KV, D, R, HS>(p, pc, lane, st);
                else
                    have_last = true;
            } else {
                mfma_write_partial<KV, D, R, HS>(p, pc, lane, st);
            }
            if (!has_next) break;
            pc = pn;
            ids = ids_n;
            fold_base = fold_base_n;
            mfma_load_q<KV, D, R, SRC>(p, pc, lane, ql, cp);
            q.put(sm.qs[wave], lane, ql);
        }
        XHIP_WAVE_STAMP(p, wave, 1);
    }
#if XHIP_TRACING
    XHIP_WAVE_PUT(p, wave, 2, (unsigned long long)n_tiles | ((unsigned long long)n_pieces << 32));
#endif

    if constexpr (FIX == 2) {
        // As below, with the one relay slot (which overlays the query rows:
        // every wavefront is past its tiles from here on).
        __syncthreads();
        for (int i = NW - 1; i >= 0; i--) {
            if (wave == i && have_last) {
                const bool cut_start = pc.t_begin > 0;
                bool ends = pc.t_end >= pc.L;
                if (!ends && i < NW - 1) {
                    if (sm.relayed[i + 1]) {
#pragma unroll
                        for (int b = 0; b < R; b++) {
                            const float mo = sm.relay.m[b][lane];
                            const float M = fmaxf(st[b].m, mo);
                            const float Ms = (M == -INFINITY) ? 0.0f : M;
                            const float a = fast_exp2(st[b].m - Ms), wt = fast_exp2(mo - Ms);
                            st[b].l = st[b].l * a + sm.relay.l[b][lane] * wt;
#pragma unroll
                            for (int n = 0; n < G::kDimBlocks; n++)
                                st[b].o[n] = st[b].o[n] * a + sm.relay.o[b][n][lane] * wt;
                            st[b].m = M;
                        }
                        ends = sm.ends[i + 1] != 0;
                    } else {
                        // the neighbour's first piece, followed by more
                        // pieces, was written as a partial in its slot 0;
                        // it ends the segment in that range
                        absorb_partial<KV, D, R, HS>(p, (w + 1) * 2, pc.ht, lane, st);
                        ends = true;
                    }
                }
                if (cut_start && i > 0) {
#pragma unroll
                    for (int b = 0; b < R; b++) {
#pragma unroll
                        for (int n = 0; n < G::kDimBlocks; n++) sm.relay.o[b][n][lane] = st[b].o[n];
                        sm.relay.m[b][lane] = st[b].m;
                        sm.relay.l[b][lane] = st[b].l;
                    }
                    if (lane == 0) {
                        sm.relayed[i] = 1;
                        sm.ends[i] = ends ? 1 : 0;
                    }
                } else if (!cut_start && ends) {
                    mfma_write_rows<KV, D, R, HS>(p, pc, lane, st);
                } else {
                    mfma_write_partial<KV, D, R, HS>(p, pc, lane, st);
                }
            }
            __syncthreads();
        }
    }
    if constexpr (FIX == 1) {
        // The wavefronts of a workgroup hold consecutive ranges.  First, a
        // wavefront whose last piece continues its left neighbour's (cut at
        // the start; its range is that one piece) puts the state in its slot,
        // as a cut first piece followed by more pieces already did in the
        // loop.  Then, after one barrier, the leftmost holder of each
        // segment in the workgroup absorbs the slots of the neighbours its
        // piece continues into, left to right, and writes the segment:
        // finished rows when it lay in the workgroup, else one partial.
        const bool cut_start = have_last && pc.t_begin > 0;
        if (have_last && cut_start && wave > 0) {
            fix_store<KV, D>(sm.fix[wave], lane, st[0]);
            if (lane == 0) sm.fix[wave].ends = pc.t_end >= pc.L ? 1 : 0;
        }
        __syncthreads();
        if (first_saved) {
            MfmaState<KV, D> sf[R];
            fix_load<KV, D>(sm.fix[0], lane, sf[0]);
            mfma_write_partial<KV, D, R, HS>(p, pc_first, lane, sf);
        }
        if (have_last && !(cut_start && wave > 0)) {
            bool ends = pc.t_end >= pc.L;
            for (int j = wave + 1; !ends && j < NW; j++) {
                fix_absorb<KV, D>(sm.fix[j], lane, st[0]);
                ends = sm.fix[j].ends != 0;
            }
            if (!cut_start && ends)
                mfma_write_rows<KV, D, R, HS>(p, pc, lane, st);
            else
                mfma_write_partial<KV, D, R, HS>(p, pc, lane, st);
        }
    }
}


template <int KV, int D, int R>
__global__ __launch_bounds__(64 * kMfmaWavesPerGroup, (mfma_waves_per_simd(MfmaGeometry<KV, D>::kRowBytes, kMfmaHeads * R))) void paged_decode_partition_mfma_kernel(
    const DecodeParams p, const int *__restrict__ lens, const int *__restrict__ tables) {
    // lens / tables are p.seq_lens / p.block_tables again: as restrict
    // kernel arguments their wavefront-uniform reads become scalar loads,
    // which do not wait behind the K/V loads in flight.
    extern __shared__ int pre[];  // num_seqs + 1 split-unit prefixes
    __shared__ MfmaLds<KV, D, R> sm;
    XHIP_WG_BEGIN(p);
    batch_prefix<16, kMfmaWavesPerGroup>(p, pre);
    XHIP_WG_STAMP(p, 1);
    const int lb = logical_block(p, pre[p.num_seqs]);
    XHIP_WG_PUT(p, 3, lb);
    mfma_partition_body<KV, D, R>(p, lens, tables, pre, lb, p.num_waves, sm);
    if (blockIdx.x == 0 && threadIdx.x == 0)  // for the merge
        p.ws_prefix[p.num_seqs + 1] =
            tiles_per_wave(pre[p.num_seqs], p.num_waves, p.min_tiles_per_wave);
    XHIP_WG_FLUSH(p);
}

}  // namespace xhip
