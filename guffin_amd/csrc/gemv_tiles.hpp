// Wave-tile operand code shared by the kernels that stream repacked weights: tile registers, the
// matrix-core product of one tile with the activation image, and the walk over a run of blocks.
// The layout of a tile and of the activation receipt is described in gemv_packed.hip / receipt.hpp.
#pragma once
#include "common.hpp"
#include "receipt.hpp"

#include <type_traits>
#include <utility>

namespace guffin {
namespace {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

constexpr uint32_t kTileCols = 64;

__host__ __device__ constexpr uint32_t block_bytes(int dtype) {
    return dtype == GUFFIN_Q8_0 ? 34u : dtype == GUFFIN_Q4_K ? 144u : 210u;
}
__host__ __device__ constexpr uint32_t block_elems(int dtype) { return dtype == GUFFIN_Q8_0 ? 32u : 256u; }

// bytes {0,2} and {1,3} of v as 16-bit fields
__device__ __forceinline__ uint32_t even_bytes(uint32_t v) { return __builtin_amdgcn_perm(0u, v, 0x0c020c00u); }
__device__ __forceinline__ uint32_t odd_bytes(uint32_t v) { return __builtin_amdgcn_perm(0u, v, 0x0c030c01u); }


// =======================================================================================
// Q4_K
// =======================================================================================
// Matrix-core path (Q4_K and Q6_K).  A wave covers 64 columns x one 256-element block; lane l owns column l for everything: its
// quants, its scales, its result.  One v_mfma_f32_4x4x4_16b_f16 multiplies four elements of every column with the four variants
// (hi/lo x row) of the activation image: sixteen 4x4 products side by side, block l / 4 of the B side holding the columns of lanes
// 4 (l / 4) .. + 3, the A side one block of four elements broadcast to all sixteen (CBSZ 4, ABID the block).  So a lane's 8 bytes
// of the image, block l / 4 for variant l % 4, are the operand of 64 elements, and 8 registers that of a whole 256-element block.
// B: the quants as fp16 bit patterns below 2048 (q * 2^-24 times a power of two, exact).  Eight chained instructions are a 32-group
// (four a 16-element half of Q6_K), and every lane finds the four variant sums of its own column in its own registers; it scales them
// by d*sc in fp32.  The -dmin*m term uses the 32-sums.
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

// Weight bytes are used once: streaming (non-temporal) loads keep the caches for the activation
// image, which every wave re-reads.
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 stream_load(const uint8_t* p) {
    const uint4_t v = __builtin_nontemporal_load(reinterpret_cast<const uint4_t*>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}

typedef _Float16 half4_t __attribute__((ext_vector_type(4)));

// bytes from the start of a 256-element tile to the pieces of the lane's column: its 16-byte pieces lie 256 bytes apart (k-slices),
// 16 columns side by side, the column groups 2048 bytes apart (1024 for the high bits of Q6_K)
__device__ __forceinline__ uint32_t column_at(uint32_t lane) { return (lane >> 4) * 2048u + (lane & 15u) * 16u; }

// q[4 h + s]: k-slice s of chunks 2h and 2h + 1
struct Q4Tile { uint4 q[8]; uint4 hdr; };

// Loads come back in the order of their requests: the scales and the pieces of the first four sub-blocks go
// first, so that their products run while the other half of the tile is still on its way.
__device__ __forceinline__ void load_tile(Q4Tile& t, const uint8_t* tile, uint32_t lane) {
    t.hdr = stream_load(tile + 8192 + lane * 16);
    const uint8_t* p = tile + column_at(lane);
#pragma unroll
    for (int i = 0; i < 8; ++i) t.q[i] = stream_load(p + 1024 * (i >> 2) + 256 * (i & 3));
}

__device__ __forceinline__ half8_t as_half8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(half8_t, make_uint4(a, b, c, d));
}

// The operand of a 256-element block: groups 2p and 2p + 1 in a[set][p], A-side block 8 (g % 2) + i holding elements 4i .. 4i + 3
// of group g; one set of four variants for up to two rows, two for three and four.  image: this block's 8 groups of the activation
// image, already offset for this lane.
constexpr int operand_sets(int rows) { return rows > 2 ? 2 : 1; }
template <int R> struct BlockOperand { half4_t a[operand_sets(R)][4]; };
template <int R>
__device__ __forceinline__ uint32_t operand_lane(uint32_t lane) {
    return (lane >> 5) * (256u * operand_sets(R)) + (lane & 3u) * 64u + ((lane >> 2) & 7u) * 8u;
}
template <int R>
__device__ __forceinline__ void load_operand(BlockOperand<R>& o, const uint8_t* __restrict__ image) {
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int set = 0; set < operand_sets(R); ++set)
            o.a[set][p] = __builtin_bit_cast(half4_t, *reinterpret_cast<const uint2*>(image + 512 * operand_sets(R) * p + 256 * set));
}
template <int BLOCK>
__device__ __forceinline__ float4_t mac4(half4_t a, uint32_t b0, uint32_t b1, float4_t c) {
    return __builtin_amdgcn_mfma_f32_4x4x4f16(a, __builtin_bit_cast(half4_t, make_uint2(b0, b1)), c, 4, BLOCK, 0);
}
template <typename F, int... I>
__device__ __forceinline__ void each_slice(F f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }

// mult / xs32: this block's 8 multipliers / 32-sums of row 0 (rows `per_mult` / `per_row` apart)
template <int R>
__device__ __forceinline__ void compute_tile(const Q4Tile& t, const BlockOperand<R>& op,
                                             const float* __restrict__ mult, uint32_t per_mult,
                                             const float* __restrict__ xs32, uint32_t per_row, float (&acc)[R]) {
    const float d = h2f(t.hdr.x & 0xFFFFu), dmin = h2f(t.hdr.x >> 16);
    const uint32_t s0 = t.hdr.y, s1 = t.hdr.z, s2 = t.hdr.w;
    const uint32_t sc_a = s0 & 0x3F3F3F3Fu, mn_a = s1 & 0x3F3F3F3Fu;
    const uint32_t sc_b = (s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u);
    const uint32_t mn_b = ((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u);
    const float d_lo = d * (1.f / 128), d_hi = d * (1.f / 16);  // nibbles enter as 128 q and 16 q
    float mt[R];
#pragma unroll
    for (int r = 0; r < R; ++r) mt[r] = 0.f;
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) {  // 32-byte chunk: sub-blocks 2ch (low nibbles) and 2ch+1 (high)
        float4_t lo[operand_sets(R)], hi[operand_sets(R)];
#pragma unroll
        for (int set = 0; set < operand_sets(R); ++set) lo[set] = hi[set] = zero;
        each_slice([&](auto slice) {
            constexpr int S = slice;
            const uint4 piece = t.q[4 * (ch >> 1) + S];
            const uint32_t w0 = (ch & 1) ? piece.z : piece.x, w1 = (ch & 1) ? piece.w : piece.y;
            // low nibbles sit in bits 7-10 of their half, high ones in bits 4-7 (128 q and 16 q as bit patterns below 2048, which
            // read as n 2^-24): the matrix instruction does not normalise such operands, so a pattern with leading zeros loses
            // that many bits of every product it meets once the products of a sum are aligned.  (Where the low nibbles go costs
            // the same; the high ones further up would take one more shift per word.  Both in bits 4-7: rms error on
            // activations with a 512-fold range, K = 3840, 5.2e-7 of the result's rms.)
            constexpr uint32_t L = 0x07800780u, M = 0x00F000F0u;
            const uint32_t l[4] = {(w0 << 7) & L, (w0 >> 1) & L, (w1 << 7) & L, (w1 >> 1) & L};
            const uint32_t u[4] = {w0 & M, (w0 >> 8) & M, w1 & M, (w1 >> 8) & M};
#pragma unroll
            for (int set = 0; set < operand_sets(R); ++set) {
                lo[set] = mac4<2 * S>(op.a[set][ch], l[0], l[1], lo[set]);
                hi[set] = mac4<8 + 2 * S>(op.a[set][ch], u[0], u[1], hi[set]);
            }
#pragma unroll
            for (int set = 0; set < operand_sets(R); ++set) {
                lo[set] = mac4<2 * S + 1>(op.a[set][ch], l[2], l[3], lo[set]);
                hi[set] = mac4<8 + 2 * S + 1>(op.a[set][ch], u[2], u[3], hi[set]);
            }
        }, std::make_integer_sequence<int, 4>{});
        const uint32_t scw = ch < 2 ? sc_a : sc_b, mnw = ch < 2 ? mn_a : mn_b;
        const float sc_lo = (ch & 1) ? ub2(scw) : ub0(scw), sc_hi = (ch & 1) ? ub3(scw) : ub1(scw);
        const float mn_lo = (ch & 1) ? ub2(mnw) : ub0(mnw), mn_hi = (ch & 1) ? ub3(mnw) : ub1(mnw);
        const float f_lo = d_lo * sc_lo, f_hi = d_hi * sc_hi;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float m_lo = mult[r * per_mult + 2 * ch], m_hi = mult[r * per_mult + 2 * ch + 1];
            acc[r] = fmaf(f_lo * m_lo, lo[r >> 1][2 * (r & 1)] + lo[r >> 1][2 * (r & 1) + 1], acc[r]);
            acc[r] = fmaf(f_hi * m_hi, hi[r >> 1][2 * (r & 1)] + hi[r >> 1][2 * (r & 1) + 1], acc[r]);
            mt[r] = fmaf(mn_lo, xs32[r * per_row + 2 * ch], mt[r]);
            mt[r] = fmaf(mn_hi, xs32[r * per_row + 2 * ch + 1], mt[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = fmaf(-dmin, mt[r], acc[r]);
}

// =======================================================================================
// Q6_K
// =======================================================================================
// Same operand scheme as Q4_K; a scale covers 16 elements, so a 32-group is two chains of four instructions.
// ql[4 n + s]: k-slice s of half n; qh[s]: k-slice s of both halves
struct Q6Tile { uint4 ql[8]; uint4 qh[4]; uint4 sc; uint32_t d; };

// What the first 128 elements need goes first, then the low nibbles of the other half.
__device__ __forceinline__ void load_tile(Q6Tile& t, const uint8_t* tile, uint32_t lane) {
    const uint8_t* p = tile + column_at(lane);
    const uint8_t* ph = tile + 8192 + (lane >> 4) * 1024u + (lane & 15u) * 16u;
    t.sc = *reinterpret_cast<const uint4*>(tile + 12288 + lane * 16);
    t.d = *reinterpret_cast<const uint16_t*>(tile + 13312 + lane * 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) { t.ql[i] = stream_load(p + 256 * i); t.qh[i] = stream_load(ph + 256 * i); }
#pragma unroll
    for (int i = 4; i < 8; ++i) t.ql[i] = stream_load(p + 1024 + 256 * (i & 3));
}

__device__ __forceinline__ float sbyte(uint32_t w, int i) {
    return i == 0 ? sb0(w) : i == 1 ? sb1(w) : i == 2 ? sb2(w) : sb3(w);
}

template <int R>
__device__ __forceinline__ void compute_tile(const Q6Tile& t, const BlockOperand<R>& op,
                                             const float* __restrict__ mult, uint32_t per_mult,
                                             const float* __restrict__ xs16, uint32_t per_row, float (&acc)[2][R]) {
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
    float part[2][R], off[2][R];   // of the first and of the second halves of the groups: two sums half as long
#pragma unroll
    for (int r = 0; r < R; ++r) part[0][r] = part[1][r] = off[0][r] = off[1][r] = 0.f;
    each_slice([&](auto group) {  // 32-element group: half n, quadrant qd
        constexpr int G = group, n = G >> 2, qd = G & 3, ls = qd >= 2 ? 4 : 0, AT = 8 * (G & 1);
        float4_t first[operand_sets(R)], second[operand_sets(R)];
#pragma unroll
        for (int set = 0; set < operand_sets(R); ++set) first[set] = second[set] = zero;
        auto slice_operand = [&](int s, uint32_t (&b)[4]) {
            const uint4 lq = t.ql[4 * n + s], hq = t.qh[s];
            const uint32_t w[2] = {(qd & 1) ? lq.z : lq.x, (qd & 1) ? lq.w : lq.y};
            const uint32_t h[2] = {n ? hq.z : hq.x, n ? hq.w : hq.y};
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                // the 6-bit quant sits in bits 4-9 of its half (16 q as a bit pattern: see the Q4_K tile)
                const uint32_t lo0 = (ls ? w[k] : w[k] << 4) & 0x00F000F0u, lo1 = (w[k] >> (ls + 4)) & 0x00F000F0u;
                // 2-bit field of quadrant qd moved to bits 8-9 of each half
                const uint32_t hs0 = h[k] << (8 - 2 * qd), hs1 = qd == 0 ? h[k] : h[k] >> (2 * qd);
                b[2 * k] = (hs0 & 0x03000300u) | lo0;
                b[2 * k + 1] = (hs1 & 0x03000300u) | lo1;
            }
        };
        each_slice([&](auto slice) {   // slices s (first 16 elements) and s + 2 (second)
            constexpr int S = slice;
            uint32_t b[4], c[4];
            slice_operand(S, b);
            slice_operand(S + 2, c);
#pragma unroll
            for (int set = 0; set < operand_sets(R); ++set) {
                first[set] = mac4<AT + 2 * S>(op.a[set][G >> 1], b[0], b[1], first[set]);
                second[set] = mac4<AT + 2 * S + 4>(op.a[set][G >> 1], c[0], c[1], second[set]);
            }
#pragma unroll
            for (int set = 0; set < operand_sets(R); ++set) {
                first[set] = mac4<AT + 2 * S + 1>(op.a[set][G >> 1], b[2], b[3], first[set]);
                second[set] = mac4<AT + 2 * S + 5>(op.a[set][G >> 1], c[2], c[3], second[set]);
            }
        }, std::make_integer_sequence<int, 2>{});
        const uint32_t wv = (G >> 1) == 0 ? t.sc.x : (G >> 1) == 1 ? t.sc.y : (G >> 1) == 2 ? t.sc.z : t.sc.w;
        const float s_first = sbyte(wv, 2 * (G & 1)), s_second = sbyte(wv, 2 * (G & 1) + 1);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float m = mult[r * per_mult + G];
            part[0][r] = fmaf(s_first * m, first[r >> 1][2 * (r & 1)] + first[r >> 1][2 * (r & 1) + 1], part[0][r]);
            part[1][r] = fmaf(s_second * m, second[r >> 1][2 * (r & 1)] + second[r >> 1][2 * (r & 1) + 1], part[1][r]);
            off[0][r] = fmaf(s_first, xs16[r * per_row + 2 * G], off[0][r]);
            off[1][r] = fmaf(s_second, xs16[r * per_row + 2 * G + 1], off[1][r]);
        }
    }, std::make_integer_sequence<int, 8>{});
    const float d = h2f(t.d);
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[half][r] = fmaf(d, fmaf(-32.0f, off[half][r], 0.0625f * part[half][r]), acc[half][r]);
}

// =======================================================================================
// Q8_0
// =======================================================================================
// One 32-element block per MFMA and column group; the int8 quants enter biased by 128 as fp16
// subnormals, the bias comes back through the 32-sum.
struct Q8Tile { uint4 q[2]; uint32_t d; };

__device__ __forceinline__ void load_tile(Q8Tile& t, const uint8_t* p, uint32_t lane) {
    t.q[0] = stream_load(p);
    t.q[1] = stream_load(p + 1024);
    t.d = *reinterpret_cast<const uint16_t*>(p - lane * 16 + 2048 + lane * 2);
}

template <int R>
__device__ __forceinline__ void compute_tile(const Q8Tile& t, const half8_t a,
                                             const float* __restrict__ mult, uint32_t per_mult,
                                             const float* __restrict__ xs32, uint32_t per_row,
                                             uint32_t lane_group, float (&acc)[R]) {
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
    float4_t own = zero;
#pragma unroll
    for (int cg = 0; cg < 4; ++cg) {
        const uint4 piece = t.q[cg >> 1];
        const uint32_t w0 = ((cg & 1) ? piece.z : piece.x) ^ 0x80808080u, w1 = ((cg & 1) ? piece.w : piece.y) ^ 0x80808080u;
        // the biased byte sits in bits 3-10 of its half (8 (q + 128) as a bit pattern: see the Q4_K tile)
        const float4_t d4 = __builtin_amdgcn_mfma_f32_16x16x32_f16(
            a, as_half8(even_bytes(w0) << 3, odd_bytes(w0) << 3, even_bytes(w1) << 3, odd_bytes(w1) << 3), zero, 0, 0, 0);
        if (lane_group == uint32_t(cg)) own = d4;
    }
    const float d = h2f(t.d);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float v = fmaf(0.125f * mult[r * per_mult], own[2 * r] + own[2 * r + 1], -128.0f * xs32[r * per_row]);
        acc[r] = fmaf(d, v, acc[r]);
    }
}

// =======================================================================================
// The streaming kernel: one wave = one (column tile, k-slice)
// =======================================================================================
// One wave: `count` consecutive blocks of one column tile, the first at `tiles` (its 64 x block bytes),
// against the operand blocks ob0 .. ob0 + count - 1 of the receipt `xsums` (a blob laid out for R rows
// of K activations, in global memory or in LDS); returns the per-lane column sums.
// How a wave walks its blocks.  Ahead: the next block's tile and operand are requested before a block's products (two tiles in
// registers).  One: the run has at most one block.  Serial: one tile in registers at a time.
constexpr int kWalkAhead = 0, kWalkOne = 1, kWalkSerial = 2;
template <int DTYPE, int R, int WALK = kWalkAhead>
__device__ __forceinline__ void run_blocks_at(const uint8_t* __restrict__ tiles, const float* __restrict__ xsums,
                                              uint32_t K, uint32_t ob0, uint32_t count, float (&acc)[R],
                                              uint32_t lane = threadIdx.x & 63) {
    constexpr uint32_t TB = kTileCols * block_bytes(DTYPE);
    const uint32_t n16 = K / 16, per_row = n16 + K / 32;
    // Q6_K consumes 16-sums (16 per block), Q4_K 32-sums (8 per block), Q8_0 one 32-sum per block
    const float* xs = DTYPE == GUFFIN_Q6_K ? xsums : xsums + n16;
    const uint8_t* tp = tiles + lane * 16;
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.f;
    const ReceiptLayout L = receipt_layout(R, K);
    const uint8_t* blob = reinterpret_cast<const uint8_t*>(xsums);
    const float* mult = reinterpret_cast<const float*>(blob + L.mult_off);
    // lane (i = lane % 16, s = lane / 16) of the A operand: variant i % 4, k-slice s
    const uint8_t* image = blob + L.image_off + (lane & 3u) * 64u + (lane >> 4) * 16u;
    const uint32_t ob1 = ob0 + count;
    if constexpr (DTYPE != GUFFIN_Q8_0) {
        using Tile = std::conditional_t<DTYPE == GUFFIN_Q4_K, Q4Tile, Q6Tile>;
        constexpr uint32_t xs_block = DTYPE == GUFFIN_Q4_K ? 8 : 16;
        constexpr uint32_t image_block = 2048u * operand_sets(R);
        const uint8_t* im = blob + L.image_off + operand_lane<R>(lane);
        float halves[2][R];   // Q6_K
        auto product = [&](const Tile& t, const BlockOperand<R>& o, uint32_t b) {
            const float *mb = mult + b * 8u, *xb = xs + b * xs_block;
            if constexpr (DTYPE == GUFFIN_Q6_K) compute_tile<R>(t, o, mb, K / 32, xb, per_row, halves);
            else compute_tile<R>(t, o, mb, K / 32, xb, per_row, acc);
        };
        if constexpr (DTYPE == GUFFIN_Q6_K) {
#pragma unroll
            for (int r = 0; r < R; ++r) halves[0][r] = halves[1][r] = 0.f;
        }
        // a block's operand (a hit in the caches) is requested ahead of its weight tile, which comes from HBM:
        // behind it it would cost the wave a second trip before its first product
        if constexpr (WALK == kWalkSerial) {
            for (uint32_t b = ob0; b < ob1; ++b) {
                Tile cur;
                BlockOperand<R> op;
                load_operand<R>(op, im + size_t(b) * image_block);
                load_tile(cur, tiles + size_t(b - ob0) * TB, lane);
                product(cur, op, b);
            }
        } else if (WALK == kWalkOne || count <= 1) {
            if (count) {
                Tile only;
                BlockOperand<R> op;
                load_operand<R>(op, im + size_t(ob0) * image_block);
                load_tile(only, tiles, lane);
                product(only, op, ob0);
            }
        } else {
            // Two tiles by name, and a copy of the products for the run's end: behind a branch around the next block's requests the
            // compiler has to count as if they had not been made, and a block waits for the next one's tile; copied from one name
            // to the other, it waits for all of it.
            Tile even, odd;
            BlockOperand<R> even_op, odd_op;
            auto request = [&](Tile& t, BlockOperand<R>& o, uint32_t b) {
                load_operand<R>(o, im + size_t(b) * image_block);
                load_tile(t, tiles + size_t(b - ob0) * TB, lane);
                __builtin_amdgcn_sched_barrier(0);
            };
            request(even, even_op, ob0);
            for (uint32_t b = ob0;; b += 2) {   // (two blocks at least)
                request(odd, odd_op, b + 1);
                product(even, even_op, b);
                if (b + 2 >= ob1) { product(odd, odd_op, b + 1); break; }
                request(even, even_op, b + 2);
                product(odd, odd_op, b + 1);
                if (b + 3 >= ob1) { product(even, even_op, b + 2); break; }
            }
        }
        if constexpr (DTYPE == GUFFIN_Q6_K) {
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r] = halves[0][r] + halves[1][r];
        }
    } else {
        Q8Tile cur, nxt;
        auto operand = [&](uint32_t b) { return __builtin_bit_cast(half8_t, *reinterpret_cast<const uint4*>(image + size_t(b) * 256u)); };
        half8_t a = {}, an = {};
        if (count) { a = operand(ob0); load_tile(cur, tp, lane); }
        for (uint32_t b = ob0; b < ob1; ++b) {
            if (b + 1 < ob1) { an = operand(b + 1); load_tile(nxt, tp + size_t(b + 1 - ob0) * TB, lane); }
            compute_tile<R>(cur, a, mult + b, K / 32, xs + b, per_row, lane >> 4, acc);
            cur = nxt;
            a = an;
        }
    }
}

// The first two Q8_0 tiles of a wave's run, requested ahead of time (before a wait that the operand needs
// and the weights do not), and the run itself starting from them.
struct Q8Ahead { Q8Tile t[2]; };

__device__ __forceinline__ void load_ahead(Q8Ahead& ahead, const uint8_t* __restrict__ tiles, uint32_t count, uint32_t lane) {
    constexpr uint32_t TB = kTileCols * block_bytes(GUFFIN_Q8_0);
    const uint8_t* tp = tiles + lane * 16;
    ahead.t[0] = Q8Tile{};
    ahead.t[1] = Q8Tile{};
    if (count > 0) load_tile(ahead.t[0], tp, lane);
    if (count > 1) load_tile(ahead.t[1], tp + TB, lane);
}

template <int R>
__device__ __forceinline__ void run_blocks_ahead(const Q8Ahead& ahead, const uint8_t* __restrict__ tiles,
                                                 const float* __restrict__ xsums, uint32_t K, uint32_t ob0, uint32_t count,
                                                 float (&acc)[R], uint32_t lane = threadIdx.x & 63) {
    constexpr uint32_t TB = kTileCols * block_bytes(GUFFIN_Q8_0);
    const uint32_t n16 = K / 16, per_row = n16 + K / 32;
    const float* xs = xsums + n16;
    const uint8_t* tp = tiles + lane * 16;
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.f;
    const ReceiptLayout L = receipt_layout(R, K);
    const uint8_t* blob = reinterpret_cast<const uint8_t*>(xsums);
    const float* mult = reinterpret_cast<const float*>(blob + L.mult_off);
    const uint8_t* image = blob + L.image_off + (lane & 3u) * 64u + (lane >> 4) * 16u;
    const uint32_t ob1 = ob0 + count;
    auto operand = [&](uint32_t b) { return __builtin_bit_cast(half8_t, *reinterpret_cast<const uint4*>(image + size_t(b) * 256u)); };
    Q8Tile cur = ahead.t[0], nxt = ahead.t[1], far = Q8Tile{};
    half8_t a = {}, an = {};
    if (count) a = operand(ob0);
    for (uint32_t b = ob0; b < ob1; ++b) {
        if (b + 1 < ob1) an = operand(b + 1);
        if (b + 2 < ob1) load_tile(far, tp + size_t(b + 2 - ob0) * TB, lane);
        compute_tile<R>(cur, a, mult + b, K / 32, xs + b, per_row, lane >> 4, acc);
        cur = nxt;
        nxt = far;
        a = an;
    }
}

// One wave: blocks [b0, b1) of column tile `ct` of a whole matrix whose operand is the receipt of its K inputs.
template <int DTYPE, int R, int WALK = kWalkAhead>
__device__ __forceinline__ void run_blocks(const uint8_t* __restrict__ wt, const float* __restrict__ xsums, uint32_t K, uint32_t nblk,
                                           uint32_t ct, uint32_t b0, uint32_t b1, float (&acc)[R]) {
    constexpr uint32_t TB = kTileCols * block_bytes(DTYPE);
    run_blocks_at<DTYPE, R, WALK>(wt + (size_t(ct) * nblk + b0) * TB, xsums, K, b0, b1 > b0 ? b1 - b0 : 0u, acc);
}

}  // namespace
}  // namespace guffin
