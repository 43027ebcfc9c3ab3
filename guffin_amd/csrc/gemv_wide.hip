// The streaming product for 3 and 4 rows (verify trees, the shortest prompt runs).
//
// Same tiles, operands and arithmetic as the kernels of gemv_packed.hip.  There the 16 rows of the matrix instruction's A side
// hold the 4 variants (hi, lo of two rows) four times over, so that every lane group finds the sums of its own column group;
// with four rows the 8 variants are there twice, and the matrix instructions of a tile stay the same in number:
//   Q4_K, Q8_0   lane (j, g): rows 2 (g % 2) and + 1, columns 32 (g / 2) + j and + 16
//   Q6_K         the two halves of a 32-group take the place of the repetition: lane (j, g): rows 2 (g % 2) and + 1, the
//                16-element half g / 2, columns j, j + 16, j + 32, j + 48; the halves are added across lanes at the end
// So a weight byte is fetched and unpacked once for four rows where two passes of two rows do it twice, and the launch is bound by
// the weight stream and its ramp as before.  Eight waves a workgroup: a lane holds two tiles, which is more than the 128
// registers sixteen waves would leave it.
// Blocks of a 12B-shaped stack, four rows, one launch here / two launches of two rows (us): q/k/v 9.1 / 16.6, o 5.3 / 9.9,
// gate + up 19.6 / 34, down 15.5 / 26, the 262144-row head 144 / 286.
// Three rows leave the last pair of variants zero and its row unwritten.
#include "common.hpp"
#include "receipt.hpp"
#include "gemv_tiles.hpp"

#include <type_traits>

namespace guffin {
namespace {

constexpr uint32_t kWideWaves = 8;
constexpr int kWideMixed = 3;   // Q4_K and Q6_K matrices in one launch

__host__ __device__ constexpr int wide_cols(int dtype) { return dtype == GUFFIN_Q6_K ? 4 : 2; }

// ---- the operand of a block, in LDS -----------------------------------------------------------------------------
// Every wave copies its blocks' operand into LDS two blocks deep with the memory-to-LDS path, ahead of the tiles: operand loads
// into registers come back behind the next tile's (loads return in order), which made every 32-group of a Q6_K tile wait for
// HBM (down projection 23 us against 15.5, q/k/v 11.6 against 9.1, head 218 against 144), and eight of them per block is what a lane has no registers for.
//   [0, 4096)     the block's eight groups of the image, 8 variants of 64 bytes each
//   [4096, ..)    Q4_K: mult[4][8], sums of 32 [4][8];  Q6_K: sums of 16 [4][16], mult[4][8] (twice: the load is a whole wave's)
constexpr uint32_t kSlotBytes = 4608;
constexpr uint32_t kWideLds = kWideWaves * 2 * kSlotBytes;
template <int DTYPE> constexpr uint32_t operand_loads() { return DTYPE == GUFFIN_Q6_K ? 6 : 5; }

__device__ __forceinline__ void to_lds(__amdgpu_buffer_rsrc_t r, uint8_t* to, uint32_t lane_off, uint32_t uniform_off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)to, 16, static_cast<int>(lane_off), static_cast<int>(uniform_off), 0, 0);
}
__device__ __forceinline__ void to_lds4(__amdgpu_buffer_rsrc_t r, uint8_t* to, uint32_t lane_off, uint32_t uniform_off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)to, 4, static_cast<int>(lane_off), static_cast<int>(uniform_off), 0, 0);
}

// where a lane's words of a block's multipliers and sums are, from the start of the receipt
struct OperandAt { uint32_t image, words, mult; };
template <int DTYPE>
__device__ __forceinline__ OperandAt operand_at(const ReceiptLayout& L, uint32_t K, uint32_t lane) {
    const uint32_t n16 = K / 16, n32 = K / 32, per_row = n16 + n32, l = lane & 31u;
    const uint32_t mult = static_cast<uint32_t>(L.mult_off) + ((l >> 3) * n32 + (l & 7u)) * 4;
    if constexpr (DTYPE == GUFFIN_Q6_K) return {static_cast<uint32_t>(L.image_off), ((lane >> 4) * per_row + (lane & 15u)) * 4, mult};
    return {static_cast<uint32_t>(L.image_off), lane < 32 ? mult : ((l >> 3) * per_row + n16 + (l & 7u)) * 4, 0};
}
template <int DTYPE>
__device__ __forceinline__ void stage_operand(__amdgpu_buffer_rsrc_t r, const OperandAt& at, uint8_t* slot, uint32_t b, uint32_t lane) {
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) to_lds(r, slot + 1024 * i, lane * 16, at.image + b * 4096 + 1024 * i);
    to_lds4(r, slot + 4096, at.words, b * (DTYPE == GUFFIN_Q6_K ? 64 : 32));
    if constexpr (DTYPE == GUFFIN_Q6_K) to_lds4(r, slot + 4352, at.mult, b * 32);
}
// The order of requests is what the counts below rely on: nothing moves across.
__device__ __forceinline__ void fence_order() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
template <uint32_t N>
__device__ __forceinline__ void wait_younger() {   // all but the N youngest requests are back
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// The sums are wanted here: left to itself the compiler puts off a tile's products to its end, and holds them all till then.
template <int C>
__device__ __forceinline__ void keep_here(float (&v)[C][2]) {
#pragma unroll
    for (int c = 0; c < C; ++c) asm volatile("" : "+v"(v[c][0]), "+v"(v[c][1]));
    __builtin_amdgcn_sched_barrier(0);
}

struct Q4Wide { uint4 q[8]; uint4 hdr[2]; };

__device__ __forceinline__ void load_tile(Q4Wide& t, const uint8_t* p, uint32_t lane) {
    const uint8_t* hdr = p - lane * 16 + 8192 + (32u * (lane >> 5) + (lane & 15u)) * 16;
    t.hdr[0] = stream_load(hdr);
    t.hdr[1] = stream_load(hdr + 256);
#pragma unroll
    for (int i = 0; i < 8; i += 2) t.q[i] = stream_load(p + 1024 * i);
#pragma unroll
    for (int i = 1; i < 8; i += 2) t.q[i] = stream_load(p + 1024 * i);
}

__device__ __forceinline__ void compute_tile(const Q4Wide& t, const uint8_t* slot, uint32_t lane, float (&acc)[2][2]) {
    const bool upper = lane >= 32;
    const uint8_t* image = slot + (lane & 7u) * 64 + (lane >> 4) * 16;   // lane (i, s): variant i % 8, k-slice s
    const float* words = reinterpret_cast<const float*>(slot + 4096) + ((lane >> 4) & 1u) * 16;   // this lane's pair of rows
    float d_q[2], dmin[2], mt[2][2];
    uint32_t sc_a[2], mn_a[2], sc_b[2], mn_b[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const uint32_t s0 = t.hdr[c].y, s1 = t.hdr[c].z, s2 = t.hdr[c].w;
        d_q[c] = h2f(t.hdr[c].x & 0xFFFFu) * 0.0625f;   // nibbles enter as 16 q
        dmin[c] = h2f(t.hdr[c].x >> 16);
        sc_a[c] = s0 & 0x3F3F3F3Fu; mn_a[c] = s1 & 0x3F3F3F3Fu;
        sc_b[c] = (s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u);
        mn_b[c] = ((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u);
        mt[c][0] = mt[c][1] = 0.f;
    }
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) {
        float4_t lo[2] = {zero, zero}, hi[2] = {zero, zero};
        const half8_t a_lo = *reinterpret_cast<const half8_t*>(image + 1024 * ch), a_hi = *reinterpret_cast<const half8_t*>(image + 1024 * ch + 512);
        float2 mult[2], xs32[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            mult[r] = *reinterpret_cast<const float2*>(words + 8 * r + 2 * ch);
            xs32[r] = *reinterpret_cast<const float2*>(words + 32 + 8 * r + 2 * ch);
        }
#pragma unroll
        for (int cg = 0; cg < 4; ++cg) {
            const uint4 piece = t.q[2 * cg + (ch >> 1)];
            const uint32_t w0 = (ch & 1) ? piece.z : piece.x, w1 = (ch & 1) ? piece.w : piece.y;
            constexpr uint32_t M = 0x00F000F0u;   // 16 q: see the two-row tile
            const half8_t blo = as_half8((w0 << 4) & M, (w0 >> 4) & M, (w1 << 4) & M, (w1 >> 4) & M);
            const half8_t bhi = as_half8(w0 & M, (w0 >> 8) & M, w1 & M, (w1 >> 8) & M);
            const float4_t dlo = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_lo, blo, zero, 0, 0, 0);
            const float4_t dhi = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_hi, bhi, zero, 0, 0, 0);
            if (upper == (cg >= 2)) { lo[cg & 1] = dlo; hi[cg & 1] = dhi; }
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const uint32_t scw = ch < 2 ? sc_a[c] : sc_b[c], mnw = ch < 2 ? mn_a[c] : mn_b[c];
            const float f_lo = d_q[c] * ((ch & 1) ? ub2(scw) : ub0(scw)), f_hi = d_q[c] * ((ch & 1) ? ub3(scw) : ub1(scw));
            const float mn_lo = (ch & 1) ? ub2(mnw) : ub0(mnw), mn_hi = (ch & 1) ? ub3(mnw) : ub1(mnw);
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                acc[c][r] = fmaf(f_lo * mult[r].x, lo[c][2 * r] + lo[c][2 * r + 1], acc[c][r]);
                acc[c][r] = fmaf(f_hi * mult[r].y, hi[c][2 * r] + hi[c][2 * r + 1], acc[c][r]);
                mt[c][r] = fmaf(mn_lo, xs32[r].x, mt[c][r]);
                mt[c][r] = fmaf(mn_hi, xs32[r].y, mt[c][r]);
            }
        }
        keep_here(acc);
        keep_here(mt);
    }
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 2; ++r) acc[c][r] = fmaf(-dmin[c], mt[c][r], acc[c][r]);
}

// sc: the eight scales of the lane's half of every group of a column; d: the columns' in pairs
struct Q6Wide { uint4 ql[8]; uint4 qh[4]; uint4 sc[4]; uint32_t d[4]; };

__device__ __forceinline__ void load_tile(Q6Wide& t, const uint8_t* p, uint32_t lane) {
#pragma unroll
    for (int i = 0; i < 8; ++i) t.ql[i] = stream_load(p + 1024 * i);
#pragma unroll
    for (int i = 0; i < 4; ++i) t.qh[i] = stream_load(p + 8192 + 1024 * i);
    const uint8_t* base = p - lane * 16;
    const uint32_t col = lane & 15u;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        t.sc[c] = *reinterpret_cast<const uint4*>(base + 12288 + (col + 16 * c) * 16);
        t.d[c] = *reinterpret_cast<const uint16_t*>(base + 13312 + (col + 16 * c) * 2);
    }
}

__device__ __forceinline__ void compute_tile(const Q6Wide& t, const uint8_t* slot, uint32_t lane, float (&acc)[4][2]) {
    const uint8_t* image = slot + (lane & 7u) * 64 + (lane >> 4) * 16;
    // A rows 0-7 see the first 16 elements of a group, rows 8-15 the second 16
    const uint32_t keep = ((lane & 15u) >> 3) == (lane >> 5) ? 0xFFFFFFFFu : 0u;
    const float* xs16 = reinterpret_cast<const float*>(slot + 4096) + ((lane >> 4) & 1u) * 32 + (lane >> 5);
    const float* mult = reinterpret_cast<const float*>(slot + 4352) + ((lane >> 4) & 1u) * 16;
    const bool second = lane >= 32;   // the 16-element half this lane's sums cover
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
    float part[4][2];
#pragma unroll
    for (int c = 0; c < 4; ++c) part[c][0] = part[c][1] = 0.f;
#pragma unroll
    for (int g = 0; g < 8; ++g) {
        const int n = g >> 2, qd = g & 3;
        uint4 av = *reinterpret_cast<const uint4*>(image + 512 * g);
        float m[2], s16[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) { m[r] = 0.0625f * mult[8 * r + g]; s16[r] = -32.0f * xs16[16 * r + 2 * g]; }
        av.x &= keep; av.y &= keep; av.z &= keep; av.w &= keep;
        const half8_t a = __builtin_bit_cast(half8_t, av);
#pragma unroll
        for (int cg = 0; cg < 4; ++cg) {
            const uint4 lq = t.ql[2 * cg + n], hq = t.qh[cg];
            const uint32_t w0 = (qd & 1) ? lq.z : lq.x, w1 = (qd & 1) ? lq.w : lq.y;
            const uint32_t h0 = n ? hq.z : hq.x, h1 = n ? hq.w : hq.y;
            const int ls = qd >= 2 ? 4 : 0;
            uint32_t b[4];
#pragma unroll
            for (int k = 0; k < 2; ++k) {   // 16 q: see the two-row tile
                const uint32_t w = k ? w1 : w0, h = k ? h1 : h0;
                const uint32_t lo0 = (ls ? w : w << 4) & 0x00F000F0u, lo1 = (w >> (ls + 4)) & 0x00F000F0u;
                b[2 * k] = ((h << (8 - 2 * qd)) & 0x03000300u) | lo0;
                b[2 * k + 1] = ((qd == 0 ? h : h >> (2 * qd)) & 0x03000300u) | lo1;
            }
            const float4_t D = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, as_half8(b[0], b[1], b[2], b[3]), zero, 0, 0, 0);
            const int word = g >> 1;
            const uint32_t wv = word == 0 ? t.sc[cg].x : word == 1 ? t.sc[cg].y : word == 2 ? t.sc[cg].z : t.sc[cg].w;
            const float sc = sbyte(second ? wv >> 8 : wv, 2 * (g & 1));
#pragma unroll
            for (int r = 0; r < 2; ++r)   // scale (q - 32): the offset taken off inside the half, 16 q as 16 q
                part[cg][r] = fmaf(sc, fmaf(m[r], D[2 * r] + D[2 * r + 1], s16[r]), part[cg][r]);
        }
        keep_here(part);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float d = h2f(t.d[c]);
#pragma unroll
        for (int r = 0; r < 2; ++r) acc[c][r] = fmaf(d, part[c][r], acc[c][r]);
    }
}

struct Q8Wide { uint4 q[2]; uint32_t d[2]; };

__device__ __forceinline__ void load_tile(Q8Wide& t, const uint8_t* p, uint32_t lane) {
    t.q[0] = stream_load(p);
    t.q[1] = stream_load(p + 1024);
    const uint8_t* d = p - lane * 16 + 2048 + (32u * (lane >> 5) + (lane & 15u)) * 2;
    t.d[0] = *reinterpret_cast<const uint16_t*>(d);
    t.d[1] = *reinterpret_cast<const uint16_t*>(d + 32);
}

__device__ __forceinline__ void compute_tile(const Q8Wide& t, const half8_t a, const float (&mult)[2], const float (&xs32)[2], uint32_t lane,
                                             float (&acc)[2][2]) {
    const bool upper = lane >= 32;
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
    float4_t own[2] = {zero, zero};
#pragma unroll
    for (int cg = 0; cg < 4; ++cg) {
        const uint4 piece = t.q[cg >> 1];
        const uint32_t w0 = ((cg & 1) ? piece.z : piece.x) ^ 0x80808080u, w1 = ((cg & 1) ? piece.w : piece.y) ^ 0x80808080u;
        const float4_t d4 = __builtin_amdgcn_mfma_f32_16x16x32_f16(
            a, as_half8(even_bytes(w0) << 3, odd_bytes(w0) << 3, even_bytes(w1) << 3, odd_bytes(w1) << 3), zero, 0, 0, 0);
        if (upper == (cg >= 2)) own[cg & 1] = d4;
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const float d = h2f(t.d[c]);
#pragma unroll
        for (int r = 0; r < 2; ++r)
            acc[c][r] = fmaf(d, fmaf(0.125f * mult[r], own[c][2 * r] + own[c][2 * r + 1], -128.0f * xs32[r]), acc[c][r]);
    }
}

// One wave: blocks [b0, b1) of column tile `ct` against the receipt of four rows of K activations, staged in the wave's two
// slots.  The sums come back per lane: columns and rows as the head of this file says.
template <int DTYPE>
__device__ __forceinline__ void run_wide(const uint8_t* __restrict__ wt, const float* __restrict__ xsums, uint32_t K, uint32_t nblk,
                                         uint32_t ct, uint32_t b0, uint32_t b1, uint8_t* slots, uint32_t lane, float (&acc)[wide_cols(DTYPE)][2]) {
    constexpr uint32_t TB = kTileCols * block_bytes(DTYPE);
    constexpr int C = wide_cols(DTYPE);
    const ReceiptLayout L = receipt_layout(kWideRows, K);
    const uint8_t* tp = wt + (size_t(ct) * nblk + b0) * TB + lane * 16;
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c][0] = acc[c][1] = 0.f;
    if constexpr (DTYPE != GUFFIN_Q8_0) {
        using Tile = std::conditional_t<DTYPE == GUFFIN_Q4_K, Q4Wide, Q6Wide>;
        constexpr uint32_t tile_loads = DTYPE == GUFFIN_Q4_K ? 10 : 20;
        const __amdgpu_buffer_rsrc_t blob = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(xsums), 0, static_cast<int>(L.bytes), 0x00020000);
        const OperandAt at = operand_at<DTYPE>(L, K, lane);
        Tile even, odd;
        // block b, its tile in `now`: the next block's operand and tile are requested first.  (Two tiles by name and a loop of two
        // blocks: a copy from one to the other at the end of a block waits for every load of the copied one.)
        auto block = [&](Tile& now, Tile& next, uint32_t b, uint32_t at_slot) {
            if (b + 1 < b1) {
                // (the other slot was last read for block b - 1, whose products have been formed)
                stage_operand<DTYPE>(blob, at, slots + (1u - at_slot) * kSlotBytes, b + 1, lane);
                fence_order();
                load_tile(next, tp + size_t(b + 1 - b0) * TB, lane);
                wait_younger<tile_loads + operand_loads<DTYPE>() + tile_loads>();   // the operand of block b; its tile is waited for piece by piece
            } else {
                wait_younger<tile_loads>();
            }
            compute_tile(now, slots + at_slot * kSlotBytes, lane, acc);
        };
        if (b0 < b1) {
            stage_operand<DTYPE>(blob, at, slots, b0, lane);
            fence_order();
            load_tile(even, tp, lane);
            fence_order();
        }
        for (uint32_t b = b0; b < b1; b += 2) {
            block(even, odd, b, 0);
            if (b + 1 < b1) block(odd, even, b + 1, 1);
        }
    } else {
        const uint32_t n16 = K / 16, n32 = K / 32, per_row = n16 + n32, pair = (lane >> 4) & 1u;
        const uint8_t* base = reinterpret_cast<const uint8_t*>(xsums);
        const float* mult = reinterpret_cast<const float*>(base + L.mult_off) + 2 * pair * size_t(n32);
        const float* xs = xsums + 2 * pair * size_t(per_row) + n16;
        const uint8_t* image = base + L.image_off + (lane & 7u) * 64u + (lane >> 4) * 16u;
        Q8Wide cur, nxt;
        if (b0 < b1) load_tile(cur, tp, lane);
        for (uint32_t b = b0; b < b1; ++b, tp += TB) {
            const half8_t a = __builtin_bit_cast(half8_t, *reinterpret_cast<const uint4*>(image + size_t(b) * 512u));
            const float m[2] = {mult[b], mult[n32 + b]}, x[2] = {xs[b], xs[per_row + b]};
            if (b + 1 < b1) load_tile(nxt, tp + TB, lane);
            compute_tile(cur, a, m, x, lane, acc);
            cur = nxt;
        }
    }
    if constexpr (DTYPE == GUFFIN_Q6_K) {
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int r = 0; r < 2; ++r) acc[c][r] += __shfl_xor(acc[c][r], 32, kWave);
    }
}

// A wave's sums to red[row][64 columns].  Q6_K: either half of the wave holds all four columns and writes two of them.
template <int C>
__device__ __forceinline__ void put_sums(const float (&acc)[C][2], float* red, uint32_t lane) {
    const uint32_t j = lane & 15u, half = lane >> 5, pair = (lane >> 4) & 1u;
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const float v = C == 2 ? acc[c][r] : half ? acc[C / 2 + c][r] : acc[c][r];
            red[(2 * pair + r) * 64 + 32 * half + 16 * c + j] = v;
        }
}

struct WideCfg { uint32_t K, nblk, bps, W, rows; };
struct WideMeta { const uint8_t* tiles[3]; float* part[3]; uint32_t N[3], dtype[3], tile_end[3]; };

// Up to three matrices of the same rows, their column tiles side by side along grid x; grid y: planes.
template <int MODE>
__global__ void __launch_bounds__(64 * kWideWaves)
gemv_wide_kernel(const float* __restrict__ xsums, const WideMeta m, const WideCfg c) {
    extern __shared__ __attribute__((aligned(256))) uint8_t lds[];   // the waves' operand slots, then their sums
    const uint32_t which = blockIdx.x >= m.tile_end[1] ? 2u : blockIdx.x >= m.tile_end[0] ? 1u : 0u;
    const uint8_t* wt = which == 0 ? m.tiles[0] : which == 1 ? m.tiles[1] : m.tiles[2];
    float* part = which == 0 ? m.part[0] : which == 1 ? m.part[1] : m.part[2];
    const uint32_t N = which == 0 ? m.N[0] : which == 1 ? m.N[1] : m.N[2];
    [[maybe_unused]] const uint32_t dtype = which == 0 ? m.dtype[0] : which == 1 ? m.dtype[1] : m.dtype[2];
    const uint32_t ct = blockIdx.x - (which == 0 ? 0u : which == 1 ? m.tile_end[0] : m.tile_end[1]);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t slice = blockIdx.y * c.W + wave, b0 = min(slice * c.bps, c.nblk), b1 = min(b0 + c.bps, c.nblk);
    uint8_t* slots = lds + wave * 2 * kSlotBytes;
    float* red = reinterpret_cast<float*>(lds);
    auto finish = [&](const auto& acc) {
        __syncthreads();   // the slots are done with
        put_sums(acc, red + wave * kWideRows * 64, lane);
    };
    if constexpr (MODE == kWideMixed) {
        if (dtype == GUFFIN_Q4_K) {
            float acc[wide_cols(GUFFIN_Q4_K)][2];
            run_wide<GUFFIN_Q4_K>(wt, xsums, c.K, c.nblk, ct, b0, b1, slots, lane, acc);
            finish(acc);
        } else {
            float acc[wide_cols(GUFFIN_Q6_K)][2];
            run_wide<GUFFIN_Q6_K>(wt, xsums, c.K, c.nblk, ct, b0, b1, slots, lane, acc);
            finish(acc);
        }
    } else {
        float acc[wide_cols(MODE)][2];
        run_wide<MODE>(wt, xsums, c.K, c.nblk, ct, b0, b1, slots, lane, acc);
        finish(acc);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < c.rows * 64; i += blockDim.x) {
        float t = red[i];
        for (uint32_t w = 1; w < c.W; ++w) t += red[w * kWideRows * 64 + i];
        part[(size_t(blockIdx.y) * c.rows + (i >> 6)) * N + ct * kTileCols + (i & 63u)] = t;
    }
}

// gate and up of one column tile and GeGLU, as gateup_geglu_kernel: waves [0, W) gate, [W, 2W) up
template <int DTYPE>
__global__ void __launch_bounds__(64 * kWideWaves)
gateup_wide_kernel(const uint8_t* __restrict__ gate_tiles, const uint8_t* __restrict__ up_tiles, const float* __restrict__ xsums,
                   float* __restrict__ h, void* __restrict__ h_receipt, uint32_t F, const WideCfg c) {
    extern __shared__ __attribute__((aligned(256))) uint8_t lds[];
    __shared__ float vals[kWideRows * 64];
    float* red = reinterpret_cast<float*>(lds);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const bool is_up = wave >= c.W;
    const uint32_t slice = is_up ? wave - c.W : wave, b0 = min(slice * c.bps, c.nblk), b1 = min(b0 + c.bps, c.nblk);
    float acc[wide_cols(DTYPE)][2];
    run_wide<DTYPE>(is_up ? up_tiles : gate_tiles, xsums, c.K, c.nblk, blockIdx.x, b0, b1, lds + wave * 2 * kSlotBytes, lane, acc);
    __syncthreads();
    put_sums(acc, red + wave * kWideRows * 64, lane);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < c.rows * 64; i += blockDim.x) {
        float g = red[i], u = red[c.W * kWideRows * 64 + i];
        for (uint32_t w = 1; w < c.W; ++w) { g += red[w * kWideRows * 64 + i]; u += red[(c.W + w) * kWideRows * 64 + i]; }
        const float v = geglu_value(g, u);
        h[size_t(i >> 6) * F + blockIdx.x * kTileCols + (i & 63u)] = v;
        vals[i] = v;
    }
    __syncthreads();
    for (uint32_t r = 0; r < c.rows; ++r) emit_receipt(vals + r * 64, blockIdx.x * kTileCols, kTileCols, r, c.rows, F, h_receipt);
}

__global__ void wide_reduce_kernel(const float* __restrict__ part, float* __restrict__ y, uint32_t planes, uint32_t count) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) y[i] = load_planes(part + i, planes, count);
}

// dynamic LDS of a launch of W waves
template <typename Kernel>
int raise_lds(Kernel* kernel) {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kWideLds) != hipSuccess;
}

int wide_split(uint32_t count, const int* dtypes, const uint32_t* N, uint32_t K, GemvSplit* split, int* mode) {
    uint32_t tiles = 0;
    *mode = dtypes[0];
    for (uint32_t i = 0; i < count; ++i) {
        const int d = dtypes[i];
        if (d < GUFFIN_Q8_0 || d > GUFFIN_Q6_K || K == 0 || N[i] == 0 || K % block_elems(d) != 0 || N[i] % kTileCols != 0
            || block_elems(d) != block_elems(dtypes[0]))
            return fail(GUFFIN_E_SHAPE, "gemv_wide: need K % block == 0, N % 64 == 0 and one block length");
        if (d != dtypes[0]) *mode = kWideMixed;
        tiles += N[i] / kTileCols;
    }
    *split = gemv_split(K / block_elems(dtypes[0]), tiles, kWideWaves, kWideWaves);
    return GUFFIN_OK;
}

}  // namespace

int gemv_wide_init() {
    return raise_lds(gemv_wide_kernel<GUFFIN_Q4_K>) | raise_lds(gemv_wide_kernel<GUFFIN_Q6_K>) | raise_lds(gemv_wide_kernel<GUFFIN_Q8_0>)
         | raise_lds(gemv_wide_kernel<kWideMixed>) | raise_lds(gateup_wide_kernel<GUFFIN_Q4_K>) | raise_lds(gateup_wide_kernel<GUFFIN_Q8_0>);
}

uint32_t gemv_wide_planes(uint32_t count, const int* dtypes, const uint32_t* N, uint32_t K) {
    GemvSplit sp {};
    int mode = 0;
    return wide_split(count, dtypes, N, K, &sp, &mode) ? 0u : sp.planes;
}

int gemv_wide(hipStream_t s, uint32_t count, const int* dtypes, const void* const* tiles, const uint32_t* N, float* const* partials,
              const float* xsums, float* y, uint32_t rows, uint32_t K) {
    if (count == 0 || count > 3 || rows == 0 || rows > kWideRows) return fail(GUFFIN_E_SHAPE, "gemv_wide: 1 to 3 matrices, 1 to 4 rows");
    GemvSplit sp {};
    int mode = 0;
    if (int rc = wide_split(count, dtypes, N, K, &sp, &mode)) return rc;
    WideMeta m {};
    uint32_t end = 0;
    for (uint32_t i = 0; i < 3; ++i) {
        const uint32_t k = i < count ? i : 0;
        if (i < count) end += N[i] / kTileCols;
        m.tiles[i] = static_cast<const uint8_t*>(tiles[k]); m.part[i] = partials[k]; m.N[i] = N[k];
        m.dtype[i] = static_cast<uint32_t>(dtypes[k]); m.tile_end[i] = end;
    }
    if (y && sp.planes == 1) m.part[0] = y;   // one plane is the result
    const WideCfg c {K, K / block_elems(dtypes[0]), sp.bps, sp.W, rows};
    const dim3 grid(end, sp.planes), block(64 * sp.W);
    const uint32_t lds = sp.W * 2 * kSlotBytes;
    if (mode == GUFFIN_Q4_K) launch(gemv_wide_kernel<GUFFIN_Q4_K>, grid, block, lds, s, xsums, m, c);
    else if (mode == GUFFIN_Q6_K) launch(gemv_wide_kernel<GUFFIN_Q6_K>, grid, block, lds, s, xsums, m, c);
    else if (mode == GUFFIN_Q8_0) launch(gemv_wide_kernel<GUFFIN_Q8_0>, grid, block, lds, s, xsums, m, c);
    else launch(gemv_wide_kernel<kWideMixed>, grid, block, lds, s, xsums, m, c);
    if (int rc = check_launch("gemv_wide")) return rc;
    if (!y || sp.planes == 1) return GUFFIN_OK;
    const uint32_t n = rows * N[0];
    launch(wide_reduce_kernel, dim3((n + 255) / 256), dim3(256), 0, s, partials[0], y, sp.planes, n);
    return check_launch("gemv_wide_reduce");
}

int gateup_wide(hipStream_t s, int dtype, const void* gate_tiles, const void* up_tiles, const float* xsums, float* h, float* h_sums,
                uint32_t rows, uint32_t K, uint32_t F) {
    if (dtype != GUFFIN_Q4_K && dtype != GUFFIN_Q8_0) return fail(GUFFIN_E_SHAPE, "gateup_wide: Q4_K or Q8_0 pairs only");
    if (rows == 0 || rows > kWideRows || K % block_elems(dtype) != 0 || F % kTileCols != 0) return fail(GUFFIN_E_SHAPE, "gateup_wide: bad shape");
    const uint32_t nblk = K / block_elems(dtype);
    GemvSplit sp = gemv_split(nblk, 2 * (F / kTileCols), kWideWaves / 2, kWideWaves);
    if (sp.planes > 1) {   // all k-slices of a tile in one workgroup
        sp.bps = (nblk + kWideWaves / 2 - 1) / (kWideWaves / 2);
        sp.W = (nblk + sp.bps - 1) / sp.bps;
    }
    const WideCfg c {K, nblk, sp.bps, sp.W, rows};
    const dim3 grid(F / kTileCols), block(2 * sp.W * 64);
    const uint32_t lds = 2 * sp.W * 2 * kSlotBytes;
    const uint8_t *g = static_cast<const uint8_t*>(gate_tiles), *u = static_cast<const uint8_t*>(up_tiles);
    if (dtype == GUFFIN_Q4_K) launch(gateup_wide_kernel<GUFFIN_Q4_K>, grid, block, lds, s, g, u, xsums, h, static_cast<void*>(h_sums), F, c);
    else launch(gateup_wide_kernel<GUFFIN_Q8_0>, grid, block, lds, s, g, u, xsums, h, static_cast<void*>(h_sums), F, c);
    return check_launch("gateup_wide");
}

}  // namespace guffin
