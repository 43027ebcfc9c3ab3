// The matrix-core operand of M activation rows ("image"), shared by everything that writes it (pack kernel, norms,
// GeGLU, attention) and by the prefill GEMM that reads it.
//
//   img  : half  [K/32][Mpad/16][hi, lo][64 lanes][8]   one 1 KB record per (32-group, 16 rows, half) in the order the
//                                        matrix instruction wants its A operand: lane (i, s) = i + 16 s holds k-slice s
//                                        (elements 8s..8s+7) of row i, inside it the halves at {0,2,1,3,4,6,5,7}
//   mult : float [K/span][Mpad]          2^E of (row, span); |x| 2^-E < 2^15 and hi + lo = x 2^-E to 22 bits, for what lies
//                                        below 2^-18 of the span's largest to 2^-40 of that
//   sums : half  [K/256][Mpad/16][32 lanes][8]   (K % 256 == 0) the 8 group sums of a 256-element block times 2^-(E+5), lane
//                                        i the hi and lane 16 + i the lo half of row i, group t at {0,2,1,3,4,6,5,7}[t]
//
// span is 256 when K is a multiple of 256 (a K-quant block), else 32.  Mpad is M rounded up to 16; the padding rows
// are not written: a row of A reaches only its own row of the product, which is not stored.
#pragma once
#include "common.hpp"

namespace guffin {

// a workgroup of the GEMM reads whole chunks of up to four row tiles: past the last tile it reads on into what follows
// (three records of a group, 2 KB of sums, 256 bytes of multipliers), which has to be there
constexpr size_t kImageSlack = 8192;

struct ImageLayout { size_t mult_off, sums_off, bytes; uint32_t mpad, span; };

__host__ __device__ inline ImageLayout image_layout(uint32_t M, uint32_t K) {
    ImageLayout L {};
    L.mpad = (M + 15) & ~15u;
    L.span = K % 256 == 0 ? 256 : 32;
    L.mult_off = size_t(K / 32) * L.mpad * 128;
    L.sums_off = (L.mult_off + size_t(K / L.span) * L.mpad * 4 + 255) & ~size_t{255};
    const size_t blocks = L.span == 256 ? K / 256 : 0;
    L.bytes = L.sums_off + blocks * L.mpad * 32 + kImageSlack;
    return L;
}

// biased exponent of a span's largest, clamped so that both scale factors are normal floats; the span's multiplier
__device__ __forceinline__ uint32_t image_exponent(float largest) {
    const uint32_t eb = __float_as_uint(largest) >> 23;
    return eb < 15u ? 15u : eb > 244u ? 244u : eb;
}
__device__ __forceinline__ float image_multiplier(float largest) { return __uint_as_float((image_exponent(largest) - 14u) << 23); }

// the order of a lane's eight halves in a record, and of a block's eight group sums
constexpr int kImageOrder[8] = {0, 2, 1, 3, 4, 6, 5, 7};

// a lane's eight elements as halves, hi + lo = x inv
__device__ __forceinline__ void image_halves(const float (&v)[8], float inv, uint4& hi, uint4& lo) {
    uint32_t h4[4], l4[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        uint32_t hw = 0, lw = 0;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const float xv = v[kImageOrder[2 * p + q]] * inv;
            const _Float16 h = static_cast<_Float16>(xv);
            const _Float16 l = static_cast<_Float16>(xv - static_cast<float>(h));
            hw |= uint32_t(__builtin_bit_cast(uint16_t, h)) << (16 * q);
            lw |= uint32_t(__builtin_bit_cast(uint16_t, l)) << (16 * q);
        }
        h4[p] = hw; l4[p] = lw;
    }
    hi = make_uint4(h4[0], h4[1], h4[2], h4[3]);
    lo = make_uint4(l4[0], l4[1], l4[2], l4[3]);
}
// what a span's elements are multiplied with: 1 / its multiplier
__device__ __forceinline__ float image_scale(float largest) { return __uint_as_float((268u - image_exponent(largest)) << 23); }
// the sum of a row's 32-group g (K % 256 == 0)
__device__ __forceinline__ void emit_group_sum(float sum, float inv, uint32_t g, uint32_t row, const ImageLayout& L, uint8_t* blob) {
    const float sv = sum * (inv * 0.03125f);   // |sum| <= 32 times the span's largest
    const _Float16 h = static_cast<_Float16>(sv), l = static_cast<_Float16>(sv - static_cast<float>(h));
    uint8_t* rec = blob + L.sums_off + (size_t(g >> 3) * (L.mpad / 16) + (row >> 4)) * 512 + (row & 15u) * 16 + kImageOrder[g & 7u] * 2;
    *reinterpret_cast<uint16_t*>(rec) = __builtin_bit_cast(uint16_t, h);
    *reinterpret_cast<uint16_t*>(rec + 256) = __builtin_bit_cast(uint16_t, l);
}

// A record's share of a lane: elements 8s .. 8s+7 of 32-group g of a row whose span of 256 holds `largest`.  The lanes (row, 0 .. 3) of
// a row, 16 apart, run it together.
__device__ __forceinline__ void emit_image_record(const float (&v)[8], float largest, uint32_t g, uint32_t s, uint32_t row, const ImageLayout& L, uint8_t* blob) {
    const float inv = image_scale(largest);
    float sum = v[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) sum += v[i];
    sum += __shfl_xor(sum, 16, kWave);
    sum += __shfl_xor(sum, 32, kWave);
    if (s == 0) emit_group_sum(sum, inv, g, row, L, blob);
    uint4 hi, lo;
    image_halves(v, inv, hi, lo);
    uint8_t* base = blob + (size_t(g) * (L.mpad / 16) + (row >> 4)) * 2048 + ((row & 15u) + 16 * s) * 16;
    *reinterpret_cast<uint4*>(base) = hi;
    *reinterpret_cast<uint4*>(base + 1024) = lo;
}

// Elements 8t .. 8t+7 of row `row` (t counts along K).  The lanes of a span (32 or 4 consecutive t in consecutive,
// aligned lanes) must run it together.  records: where a workgroup that holds 8 rows of eight groups collects their pieces of the
// records (16 KB of LDS) instead of writing 16 bytes at a time to lines that it shares with other rows.
__device__ __forceinline__ void emit_image_values(const float (&v)[8], uint32_t t, uint32_t row, const ImageLayout& L, uint8_t* blob,
                                                  uint8_t* records = nullptr) {
    const uint32_t g = t >> 2, s = t & 3u;
    float sum = v[0], m = fabsf(v[0]);
#pragma unroll
    for (int i = 1; i < 8; ++i) { sum += v[i]; m = fmaxf(m, fabsf(v[i])); }
    m = fmaxf(m, lane_cross<0xB1>(m));
    m = fmaxf(m, lane_cross<0x4E>(m));
    if (L.span == 256) {
        m = fmaxf(m, lane_cross<0x141>(m));
        m = fmaxf(m, lane_cross<0x140>(m));
        m = both_max(rows_beside(__float_as_uint(m)));
    }
    const float inv = image_scale(m);
    const uint32_t tile = row >> 4, i16 = row & 15u;
    if (L.span == 256 ? (t & 31u) == 0 : s == 0)
        reinterpret_cast<float*>(blob + L.mult_off)[size_t(L.span == 256 ? t >> 5 : g) * L.mpad + row] = image_multiplier(m);
    if (L.span == 256) {
        const float sum16 = sum + lane_cross<0xB1>(sum);
        const float sum32 = sum16 + lane_cross<0x4E>(sum16);
        if (s == 0) emit_group_sum(sum32, inv, g, row, L, blob);
    }
    uint4 hi, lo;
    image_halves(v, inv, hi, lo);
    uint8_t* base = records ? records + (g & 7u) * 2048 : blob + (size_t(g) * (L.mpad / 16) + tile) * 2048;
    base += (i16 + 16 * s) * 16;
    *reinterpret_cast<uint4*>(base) = hi;
    *reinterpret_cast<uint4*>(base + 1024) = lo;
}

}  // namespace guffin
