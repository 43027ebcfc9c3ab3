// One element of an embedding row, as the model file holds it (canonical block stream, a row = width / elements blocks).
#pragma once
#include "common.hpp"

namespace guffin {

template <int DTYPE> constexpr uint32_t kEmbedElems = DTYPE == GUFFIN_Q8_0 ? 32 : 256;
template <int DTYPE> constexpr uint32_t kEmbedBytes = DTYPE == GUFFIN_Q8_0 ? 34 : DTYPE == GUFFIN_Q4_K ? 144 : 210;

template <int DTYPE>
__device__ __forceinline__ const uint8_t* embed_row(const uint8_t* w, uint32_t token, uint32_t width) {
    return w + size_t(token) * (width / kEmbedElems<DTYPE>) * kEmbedBytes<DTYPE>;
}

template <int DTYPE>
__device__ __forceinline__ float embed_element(const uint8_t* row, uint32_t c) {
    constexpr uint32_t be = kEmbedElems<DTYPE>, bb = kEmbedBytes<DTYPE>;
    const uint8_t* b = row + size_t(c / be) * bb;
    const uint32_t i = c % be;
    float v;
    if constexpr (DTYPE == GUFFIN_Q8_0) {
        v = __fmul_rn(h2f(ld_u16(b)), static_cast<float>(static_cast<int8_t>(b[2 + i])));
    } else if constexpr (DTYPE == GUFFIN_Q6_K) {
        const uint32_t half = i >> 7, rr = i & 127, l = rr & 31;
        const uint32_t lo_byte = b[half * 64 + ((rr >> 5) & 1) * 32 + l];
        const uint32_t lo = rr < 64 ? (lo_byte & 0x0Fu) : (lo_byte >> 4);
        const uint32_t hi = (b[128 + half * 32 + l] >> ((rr >> 5) * 2)) & 3u;
        const int q = static_cast<int>(lo | (hi << 4)) - 32;
        const float sc = static_cast<float>(static_cast<int8_t>(b[192 + (i >> 4)]));
        v = __fmul_rn(__fmul_rn(h2f(ld_u16(b + 208)), sc), static_cast<float>(q));
    } else {
        const float d = h2f(ld_u16(b)), dmin = h2f(ld_u16(b + 2));
        const uint8_t* s = b + 4;
        const uint32_t g = i >> 5;
        uint32_t sc, mn;
        if (g < 4) { sc = s[g] & 63u; mn = s[g + 4] & 63u; }
        else { sc = (s[g + 4] & 0x0Fu) | ((s[g - 4] >> 6) << 4); mn = (s[g + 4] >> 4) | ((s[g] >> 6) << 4); }
        const uint32_t byte = b[16 + (i >> 6) * 32 + (i & 31)];
        const uint32_t q = (i & 63) < 32 ? (byte & 0x0Fu) : (byte >> 4);
        v = __fsub_rn(__fmul_rn(__fmul_rn(d, static_cast<float>(sc)), static_cast<float>(q)),
                      __fmul_rn(dmin, static_cast<float>(mn)));
    }
    return v;
}

}  // namespace guffin
