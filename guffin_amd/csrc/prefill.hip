// Causal GQA attention of a run of rows over the fp16 KV rings (gfx950), and the moves of K/V rows around it.
//
// Replaces the reference's encode_f16_prefill_attention (src/tensor/backends/metal/metal_command_context.hpp:185, kernels
// metal_kernels.mm:2593-2800).
//
// prefill_attention_mfma_kernel runs on the matrix core for one, two or four query heads per KV head; prefill_attention_kernel
// on the vector unit takes rows it cannot (other alignments, no workspace).  Positions before the run come from the ring,
// the run's own from its private rows, which are published to the ring afterwards.  Both walk the visible key range in tiles
// of 32 tokens with an online softmax, fp32 math on fp16 keys and values.
#include "common.hpp"
#include "prefill_image.hpp"
#include "prefill_run.hpp"

#include <algorithm>

namespace guffin {
namespace {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

// ---- causal attention for a run of rows ------------------------------------------------
// grid (ceil(rows / 16), kv_heads), 256 threads: thread = (query slot of 16 rows x GROUP heads, one of
// 256/(16*GROUP) interleaved dim slices).  Keys/values of positions below `position` come from the
// ring, those of the run itself from its private fp16 rows [rows][kv_heads*256].
template <int GROUP>
__global__ void __launch_bounds__(256)
prefill_attention_kernel(const float* __restrict__ q, const uint16_t* __restrict__ ring_k,
                         const uint16_t* __restrict__ ring_v, const uint16_t* __restrict__ run_k,
                         const uint16_t* __restrict__ run_v, float* __restrict__ out, uint32_t rows,
                         uint32_t position, uint32_t window, uint32_t ring_mask, uint32_t q_heads,
                         uint32_t kv_heads, float scale) {
    constexpr int HD = 256, QT = 16, NQ = QT * GROUP, KT = 32;
    constexpr int TPQ = 256 / NQ;        // threads per query: 16, 8 or 4
    constexpr int DPT = HD / TPQ;        // dims per thread, interleaved: dim = part + TPQ * i
    __shared__ _Float16 ks[KT][HD + 2];
    __shared__ _Float16 vs[KT][HD + 2];
    __shared__ float sc[NQ][KT];
    const uint32_t kvh = blockIdx.y, r0 = blockIdx.x * QT;
    const uint32_t qi = threadIdx.x / TPQ, part = threadIdx.x % TPQ;
    const uint32_t row = r0 + qi / GROUP, head = kvh * GROUP + qi % GROUP;
    const bool live = row < rows;
    const uint32_t pos = position + row;
    float qv[DPT], acc[DPT];
#pragma unroll
    for (int i = 0; i < DPT; ++i) {
        qv[i] = live ? q[(size_t(row) * q_heads + head) * HD + part + TPQ * i] * scale : 0.f;
        acc[i] = 0.f;
    }
    float mx = -INFINITY, den = 0.f;
    const uint32_t last_row = min(r0 + QT, rows) - 1;
    const uint32_t hi_pos = position + last_row;
    const uint32_t lo_first = (window && position + r0 + 1 > window) ? position + r0 + 1 - window : 0;
    const uint32_t my_first = (window && pos + 1 > window) ? pos + 1 - window : 0;
    const size_t row_stride = size_t(kv_heads) * HD;
    for (uint32_t t0 = lo_first; t0 <= hi_pos; t0 += KT) {
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < KT * HD / 2; i += 256) {
            const uint32_t t = i / (HD / 2), d2 = i % (HD / 2);
            uint32_t kk = 0, vv = 0;
            const uint32_t kp = t0 + t;
            if (kp <= hi_pos) {
                const bool own = kp >= position;
                const size_t off = (own ? size_t(kp - position) : size_t(kp & ring_mask)) * row_stride + kvh * HD + 2 * d2;
                kk = *reinterpret_cast<const uint32_t*>((own ? run_k : ring_k) + off);
                vv = *reinterpret_cast<const uint32_t*>((own ? run_v : ring_v) + off);
            }
            *reinterpret_cast<uint32_t*>(&ks[t][2 * d2]) = kk;
            *reinterpret_cast<uint32_t*>(&vs[t][2 * d2]) = vv;
        }
        __syncthreads();
        float tile_max = -INFINITY;
        float s_loc[KT / TPQ];
        for (int t = 0; t < KT; ++t) {
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < DPT; ++i) s = fmaf(qv[i], static_cast<float>(ks[t][part + TPQ * i]), s);
#pragma unroll
            for (int o = TPQ / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, kWave);
            const uint32_t kp = t0 + t;
            const bool visible = live && kp <= pos && kp >= my_first;
            s = visible ? s : -INFINITY;
            if (uint32_t(t) % TPQ == part) s_loc[t / TPQ] = s;
            tile_max = fmaxf(tile_max, s);
        }
        const float new_max = fmaxf(mx, tile_max);
        const float rescale = new_max == -INFINITY ? 1.f : expf(mx - new_max);
        den *= rescale;
#pragma unroll
        for (int i = 0; i < DPT; ++i) acc[i] *= rescale;
        float add = 0.f;
#pragma unroll
        for (int u = 0; u < KT / TPQ; ++u) {
            const float p = s_loc[u] == -INFINITY ? 0.f : expf(s_loc[u] - new_max);
            sc[qi][u * TPQ + part] = p;
            add += p;
        }
#pragma unroll
        for (int o = TPQ / 2; o > 0; o >>= 1) add += __shfl_xor(add, o, kWave);
        den += add;
        mx = new_max;
        // the TPQ lanes of a query sit in one wave: their sc[] entries are visible after a wave barrier
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (int t = 0; t < KT; ++t) {
            const float p = sc[qi][t];
#pragma unroll
            for (int i = 0; i < DPT; ++i) acc[i] = fmaf(p, static_cast<float>(vs[t][part + TPQ * i]), acc[i]);
        }
    }
    if (live) {
#pragma unroll
        for (int i = 0; i < DPT; ++i) out[(size_t(row) * q_heads + head) * HD + part + TPQ * i] = acc[i] / den;
    }
}

// ---- the same attention on the matrix core ------------------------------------------------
// Values are contracted over tokens, so a lane's operand is eight tokens of one output dimension, those whose probabilities the lane has:
// a small pass first writes V^T, [kv_heads][T / 32][256][32] fp16 (a tile in one piece: with rows of T tokens an operand
// took half of each of sixteen lines), a dimension's 32 tokens in the order of value_token, for the virtual tokens
// base32 .. base32 + T (T a multiple of 32; tokens outside [first_visible, end) are zero).
__global__ void __launch_bounds__(256)
transpose_values_kernel(const uint16_t* __restrict__ ring_v, const uint16_t* __restrict__ run_v,
                        uint16_t* __restrict__ vt, uint32_t base32, uint32_t T, uint32_t first_visible,
                        uint32_t position, uint32_t end_pos, uint32_t ring_mask, uint32_t kv_heads) {
    constexpr int HD = 256, PITCH = HD + 8;
    __shared__ __attribute__((aligned(16))) uint16_t tile[32][PITCH];
    const uint32_t kvh = blockIdx.y, v0 = blockIdx.x * 32;
    const size_t row_stride = size_t(kv_heads) * HD;
    for (uint32_t c = threadIdx.x; c < 32 * (HD / 8); c += 256) {
        const uint32_t token = c / (HD / 8), d8 = c % (HD / 8);
        const uint32_t kp = base32 + v0 + token;
        uint4 val = make_uint4(0, 0, 0, 0);
        if (kp >= first_visible && kp < end_pos) {
            const uint16_t* src = kp >= position ? run_v + size_t(kp - position) * row_stride
                                                 : ring_v + size_t(kp & ring_mask) * row_stride;
            val = *reinterpret_cast<const uint4*>(src + kvh * HD + 8 * d8);
        }
        *reinterpret_cast<uint4*>(&tile[token][8 * d8]) = val;
    }
    __syncthreads();
    const uint32_t dim = threadIdx.x;
    uint32_t w[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) w[t] = uint32_t(tile[2 * t][dim]) | (uint32_t(tile[2 * t + 1][dim]) << 16);
    uint4* dst = reinterpret_cast<uint4*>(vt + size_t(kvh) * HD * T + (size_t(v0) * HD + dim * 32));
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[i] = make_uint4(w[2 * i], w[2 * i + 1], w[8 + 2 * i], w[8 + 2 * i + 1]);   // value_token's order
}

__device__ __forceinline__ void split_half8(const float (&x)[8], uint4& hi, uint4& lo) {
    uint32_t h[4], l[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        uint32_t hw = 0, lw = 0;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const _Float16 a = static_cast<_Float16>(x[2 * p + q]);
            const _Float16 b = static_cast<_Float16>(x[2 * p + q] - static_cast<float>(a));
            hw |= uint32_t(__builtin_bit_cast(uint16_t, a)) << (16 * q);
            lw |= uint32_t(__builtin_bit_cast(uint16_t, b)) << (16 * q);
        }
        h[p] = hw; l[p] = lw;
    }
    hi = make_uint4(h[0], h[1], h[2], h[3]);
    lo = make_uint4(l[0], l[1], l[2], l[3]);
}

// where the attention of a run leaves its rows: fp32 rows, or the o projection's operand (prefill_image.hpp), or, when the
// key range is cut into parts, the parts' states
struct AttentionOut { float* rows; uint8_t* image; float* part_o; float* part_ml; };
constexpr float kProbScale = 1024.0f;   // probabilities enter the matrix instruction times 2^10
constexpr float kLog2e = 1.44269504088896340736f;
// e^x of a difference of scores: v_exp_f32 (an ulp; it flushes what is below 2^-126) behind a multiplication by log2(e).  That
// stands here, where it costs the difference one rounding, and not at the queries, where every operand would be rounded once
// more ahead of the product and lose half a bit of its range, nor at the maxima, whose rounding is not small beside large scores.
__device__ __forceinline__ float exp_of(float x) { return __builtin_amdgcn_exp2f(x * kLog2e); }

// one (row, head): 8 consecutive output dimensions in 32 consecutive lanes
__device__ __forceinline__ void emit_attention(const AttentionOut& to, const float (&v)[8], uint32_t row, uint32_t rows, uint32_t head,
                                               uint32_t q_heads, uint32_t c8) {
    constexpr uint32_t HD = 256;
    if (to.image) {
        emit_image_values(v, head * (HD / 8) + c8, row, image_layout(rows, q_heads * HD), to.image);
    } else {
        float* dst = to.rows + (size_t(row) * q_heads + head) * HD + 8 * c8;
#pragma unroll
        for (int i = 0; i < 8; ++i) dst[i] = v[i];
    }
}

// a workgroup's LDS: its waves' outputs of an A tile, their states and the merged ones (queries and probabilities take less)
constexpr uint32_t kOutPitch = 256 + 4;   // floats between two pairs' outputs there: 16 lanes that store four dimensions each touch every bank once
constexpr uint32_t attention_lds(uint32_t nt, uint32_t waves) { return waves * 16 * kOutPitch * 4 + (waves + 1) * nt * 16 * 2 * 4; }
static_assert(attention_lds(2, 4) >= 2 * 16384);

// grid (kv_heads * ceil(rows * group / (16 NT)), 1, parts), W waves.  Heads run fastest and the last rows come first: consecutive
// workgroups go to different XCDs, so with eight KV heads an L2 holds one head's keys and values, and the longest lists of a causal
// block start first.  (Tiles fastest, first rows first: 2048 rows 162 us instead of 142, 333 rows 22.6 instead of 17.6.)  A workgroup serves 16 NT (row, head) pairs of one KV head
// -- the group's heads of 16 NT / group consecutive rows, as NT A tiles of 16 pairs -- and one part of the key range.  Each
// wave walks its own 32-token tiles (tile index = wave mod W) with its own online softmax state and its own output
// accumulators; the states are merged at the end.  A run of few rows is cut into parts so that the chip is full; their
// states are merged by prefill_attention_merge_kernel.
//   scores   S^T = K Q^T: keys straight from their fp16 rows as A (a lane reads 8 dims of one key per MFMA), queries (scaled, fp16
//            hi + lo, staged once in LDS in operand order) as B.  So a lane has eight scores of one pair, tokens 4 lg .. 4 lg + 3 of
//            either half of the tile, and four lanes all of that pair's
//   softmax  over those eight and two swaps of lanes; the denominator stays the lane's own until the end.  A tile that every row
//            sees whole needs no masks, and the accumulators are rescaled only where a maximum moved
//   values   O^T += V^T P^T: the lane's own probabilities times 2^10 as fp16 hi + lo as B, V^T rows as A, whose tokens lie in that
//            order; so a lane has four dimensions of its pair an instruction
// (S = Q K^T, four pairs a lane: a maximum and a sum over 16 lanes for each, the probabilities through LDS to become an operand and
// the outputs through LDS word by word: 37 rows at 1500 12.1 us, 333 rows 16.8, 2048 rows 108, the drafter's 1000 21.4; so 10.2, 15.1,
// 99 and 19.7.  Of the 37 rows' 7.6 behind the launch 2.7 are until the queries are staged, 2.0 until the scores, 0.4 the softmax, 0.9
// the values, 1.5 the merge.)
template <int NT, int W>
__global__ void __launch_bounds__(64 * W, W == 4 ? 2 : 1)
prefill_attention_mfma_kernel(const float* __restrict__ q, const uint16_t* __restrict__ ring_k,
                              const uint16_t* __restrict__ run_k, const uint16_t* __restrict__ vt,
                              uint32_t rows, uint32_t position, uint32_t window, uint32_t ring_mask, uint32_t base32, uint32_t form,
                              float scale, uint32_t T, AttentionOut to) {
    // (the arguments' order: what the first requests need goes first, see the kernels of gemv_packed.hip)
    const uint32_t kv_heads = form & 0xFFFFu, group_shift = (form >> 16) & 3u, q_heads = kv_heads << group_shift, parts = form >> 18;
    constexpr int HD = 256;
    constexpr uint32_t kPairs = 16 * NT;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    // [NT][8 k-steps][hi, lo][64 lanes] 16-byte query operands
    uint8_t* qa = lds;
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t j = lane & 15, lg = lane >> 4;
    const uint32_t kvh = blockIdx.x % kv_heads, group = 1u << group_shift;
    const uint32_t r0 = ((((rows << group_shift) + kPairs - 1) / kPairs) - 1 - blockIdx.x / kv_heads) * (kPairs >> group_shift);
    const size_t row_stride = size_t(kv_heads) * HD;
    const uint32_t last_row = min(r0 + (kPairs >> group_shift), rows) - 1;
    const uint32_t hi_pos = position + last_row;
    const uint32_t lo_first = (window && position + r0 + 1 > window) ? position + r0 + 1 - window : 0;
    const uint32_t last_first = (window && hi_pos + 1 > window) ? hi_pos + 1 - window : 0;   // of the last row
    const uint32_t tile_lo = (lo_first - base32) / 32, tiles = (hi_pos - base32) / 32 + 1 - tile_lo;
    const uint32_t begin = tile_lo + blockIdx.z * tiles / parts, end = tile_lo + (blockIdx.z + 1) * tiles / parts;

    auto ask_keys = [&](uint32_t ti, uint4 (&kb)[2][8]) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const uint32_t kp = min(base32 + 32 * ti + 16 * c + j, hi_pos);
            const uint16_t* krow = (kp >= position ? run_k + size_t(kp - position) * row_stride
                                                   : ring_k + size_t(kp & ring_mask) * row_stride) + kvh * HD + 8 * lg;
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) kb[c][ks] = *reinterpret_cast<const uint4*>(krow + 32 * ks);
        }
    };
    uint4 kb[2][8];
    constexpr uint32_t kStep = 2 * W;   // pairs staged (or stored) at a time
    float4 qv[kPairs / kStep][2];
#pragma unroll
    for (uint32_t i = 0; i < kPairs / kStep; ++i) {
        const uint32_t m = kStep * i + threadIdx.x / 32, c8 = threadIdx.x % 32;
        const uint32_t row = min(r0 + (m >> group_shift), rows - 1), head = kvh * group + (m & (group - 1));
        const float* src = q + (size_t(row) * q_heads + head) * HD + 8 * c8;
        qv[i][0] = *reinterpret_cast<const float4*>(src); qv[i][1] = *reinterpret_cast<const float4*>(src + 4);
    }
    asm volatile("" ::: "memory");   // the queries are asked for first: what is asked for before them arrives before them
    // one A tile leaves registers for the next keys beside the values: the first ones travel while the queries are staged
    if constexpr (NT == 1) ask_keys(min(begin + wave, tile_lo + tiles - 1), kb);
#pragma unroll
    for (uint32_t i = 0; i < kPairs / kStep; ++i) {
        const uint32_t m = kStep * i + threadIdx.x / 32, c8 = threadIdx.x % 32;
        const float4 a = qv[i][0], b = qv[i][1];
        const float x[8] = {a.x * scale, a.y * scale, a.z * scale, a.w * scale, b.x * scale, b.y * scale, b.z * scale, b.w * scale};
        uint4 hi, lo;
        split_half8(x, hi, lo);
        uint8_t* dst = qa + (((m >> 4) * 8 + c8 / 4) * 2) * 1024 + ((m & 15) + 16 * (c8 % 4)) * 16;
        *reinterpret_cast<uint4*>(dst) = hi;
        *reinterpret_cast<uint4*>(dst + 1024) = lo;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // the keys stay on their way

    float m[NT], l[NT];   // of pair 16 g + j: its maximum; the sum over this lane's tokens
    float4_t O[NT][16];   // [dt]: dimensions 16 dt + 4 lg .. + 3
#pragma unroll
    for (int g = 0; g < NT; ++g) {
        m[g] = -INFINITY; l[g] = 0.f;
#pragma unroll
        for (int dt = 0; dt < 16; ++dt) O[g][dt] = float4_t{0.f, 0.f, 0.f, 0.f};
    }
    constexpr int VB = NT > 1 ? 8 : 16;   // one A tile: all values of a tile in registers, asked for ahead of the scores
    for (uint32_t ti = begin + wave; ti < end; ti += W) {
        const uint32_t t0 = base32 + 32 * ti;
        if constexpr (NT > 1) ask_keys(ti, kb);
        const uint16_t* vcol = vt + size_t(kvh) * HD * T + size_t(ti) * (32 * HD) + 32 * j + 8 * lg;
        uint4 vb[VB];
        auto ask_values = [&](int first) {
#pragma unroll
            for (int i = 0; i < VB; ++i) vb[i] = *reinterpret_cast<const uint4*>(vcol + 512 * (first + i));
        };
        if constexpr (NT == 1) ask_values(0);
        // A sum rounds at the size it has grown to: the hi halves of the first four steps are one chain; the other takes the lo
        // halves, whose sums are small, and from the fifth step on both.
        float4_t S[NT][2], rest[NT][2];
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
#pragma unroll
            for (int half = 1; half >= 0; --half)
#pragma unroll
                for (int g = 0; g < NT; ++g) {
                    const half8_t q8 = __builtin_bit_cast(half8_t, *reinterpret_cast<const uint4*>(qa + ((g * 8 + ks) * 2 + half) * 1024 + lane * 16));
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        float4_t& sum = half == 0 && ks < 4 ? S[g][c] : rest[g][c];
                        sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, kb[c][ks]), q8,
                                                                     ks == 0 ? float4_t{0.f, 0.f, 0.f, 0.f} : sum, 0, 0, 0);
                    }
                }
#pragma unroll
        for (int g = 0; g < NT; ++g)
#pragma unroll
            for (int c = 0; c < 2; ++c) S[g][c] += rest[g][c];
        if constexpr (NT > 1) __builtin_amdgcn_sched_barrier(0);   // the keys' registers become the values'
        if constexpr (NT > 1) ask_values(0);
        // online softmax of a pair's 32 scores, eight in each of four lanes
        if (!(t0 >= last_first && t0 + 31 <= position + r0)) {
#pragma unroll
            for (int g = 0; g < NT; ++g) {
                const uint32_t row = r0 + ((16 * g + j) >> group_shift), pos = position + row;
                const uint32_t first = (window && pos + 1 > window) ? pos + 1 - window : 0u;
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const uint32_t kp = t0 + 16 * c + 4 * lg + r;
                        if (!(row < rows && kp <= pos && kp >= first)) S[g][c][r] = -INFINITY;
                    }
            }
        }
        float top[NT];
        bool moved = false;
#pragma unroll
        for (int g = 0; g < NT; ++g) {
            float t = fmaxf(fmaxf(fmaxf(S[g][0][0], S[g][0][1]), fmaxf(S[g][0][2], S[g][0][3])),
                            fmaxf(fmaxf(S[g][1][0], S[g][1][1]), fmaxf(S[g][1][2], S[g][1][3])));
            t = both_max(rows_beside(__float_as_uint(t)));
            top[g] = fmaxf(m[g], both_max(halves_beside(__float_as_uint(t))));
            moved |= top[g] > m[g];
        }
        if (__ballot(moved)) {
#pragma unroll
            for (int g = 0; g < NT; ++g) {
                const float resc = top[g] == -INFINITY ? 1.f : exp_of(m[g] - top[g]);
                l[g] *= resc;
                m[g] = top[g];
#pragma unroll
                for (int dt = 0; dt < 16; ++dt) O[g][dt] *= resc;
            }
        }
        half8_t pa[NT][2];
#pragma unroll
        for (int g = 0; g < NT; ++g) {
            const float from = m[g] == -INFINITY ? 0.f : m[g];   // nothing seen yet: every score is -inf
            float x[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) x[k] = exp_of(S[g][k >> 2][k & 3] - from);
            l[g] += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
#pragma unroll
            for (int k = 0; k < 8; ++k) x[k] *= kProbScale;
            uint4 hi, lo;
            split_half8(x, hi, lo);
            pa[g][0] = __builtin_bit_cast(half8_t, hi);
            pa[g][1] = __builtin_bit_cast(half8_t, lo);
        }
        __builtin_amdgcn_sched_barrier(0);   // the next keys are asked for here and not ahead of the softmax: there are no registers for that
        auto values = [&](int first) {
#pragma unroll
            for (int half = 0; half < 2; ++half)
#pragma unroll
                for (int i = 0; i < VB; ++i)
#pragma unroll
                    for (int g = 0; g < NT; ++g)
                        O[g][first + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, vb[i]), pa[g][half], O[g][first + i], 0, 0, 0);
        };
        if constexpr (NT == 1) {
            if (ti + W < end) ask_keys(ti + W, kb);
            values(0);
        } else {
            values(0);
            __builtin_amdgcn_sched_barrier(0);
            ask_values(8);
            values(8);
        }
    }
    // Merge the waves' states through LDS, an A tile at a time: every wave's outputs, scaled to the common maximum by their own
    // wave, have room together and are summed in wave order by whoever stores them.  (One wave behind the other over the same slots:
    // three more passes over them,
    // 14 us of a workgroup's 65 at 2048 rows instead of 9.)
    float* ob = reinterpret_cast<float*>(lds);  // [wave][16 pairs][kOutPitch]; the query operands are dead now
    constexpr uint32_t kWaveSlots = 16 * kOutPitch;   // of one wave's outputs
    float* states = reinterpret_cast<float*>(lds + W * kWaveSlots * 4);   // [wave][pair][2]
    float* ml = states + W * kPairs * 2;        // [pair][2], merged
#pragma unroll
    for (int g = 0; g < NT; ++g) {
        l[g] = both_sum(rows_beside(__float_as_uint(l[g])));
        l[g] = both_sum(halves_beside(__float_as_uint(l[g])));
    }
    if (lg == 0)   // (behind the queries' operands, which others may still read)
#pragma unroll
        for (int g = 0; g < NT; ++g) *reinterpret_cast<float2*>(states + (wave * kPairs + 16 * g + j) * 2) = make_float2(m[g], l[g]);
    __syncthreads();
#pragma unroll
    for (int g = 0; g < NT; ++g) {
        if (g > 0) __syncthreads();   // the tile before has been read
        const uint32_t pair = 16 * g + j;
        float2 st[W];
#pragma unroll
        for (int w = 0; w < W; ++w) st[w] = *reinterpret_cast<const float2*>(states + (w * kPairs + pair) * 2);
        float M = st[0].x;
#pragma unroll
        for (int w = 1; w < W; ++w) M = fmaxf(M, st[w].x);
        const float mine = m[g] == -INFINITY ? 0.f : exp_of(m[g] - M);
        float* slots = ob + wave * kWaveSlots + j * kOutPitch + 4 * lg;
#pragma unroll
        for (int dt = 0; dt < 16; ++dt) *reinterpret_cast<float4_t*>(slots + 16 * dt) = O[g][dt] * mine;
        if (wave == 0 && lg == 0) {
            float den = 0.f;
#pragma unroll
            for (int w = 0; w < W; ++w) den += st[w].x == -INFINITY ? 0.f : st[w].y * exp_of(st[w].x - M);
            *reinterpret_cast<float2*>(ml + pair * 2) = make_float2(M, den);
        }
        __syncthreads();
#pragma unroll 1
        for (uint32_t n = 0; n < 16 / kStep; ++n) {   // 32 consecutive lanes: one (row, head)
            const uint32_t i = kStep * n + threadIdx.x / 32, c8 = threadIdx.x % 32, p = 16 * g + i;
            const uint32_t row = r0 + (p >> group_shift), head = kvh * group + (p & (group - 1));
            if (row >= rows) continue;
            const float* src = ob + i * kOutPitch + 8 * c8;
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                float more = src[kWaveSlots + k];
#pragma unroll
                for (uint32_t w = 2; w < W; ++w) more += src[w * kWaveSlots + k];
                v[k] = src[k] + more;
            }
            if (parts == 1) {
                const float den = ml[p * 2 + 1] * kProbScale;
#pragma unroll
                for (int k = 0; k < 8; ++k) v[k] /= den;
                emit_attention(to, v, row, rows, head, q_heads, c8);
            } else {
                const size_t at = (size_t(blockIdx.z) * rows + row) * q_heads + head;
                float* dst = to.part_o + at * HD + 8 * c8;
#pragma unroll
                for (int k = 0; k < 8; ++k) dst[k] = v[k];
                if (c8 == 0) { to.part_ml[2 * at] = ml[p * 2]; to.part_ml[2 * at + 1] = ml[p * 2 + 1]; }
            }
        }
    }
}

// the parts' states of every (row, head), merged in part order; 32 lanes per pair
__global__ void __launch_bounds__(256)
prefill_attention_merge_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml, uint32_t rows, uint32_t q_heads, uint32_t parts,
                               AttentionOut to) {
    constexpr uint32_t HD = 256, kAhead = 12;   // parts asked for at once
    const uint32_t pair = blockIdx.x * 8 + threadIdx.x / 32, c8 = threadIdx.x % 32;
    if (pair >= rows * q_heads) return;
    const size_t stride = size_t(rows) * q_heads;
    // a lane a part's state, 32 at a time: their maximum and weights are two reductions instead of a walk of one trip a part
    const float2* states = reinterpret_cast<const float2*>(part_ml);
    auto top_of = [](float x) { return both_max(rows_beside(__float_as_uint(row16_max(x)))); };
    auto sum_of = [](float x) { return both_sum(rows_beside(__float_as_uint(row16_sum(x)))); };
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, den = 0.f, M = -INFINITY;
    for (uint32_t p0 = 0; p0 < parts; p0 += 32) {
        const float2 st = p0 + c8 < parts ? states[(p0 + c8) * stride + pair] : make_float2(-INFINITY, 0.f);   // a part can hold no visible token
        const float top = fmaxf(M, top_of(st.x)), base = top == -INFINITY ? 0.f : top;
        if (p0) {
            const float keep = exp_of(M - base);
            den *= keep;
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] *= keep;
        }
        M = top;
        const float w = exp_of(st.x - base);
        den += sum_of(w * st.y);
        const uint32_t n = min(parts - p0, 32u);
        for (uint32_t i0 = 0; i0 < n; i0 += kAhead) {
            float4 a[kAhead], b[kAhead];
#pragma unroll
            for (uint32_t i = 0; i < kAhead; ++i) {
                a[i] = b[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (i0 + i < n) {
                    const float* src = part_o + ((p0 + i0 + i) * stride + pair) * HD + 8 * c8;
                    a[i] = *reinterpret_cast<const float4*>(src); b[i] = *reinterpret_cast<const float4*>(src + 4);
                }
            }
#pragma unroll
            for (uint32_t i = 0; i < kAhead; ++i) {
                const float wi = __shfl(w, (threadIdx.x & 32u) + min(i0 + i, 31u), kWave), f = i0 + i < n ? wi : 0.f;
                if (f == 0.f) continue;   // nothing of a part without tokens, whatever it left
                v[0] = fmaf(f, a[i].x, v[0]); v[1] = fmaf(f, a[i].y, v[1]); v[2] = fmaf(f, a[i].z, v[2]); v[3] = fmaf(f, a[i].w, v[3]);
                v[4] = fmaf(f, b[i].x, v[4]); v[5] = fmaf(f, b[i].y, v[5]); v[6] = fmaf(f, b[i].z, v[6]); v[7] = fmaf(f, b[i].w, v[7]);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] /= den * kProbScale;
    emit_attention(to, v, pair / q_heads, rows, pair % q_heads, q_heads, c8);
}

// ring[(position + row) & mask] = run[row] for the rows that survive in a ring of this capacity.
// Rows move as 16-byte pieces asked for at 4-byte alignment: a ring may be a view that starts at any word of its
// allocation (the reference's caches are, tests/tensor/gemma3_metal_tests.cpp:765-774).
__global__ void publish_run_kernel(const U4a4* __restrict__ run_k, const U4a4* __restrict__ run_v,
                                   U4a4* __restrict__ ring_k, U4a4* __restrict__ ring_v, uint32_t rows,
                                   uint32_t first_row, uint32_t position, uint32_t ring_mask, uint32_t row_vec) {
    const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= uint64_t(rows - first_row) * row_vec) return;
    const uint32_t row = first_row + static_cast<uint32_t>(i / row_vec), c = static_cast<uint32_t>(i % row_vec);
    const size_t dst = size_t((position + row) & ring_mask) * row_vec + c;
    ring_k[dst] = run_k[size_t(row) * row_vec + c];
    ring_v[dst] = run_v[size_t(row) * row_vec + c];
}

// dst[(position + t) & dst_mask] = src[(position + t) & src_mask], keys and values
__global__ void kv_cache_copy_kernel(const U4a4* __restrict__ src_k, const U4a4* __restrict__ src_v,
                                     U4a4* __restrict__ dst_k, U4a4* __restrict__ dst_v, uint32_t tokens,
                                     uint32_t position, uint32_t src_mask, uint32_t dst_mask, uint32_t row_vec) {
    const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= uint64_t(tokens) * row_vec) return;
    const uint32_t t = static_cast<uint32_t>(i / row_vec), c = static_cast<uint32_t>(i % row_vec);
    const size_t from = size_t((position + t) & src_mask) * row_vec + c, to = size_t((position + t) & dst_mask) * row_vec + c;
    dst_k[to] = src_k[from];
    dst_v[to] = src_v[from];
}

// The same for every block of a model in one launch: a few rows of a few KB per block are a launch's latency and nothing else, and
// a launch per block made the drafter's transaction and the ticket's commit 18 to 96 of them (48 blocks, two rows: 96 launches
// -> 1).  A Publish reads, saves and overwrites a ring piece in one thread.
constexpr uint32_t kMoveLayers = 64;   // blocks per launch: their rings travel as kernel arguments
struct MoveRings { U4a4* k[kMoveLayers]; U4a4* v[kMoveLayers]; uint64_t local; };
struct MovePath { uint32_t row[kMovePath]; };
template <KvMove MOVE>
__global__ void kv_move_kernel(const MoveRings rings, U4a4* __restrict__ flat_k, U4a4* __restrict__ flat_v, uint32_t flat_rows,
                               const U4a4* __restrict__ priv_k, const U4a4* __restrict__ priv_v, uint32_t priv_rows, const MovePath path,
                               uint32_t first, uint32_t mask_local, uint32_t mask_global, uint32_t row_vec) {
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x, layer = blockIdx.y, t = blockIdx.z;
    if (c >= row_vec) return;
    const uint32_t mask = (rings.local >> layer) & 1u ? mask_local : mask_global, position = first + t;
    const size_t ring = size_t(position & mask) * row_vec + c, flat = (size_t(layer) * flat_rows + (position & (flat_rows - 1u))) * row_vec + c;
    U4a4 *rk = rings.k[layer] + ring, *rv = rings.v[layer] + ring;
    if constexpr (MOVE == KvMove::Restore) {
        *rk = flat_k[flat];
        *rv = flat_v[flat];
    } else {
        if constexpr (MOVE != KvMove::Put) {
            flat_k[flat] = *rk;
            flat_v[flat] = *rv;
        }
        if constexpr (MOVE == KvMove::Publish || MOVE == KvMove::Put) {
            const size_t from = (size_t(layer) * priv_rows + path.row[t]) * row_vec + c;
            *rk = priv_k[from];
            *rv = priv_v[from];
        }
    }
}

}  // namespace

int kv_move_rows(hipStream_t s, const guffin_model_desc& m, KvMove move, void* flat_k, void* flat_v, uint32_t flat_rows, uint32_t first,
                 uint32_t count, const void* priv_k, const void* priv_v, uint32_t priv_rows, const uint32_t* path) {
    if (count == 0) return GUFFIN_OK;
    const uint32_t kvw = m.kv_heads * m.head_dim, row_vec = kvw / 8;
    if ((move != KvMove::Put && count > flat_rows) || count > m.ring_local || count > m.ring_global)
        return fail(GUFFIN_E_CAPACITY, "kv_move_rows: more rows than one side holds");
    MovePath rows {};
    if (move == KvMove::Publish || move == KvMove::Put) {
        if (count > kMovePath) return fail(GUFFIN_E_CAPACITY, "kv_move_rows: a path of at most 8 rows");
        for (uint32_t i = 0; i < count; ++i) rows.row[i] = path[i];
    }
    for (uint32_t l = 0; l < m.layer_count; ++l) {   // nothing moves unless everything can
        const guffin_layer_desc& L = m.layers[l];
        if (!L.ring_k || !L.ring_v) return fail(GUFFIN_E_ARG, "kv_move_rows: every layer needs its rings");
        if ((reinterpret_cast<uintptr_t>(L.ring_k) | reinterpret_cast<uintptr_t>(L.ring_v)) & 3u)
            return fail(GUFFIN_E_ALIGN, "kv_move_rows: rows must be 4-byte aligned");
    }
    for (uint32_t l0 = 0; l0 < m.layer_count; l0 += kMoveLayers) {
        const uint32_t n = std::min(kMoveLayers, m.layer_count - l0);
        MoveRings r {};
        for (uint32_t i = 0; i < n; ++i) {
            const guffin_layer_desc& L = m.layers[l0 + i];
            r.k[i] = static_cast<U4a4*>(L.ring_k);
            r.v[i] = static_cast<U4a4*>(L.ring_v);
            if (layer_is_local(m.global_period, l0 + i)) r.local |= uint64_t{1} << i;
        }
        const size_t flat_at = size_t(l0) * flat_rows * row_vec, priv_at = size_t(l0) * priv_rows * row_vec;
        U4a4 *fk = flat_k ? static_cast<U4a4*>(flat_k) + flat_at : nullptr, *fv = flat_v ? static_cast<U4a4*>(flat_v) + flat_at : nullptr;
        const U4a4 *pk = priv_k ? static_cast<const U4a4*>(priv_k) + priv_at : nullptr, *pv = priv_v ? static_cast<const U4a4*>(priv_v) + priv_at : nullptr;
        const dim3 grid((row_vec + 255) / 256, n, count), block(std::min(row_vec, 256u));
#define GUFFIN_MOVE(M) launch(kv_move_kernel<M>, grid, block, 0, s, r, fk, fv, flat_rows, pk, pv, priv_rows, rows, first, m.ring_local - 1, m.ring_global - 1, row_vec)
        if (move == KvMove::Save) GUFFIN_MOVE(KvMove::Save);
        else if (move == KvMove::Restore) GUFFIN_MOVE(KvMove::Restore);
        else if (move == KvMove::Put) GUFFIN_MOVE(KvMove::Put);
        else GUFFIN_MOVE(KvMove::Publish);
#undef GUFFIN_MOVE
        if (int rc = check_launch("kv_move_rows")) return rc;
    }
    return GUFFIN_OK;
}

}  // namespace guffin

using namespace guffin;

extern "C" int guffin_hip_kv_cache_copy(void* stream, const void* src_k, const void* src_v, void* dst_k, void* dst_v,
                                        uint32_t position, uint32_t tokens, uint32_t src_mask, uint32_t dst_mask,
                                        uint32_t row_width) {
    if (!src_k || !src_v || !dst_k || !dst_v) return fail(GUFFIN_E_ARG, "kv_cache_copy: null pointer");
    if (tokens == 0 || row_width == 0 || row_width % 8 != 0) return fail(GUFFIN_E_SHAPE, "kv_cache_copy: row width must be a multiple of 8 halves");
    if ((src_mask & (src_mask + 1)) != 0 || (dst_mask & (dst_mask + 1)) != 0)
        return fail(GUFFIN_E_ARG, "kv_cache_copy: row masks must be a power of two minus one");
    if (tokens > src_mask + 1 || tokens > dst_mask + 1) return fail(GUFFIN_E_CAPACITY, "kv_cache_copy: more tokens than rows on one side");
    if (((reinterpret_cast<uintptr_t>(src_k) | reinterpret_cast<uintptr_t>(src_v) | reinterpret_cast<uintptr_t>(dst_k)
          | reinterpret_cast<uintptr_t>(dst_v)) & 3u) != 0)
        return fail(GUFFIN_E_ALIGN, "kv_cache_copy: rows must be 4-byte aligned");
    const uint64_t n = uint64_t(tokens) * (row_width / 8);
    launch(kv_cache_copy_kernel, dim3(static_cast<uint32_t>((n + 255) / 256)), dim3(256), 0, as_stream(stream),
                       static_cast<const U4a4*>(src_k), static_cast<const U4a4*>(src_v), static_cast<U4a4*>(dst_k),
                       static_cast<U4a4*>(dst_v), tokens, position, src_mask, dst_mask, row_width / 8);
    return check_launch("kv_cache_copy");
}

extern "C" int guffin_hip_publish_run(void* stream, const void* run_k, const void* run_v, void* ring_k, void* ring_v,
                                      uint32_t rows, uint32_t position, uint32_t ring_mask, uint32_t row_width) {
    if (!run_k || !run_v || !ring_k || !ring_v) return fail(GUFFIN_E_ARG, "publish_run: null pointer");
    if (rows == 0 || row_width == 0 || row_width % 8 != 0) return fail(GUFFIN_E_SHAPE, "publish_run: row width must be a multiple of 8 halves");
    if ((ring_mask & (ring_mask + 1)) != 0) return fail(GUFFIN_E_ARG, "publish_run: ring capacity must be a power of two");
    if (((reinterpret_cast<uintptr_t>(run_k) | reinterpret_cast<uintptr_t>(run_v) | reinterpret_cast<uintptr_t>(ring_k)
          | reinterpret_cast<uintptr_t>(ring_v)) & 3u) != 0)
        return fail(GUFFIN_E_ALIGN, "publish_run: rows must be 4-byte aligned");
    const uint32_t first = rows > ring_mask + 1 ? rows - (ring_mask + 1) : 0;  // older rows would be overwritten anyway
    const uint64_t n = uint64_t(rows - first) * (row_width / 8);
    launch(publish_run_kernel, dim3(static_cast<uint32_t>((n + 255) / 256)), dim3(256), 0, as_stream(stream),
                       static_cast<const U4a4*>(run_k), static_cast<const U4a4*>(run_v), static_cast<U4a4*>(ring_k),
                       static_cast<U4a4*>(ring_v), rows, first, position, ring_mask, row_width / 8);
    return check_launch("publish_run");
}

namespace {
// A tiles and waves of a workgroup, parts of the key range.  Two tiles read a key and a value row once for twice the queries, so they
// stay while they leave a workgroup per compute unit; a short run takes single tiles (half the accumulators, half the merge)
// and parts: two workgroups per compute unit, every wave of a part with a tile of its own.
struct AttentionCut { uint32_t tiles, parts, waves; };
AttentionCut attention_cut(uint32_t rows, uint32_t T, uint32_t kv_heads, uint32_t group) {
    const uint32_t pairs = rows * group, twos = (pairs + 31) / 32 * kv_heads, ones = (pairs + 15) / 16 * kv_heads;
    const uint32_t cus = compute_units();
    if (twos >= cus) return {2, 1, 4};
    // (one tile more than a wave each would be a second round for one of them: 37 rows behind 1500 tokens, 34 tiles in eight
    // parts 16.4 us, in nine 14.4; a second part costs the launch that merges them, more than a second round)
    const uint32_t parts = std::max(1u, std::min(2 * cus / ones, T < 256 ? 1 : (T + 127) / 128));
    // Two parts are eight waves of one workgroup, which merges them itself: 1000 rows of the drafter 2025 -> 1934 us a pass, 256 of the 12B
    // shapes 15442 -> 15107.  More parts in half as many such workgroups: 12 rows behind 1500 tokens 4659 -> 4793, 96 8516 -> 9083.
    return parts == 2 ? AttentionCut {1, 1, 8} : AttentionCut {1, parts, 4};
}
uint64_t transposed_bytes(uint32_t T, uint32_t kv_heads) { return (uint64_t(kv_heads) * 256 * T * 2 + 255) & ~uint64_t{255}; }
uint64_t state_bytes(uint32_t parts, uint32_t rows, uint32_t heads) { return parts > 1 ? uint64_t(parts) * rows * heads * (256 + 2) * 4 : 0; }
// The most bytes of states of any run of up to `rows` rows that sees at most T tokens.  Runs of as many single tiles are cut into as many
// parts, the longest of them has the most rows; from a number of tiles on none is cut.
uint64_t most_state_bytes(uint32_t rows, uint32_t T, uint32_t kv_heads, uint32_t group) {
    uint64_t most = 0;
    for (uint32_t tiles = 1; tiles * kv_heads <= 2 * compute_units(); ++tiles) {
        const uint32_t last = std::min(rows, 16 * tiles / group);
        if (last == 0) continue;   // one row takes more
        most = std::max(most, state_bytes(attention_cut(last, T, kv_heads, group).parts, last, kv_heads * group));
        if (last == rows) break;
    }
    return most;
}
}  // namespace

extern "C" uint64_t guffin_hip_prefill_attention_workspace_bytes(uint32_t rows, uint32_t position, uint32_t window,
                                                                 uint32_t kv_heads, uint32_t head_dim) {
    if (rows == 0 || kv_heads == 0 || head_dim != 256) return 0;
    // the values of all visible tokens transposed, then the parts' states (the query heads of a KV head are not known here: 1, 2 or 4)
    const uint32_t T = value_span(rows, position, window).T;
    uint64_t states = 0;
    for (uint32_t group = 1; group <= 4; group *= 2) states = std::max(states, most_state_bytes(rows, T, kv_heads, group));
    return transposed_bytes(T, kv_heads) + states;
}

namespace guffin {
int prefill_attention_init() {
    return allow_lds(prefill_attention_mfma_kernel<1, 4>, attention_lds(1, 4)) && allow_lds(prefill_attention_mfma_kernel<1, 8>, attention_lds(1, 8))
        && allow_lds(prefill_attention_mfma_kernel<2, 4>, attention_lds(2, 4)) ? 0 : -1;
}

bool prefill_attention_on_matrix_core(const void* q, const void* ring_k, const void* ring_v, const void* run_k, const void* run_v,
                                      uint32_t q_heads, uint32_t kv_heads) {
    const uint32_t group = q_heads / kv_heads;
    return (group == 1 || group == 2 || group == 4)
        && ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(ring_k) | reinterpret_cast<uintptr_t>(run_k)
             | reinterpret_cast<uintptr_t>(ring_v) | reinterpret_cast<uintptr_t>(run_v)) & 15u) == 0;
}

uint64_t prefill_attention_bytes(uint32_t rows, uint32_t T, uint32_t q_heads, uint32_t kv_heads) {
    return transposed_bytes(T, kv_heads) + state_bytes(attention_cut(rows, T, kv_heads, q_heads / kv_heads).parts, rows, q_heads);
}
uint64_t prefill_attention_most_bytes(uint32_t rows, uint32_t T, uint32_t q_heads, uint32_t kv_heads) {
    return transposed_bytes(T, kv_heads) + most_state_bytes(rows, T, kv_heads, q_heads / kv_heads);
}

int prefill_attention_run(hipStream_t s, const float* q, const void* ring_k, const void* run_k, float* out, uint8_t* image, uint32_t rows,
                          uint32_t position, uint32_t window, uint32_t ring_mask, uint32_t q_heads, uint32_t kv_heads, float scale,
                          void* workspace) {
    const ValueSpan vs = value_span(rows, position, window);
    const uint32_t group = q_heads / kv_heads, shift = group == 1 ? 0 : group == 2 ? 1 : 2;
    const auto [nt, parts, waves] = attention_cut(rows, vs.T, kv_heads, group);
    if (kv_heads > 0xFFFFu) return fail(GUFFIN_E_SHAPE, "prefill_attention: more KV heads than a grid has rows");
    float* states = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + transposed_bytes(vs.T, kv_heads));
    const AttentionOut to {out, image, states, states + size_t(parts) * rows * q_heads * 256};
    const uint32_t lds = attention_lds(nt, waves);
    const dim3 grid((rows * group + 16 * nt - 1) / (16 * nt) * kv_heads, 1, parts);
    const uint32_t form = kv_heads | (shift << 16) | (parts << 18);   // at most two parts a compute unit
#define GUFFIN_PA(NT_, W_) launch((prefill_attention_mfma_kernel<NT_, W_>), grid, dim3(64 * W_), lds, s, q, static_cast<const uint16_t*>(ring_k), \
                              static_cast<const uint16_t*>(run_k), static_cast<const uint16_t*>(workspace), rows, position, window, ring_mask, \
                              vs.base32, form, scale, vs.T, to)
    if (nt == 2) GUFFIN_PA(2, 4); else if (waves == 8) GUFFIN_PA(1, 8); else GUFFIN_PA(1, 4);
#undef GUFFIN_PA
    if (int rc = check_launch("prefill_attention_mfma")) return rc;
    if (parts == 1) return GUFFIN_OK;
    launch(prefill_attention_merge_kernel, dim3((rows * q_heads + 7) / 8), dim3(256), 0, s, to.part_o, to.part_ml, rows, q_heads, parts, to);
    return check_launch("prefill_attention_merge");
}
}  // namespace guffin

extern "C" int guffin_hip_prefill_attention(void* stream, const float* q, const void* ring_k, const void* ring_v,
                                            const void* run_k, const void* run_v, float* out, uint32_t rows,
                                            uint32_t position, uint32_t window, uint32_t ring_mask,
                                            uint32_t q_heads, uint32_t kv_heads, uint32_t head_dim, float scale,
                                            void* workspace) {
    if (!q || !ring_k || !ring_v || !run_k || !run_v || !out) return fail(GUFFIN_E_ARG, "prefill_attention: null pointer");
    if (rows == 0 || head_dim != 256 || kv_heads == 0 || q_heads % kv_heads != 0)
        return fail(GUFFIN_E_SHAPE, "prefill_attention: head_dim must be 256 and q_heads a multiple of kv_heads");
    if ((ring_mask & (ring_mask + 1)) != 0) return fail(GUFFIN_E_ARG, "prefill_attention: ring capacity must be a power of two");
    const uint32_t past = window ? (window - 1 < position ? window - 1 : position) : position;  // ring tokens a row can see
    if (past > ring_mask + 1) return fail(GUFFIN_E_CAPACITY, "prefill_attention: the ring does not hold the visible past");
    if (!(scale > 0.f)) return fail(GUFFIN_E_ARG, "prefill_attention: scale must be positive");
    if (reinterpret_cast<uintptr_t>(workspace) & 15u) return fail(GUFFIN_E_ALIGN, "prefill_attention: workspace must be 16-byte aligned");
    hipStream_t s = as_stream(stream);
    const uint16_t* rk = static_cast<const uint16_t*>(ring_k);
    const uint16_t* rv = static_cast<const uint16_t*>(ring_v);
    const uint16_t* uk = static_cast<const uint16_t*>(run_k);
    const uint16_t* uv = static_cast<const uint16_t*>(run_v);
    if (workspace && prefill_attention_on_matrix_core(q, ring_k, ring_v, run_k, run_v, q_heads, kv_heads)) {
        // matrix-core path: V^T first, then scores and values as MFMA chains
        const ValueSpan vs = value_span(rows, position, window);
        launch(transpose_values_kernel, dim3(vs.T / 32, kv_heads), dim3(256), 0, s, rv, uv, static_cast<uint16_t*>(workspace), vs.base32, vs.T,
                           vs.first_visible, position, position + rows, ring_mask, kv_heads);
        if (int rc = check_launch("transpose_values")) return rc;
        return prefill_attention_run(s, q, ring_k, run_k, out, nullptr, rows, position, window, ring_mask, q_heads, kv_heads, scale, workspace);
    }
    const uint32_t group = q_heads / kv_heads;
    const dim3 grid((rows + 15) / 16, kv_heads), block(256);
#define GUFFIN_PA(G_) launch(prefill_attention_kernel<G_>, grid, block, 0, s, q, rk, rv, uk, uv, out, rows, \
                                         position, window, ring_mask, q_heads, kv_heads, scale)
    if (group == 1) GUFFIN_PA(1); else if (group == 2) GUFFIN_PA(2); else if (group == 4) GUFFIN_PA(4);
    else return fail(GUFFIN_E_SHAPE, "prefill_attention: q_heads / kv_heads must be 1, 2 or 4");
#undef GUFFIN_PA
    return check_launch("prefill_attention");
}
