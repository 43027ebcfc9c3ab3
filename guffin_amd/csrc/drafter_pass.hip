// The block graph of a decode pass of a narrow Q8_0 model with one KV head -- the drafter -- as one launch of up to 24 blocks, up to
// eight contiguous rows side by side: a row on the 32 CUs of an XCD each.
//
// Operator order per block: the drafter's forward (src/engine/gemma3_draft.mm:888-972).  The placement and the bounded waits are
// those of resident.hip; as there, workgroups hand over through the XCD's L2: plain stores, reads past the L1.
//
// What bounds it: a chain of 18 x 5 phases, each a hand-over and one to two microseconds of dependent steps; the weights alone (5.9 MB
// a block at the 1.3 TB/s that one XCD takes) would be 4.5 us of a block's 11.6.  So the design is about the hand-overs and what lies
// between them:
//
//   * The words themselves are the message.  Every word of a set of exchange buffers is marked empty (kEmpty) by the workgroup that
//     will write it; a reader looks at what it wants until nothing of it is empty.  So a hand-over is a store on its way and the trip
//     of a look, instead of a store, its acknowledgement, an arrival at a counter, a look at that and then the trip for the words (1.05
//     us and the trip).  Two sets by turns; when a set's words may be marked anew stands at publisher().
//   * A wave works from its operand to its partial sums by itself.  It owns three blocks of the hidden width and forms their operand; it
//     merges just the attention outputs that its own two o-projection blocks want and loads just the GeGLU values of its own down
//     blocks.
//   * The last wave takes a row's planes, has the residual in registers and makes both norms of a pair without a meeting: 10 quads'
//     sums and two chains over its lanes.  (Shared by the workers, a meeting each: 0.2 us a pair more.)
//   * Products are exact integers: the quants are int8 as they lie in the tile, an activation is four int8 digits of a 31-bit
//     fixed-point number per group of 32, and v_mfma_i32_4x4x4_16b_i8 multiplies a column's four weights with the four digits
//     of four elements: eight instructions a block, nothing to unpack, no bias to take off again, sums without rounding.  (The
//     fp16 form of the other kernels: some 60 vector instructions a block, 22 bits of an activation.)
//   * A wave's weights of a whole block of the model (15 tiles) have registers of their own and are asked for most of a block
//     ahead, a few tiles behind each phase's own operands: spread evenly, as one XCD takes the 15 in half a block's time, and never
//     right ahead of a wave's own look, which returns behind them.  (Seven of them between the down projection's look and the next
//     q/k/v: 235 us a pass instead of 226.)
//   * Weights are read through the caches' ordinary policy: non-temporal requests take 1200 cycles instead of 700 to come back
//     (2176-byte tiles, one XCD), which is 47 us of a pass.
//   * The eighth wave has no weights.  It adds the workers' partial sums and stores them; so its looks at the planes do not wait
//     behind a weight request.
//   * Attention: a wave a query (four waves are one a SIMD: eight would share the issue slots), a token per 16 lanes with a
//     running softmax of their own, merged over lanes by register swaps; a list's first 20 tokens lie in LDS before the phase,
//     three chunks of 20 more are on their way.
//
//   * Rows depend on each other through keys and values alone.  A row writes a copy of its own past its L2, raises a flag for the block, and
//     the workgroups whose part of the list holds an earlier row's wait for that row's flag and take them over into LDS -- the last
//     wave, which has no weights under way, while the others prepare the queries.  Every row is one hand-over behind the row before
//     from the first block on, so the wait is short after that; and a row's operations are those of a pass by itself.
//
// 270M-shaped model, whole pass at position 150 / 4096 / 8180: one row 225 / 260 / 282 us, two rows 232 / 266 / 287; eight rows appended at 150 312 with
// the host's part.  (With acknowledged stores, a counter, norms shared by the workers and a chunk ahead through their registers 288 / 342 /
// 387, 302 / 346 / 392, 379; resident_blocks_kernel, three launches: one row 606 / 652, two 777 / 888; one launch per operator: 559 / 581 and 609 / 653.)
// rms error of the hidden row against 64 bits, one block, where no K/V rounding falls the other way: 6.2e-8 (6.5e-8 before).
#include "common.hpp"
#include "receipt.hpp"
#include "resident.hpp"

#include <algorithm>
#include <cmath>

namespace guffin {
namespace {

constexpr uint32_t kWaves = 8, kThreads = 64 * kWaves;
constexpr uint32_t kWorkers = 7;          // waves with weights; the last one publishes
constexpr uint32_t kParts = 3;            // parts of K in the o and down projections
constexpr uint32_t kMaxWidth = 640;       // hidden width: three blocks a worker
constexpr uint32_t kMaxFfn = 2048;        // a gate / up tile pair a workgroup
constexpr int kOwn = 3, kOwnO = 2, kOwnDown = 4;          // blocks per worker: of the hidden width, of o, of down
constexpr uint32_t kTile = 64 * 34;       // a wave tile of one Q8_0 block (gemv_packed.hip has the layout)
constexpr uint32_t kChunk = 20;           // tokens whose keys and values lie in LDS together (a window of 512: 17 a workgroup)
constexpr uint32_t kSlots = 4;            // chunks in LDS: one in work, three on their way (60 requests of 63 that a wave can have)

constexpr uint32_t kMl = 32;              // words between two workgroups' maxima and sums: a cache line each
constexpr uint32_t kEmpty = 0xFFFFFFFFu;  // a word that nobody has handed over yet

constexpr uint32_t kLine = 64;            // words between the counters of two rows
constexpr uint32_t kLayers = 24;          // blocks per launch (their pointers travel as kernel arguments)
constexpr uint32_t kFlagsAt = kRunRows * kLine, kSyncWords = kFlagsAt + kLayers * kRunRows;

struct DLayer {
    const uint8_t* tiles[7];                 // q k v o gate up down
    const float* weights[6];                 // post_attention_norm, ffn_norm, post_ffw_norm, the norm that follows the block, q_norm, k_norm
    const uint16_t *ring_k, *ring_v;
    uint32_t local, ring_mask;
};
struct DArgs {
    DLayer layer[kLayers];
    uint32_t layers, rows, H, F;
    float eps, scale;
    uint8_t* exchange;                       // a row's hand-over buffers, two sets by turns; a set's regions, all of them
    uint32_t qkv_at, out_at, ml_at, o_at, d_at, h_at, set_bytes, kv_at, exchange_bytes;
    uint32_t* sync;                          // cleared: a line with a counter for each row, then the rows' flags, block by block
    const float *x_in, *u_in;
    float *x_out, *u_out;                    // written after the last block; u_last, the receipt: the launch with the output norm alone
    float* u_last;                           // the last row's final state, or null
    void* u_receipt_out; uint32_t receipt_rows;  // of all rows, or (1) of the last one
    const float2 *rope_local, *rope_global;
    const uint32_t* schedule;                // of the launch's first block on
    uint16_t *priv_k, *priv_v;               // [block][row][256], of the launch's first block on
    uint32_t* status;
    uint32_t spin_limit;
    unsigned long long* stamps;              // profiling aid: 8 clock readings per block from workgroup 0, or null
};

typedef float f4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
typedef int i4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

struct Shared {
    float red[kWorkers][3][64];                    // the workers' column sums: q/k/v, o and gate, up, down
    float u[kMaxWidth];                            // the normalised row that the next operand is made of
    float2 rope[2][kHd / 2];                       // local, global
    uint32_t opnd[kWorkers][128];                  // a worker's operand: an element's four digits a word
    float mult[kWorkers][4];
    float head[kWaves][kHd];                       // a wave's query (then its output, where several waves share a query)
    float2 ml[kWaves];
    uint16_t k_s[kSlots][kChunk][kHd], v_s[kSlots][kChunk][kHd];   // ring rows of chunks of this workgroup's tokens
    uint16_t kp_s[kRunRows][kHd], vp_s[kRunRows][kHd];   // the private rows among them
    float weight[kWorkers][kGroups];               // a worker's partition weights, those of lane group g at 8 g ..
    uint32_t schedule[kLayers][4];                 // first ring position, ring count, first private row, private rows (this one the last)
    uint32_t dead;
};

// the workgroup meets; LDS accesses are done, loads stay in flight
__device__ __forceinline__ void meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// what this wave wrote to LDS may be read by its other lanes
__device__ __forceinline__ void own_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
// everything this wave has asked for is there (what it asks for next does not hold up what the chain waits for)
__device__ __forceinline__ void arrived() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// the other operand order of the xor-16 / xor-32 exchange, on the vector unit
__device__ __forceinline__ float swap16_sum(float v) {
    const u2_t r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r.x) + __uint_as_float(r.y);
}
__device__ __forceinline__ float swap32_sum(float v) {
    const u2_t r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r.x) + __uint_as_float(r.y);
}
__device__ __forceinline__ float swap16_max(float v) {
    const u2_t r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r.x), __uint_as_float(r.y));
}
__device__ __forceinline__ float swap32_max(float v) {
    const u2_t r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r.x), __uint_as_float(r.y));
}
__device__ __forceinline__ float lanes_sum(float v) { return swap32_sum(swap16_sum(row16_sum(v))); }

// ---- weights ---------------------------------------------------------------------------------------------
// A lane's column of one block: its 32 quants in order, its scale.
struct Tile { u2_t q[4]; uint32_t d; };
__device__ __forceinline__ uint32_t tile_lane(uint32_t lane) { return (lane >> 5) * 1024u + (lane & 15u) * 16u + ((lane >> 4) & 1u) * 8u; }
using Global = const __attribute__((address_space(1))) uint8_t*;   // (a generic pointer's loads would count as LDS accesses too)
__device__ __forceinline__ void load_tile(Tile& t, Global tile, uint32_t lane) {
    Global p = tile + tile_lane(lane);
#pragma unroll
    for (int s = 0; s < 4; ++s) t.q[s] = *reinterpret_cast<const __attribute__((address_space(1))) u2_t*>(p + 256 * s);
    t.d = *reinterpret_cast<const __attribute__((address_space(1))) uint16_t*>(tile + 2048 + lane * 2);
}
// Block i of a run of `count`; past its end the last one again, unused, so that every wave makes the same requests.  (The uniform
// part of an address stays in scalar registers: left to itself the compiler adds it to the lane's part and keeps the sums of all
// fifteen tiles in vector registers over the loop.)
__device__ __forceinline__ void ask_tile(Tile& t, const uint8_t* run, uint32_t i, uint32_t count, uint32_t lane) {
    Global p = (Global)run + (i < count ? i : max(count, 1u) - 1u) * kTile;
    asm("" : "+s"(p));
    load_tile(t, p, lane);
    asm volatile("" ::: "memory");   // here and not elsewhere
}

// ---- activations -----------------------------------------------------------------------------------------
// Fixed point for a group of 32: |x| < 2^(e+1) with e the exponent of the group's largest, n = x 2^(29-e), |n| < 2^30.  The four
// int8 digits of n (n = sum d_k 256^k, each in [-128, 127]) are the bytes of n + 0x00808080 with the lower three's top bits
// flipped.  A group with an infinity or a NaN gets a NaN for its multiplier.
struct GroupScale { float scale, mult; };
__device__ __forceinline__ GroupScale group_scale(uint32_t largest) {   // bits of the group's largest magnitude
    const uint32_t eb = min(max(largest >> 23, 30u), 254u);
    return {__uint_as_float((283u - eb) << 23), __uint_as_float(largest >= 0x7F800000u ? 0x7FC00000u : (eb - 29u) << 23)};
}
__device__ __forceinline__ uint32_t digits(float x, float scale) { return (static_cast<uint32_t>(static_cast<int>(x * scale)) + 0x00808080u) ^ 0x00808080u; }
__device__ __forceinline__ uint32_t magnitude(float v) { return __float_as_uint(v) & 0x7FFFFFFFu; }

// Four consecutive elements a lane, a group in eight aligned lanes; quad `at` of the wave's operand if `mine`.
__device__ __forceinline__ void put_quad(const f4_t v, uint32_t at, bool mine, uint32_t* opnd, float* mult) {
    uint32_t m = max(max(magnitude(v.x), magnitude(v.y)), max(magnitude(v.z), magnitude(v.w)));
    m = max(m, lane_cross_u32<0xB1, 0xF>(m));
    m = max(m, lane_cross_u32<0x4E, 0xF>(m));
    m = max(m, lane_cross_u32<0x141, 0xF>(m));
    const GroupScale g = group_scale(m);
    if (mine) {
        *reinterpret_cast<uint4*>(opnd + 4 * at) = make_uint4(digits(v.x, g.scale), digits(v.y, g.scale), digits(v.z, g.scale), digits(v.w, g.scale));
        if ((at & 7u) == 0) mult[at >> 3] = g.mult;
    }
}
// The matrix operand of blocks 2v, 2v + 1: lane 4 i + k holds digit k of elements 4i .. 4i + 3.
template <int V>
__device__ __forceinline__ void read_operand(int (&a)[V], const uint32_t* opnd, uint32_t lane) {
    const uint32_t k = lane & 3u, low = 0x0c0c0000u | (k + 4u) << 8 | k, high = (k + 4u) << 24 | k << 16 | 0x00000c0cu;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const uint4 w = *reinterpret_cast<const uint4*>(opnd + 64 * v + 4 * (lane >> 2));
        a[v] = static_cast<int>(__builtin_amdgcn_perm(w.y, w.x, low) | __builtin_amdgcn_perm(w.w, w.z, high));
    }
}

// digit sums by weight, the small ones first
__device__ __forceinline__ float digit_value(const i4_t D) {
    float f = fmaf(static_cast<float>(D[1]), 256.f, static_cast<float>(D[0]));
    f = fmaf(static_cast<float>(D[2]), 65536.f, f);
    return fmaf(static_cast<float>(D[3]), 16777216.f, f);
}
// elements 4 STEP .. 4 STEP + 3 of every block: the chains of the blocks side by side
template <int STEP, int N, int V, int I = 0>
__device__ __forceinline__ void step(const Tile (&t)[N], const int (&a)[V], i4_t (&D)[N]) {
    if constexpr (I < N) {
        const int w = static_cast<int>((STEP & 1) ? t[I].q[STEP >> 1].y : t[I].q[STEP >> 1].x);
        D[I] = __builtin_amdgcn_mfma_i32_4x4x4i8(a[I >> 1], w, STEP == 0 ? i4_t{0, 0, 0, 0} : D[I], 4, 8 * (I & 1) + STEP, 0);
        step<STEP, N, V, I + 1>(t, a, D);
    }
}
template <int N, int V, int STEP = 0>
__device__ __forceinline__ void steps(const Tile (&t)[N], const int (&a)[V], i4_t (&D)[N]) {
    if constexpr (STEP < 8) { step<STEP>(t, a, D); steps<N, V, STEP + 1>(t, a, D); }
}
// this lane's column over the wave's `count` blocks, in block order
template <int N>
__device__ __forceinline__ float fold(const Tile (&t)[N], uint32_t count, const i4_t (&D)[N], const float (&mult)[4]) {
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float sum = fmaf(h2f(t[i].d) * mult[i], digit_value(D[i]), acc);
        acc = uint32_t(i) < count ? sum : acc;
    }
    return acc;
}

// how `total` items are dealt to `ways`: the first ones get one more
struct Share { uint32_t first, count; };
__device__ __forceinline__ Share share_of(uint32_t total, uint32_t ways, uint32_t i) {
    const uint32_t base = total / ways, more = total % ways;
    return {i * base + min(i, more), base + (i < more ? 1u : 0u)};
}

// ---- attention -------------------------------------------------------------------------------------------
// The tokens of a block's row (ring rows, then private rows of the launch's rows up to this one) and this workgroup's part of them.
struct Tokens { uint32_t first, n_ring, priv_first, priv_count, t0, t1, mask; };

__device__ __forceinline__ Tokens tokens_of(const Shared& sh, uint32_t l, uint32_t mask, uint32_t slot) {
    Tokens t;
    t.first = uniform(sh.schedule[l][0]); t.n_ring = uniform(sh.schedule[l][1]);
    t.priv_first = uniform(sh.schedule[l][2]); t.priv_count = uniform(sh.schedule[l][3]);
    const uint32_t total = t.n_ring + t.priv_count, per = (total + kGroups - 1) / kGroups;
    t.t0 = min(slot * per, total); t.t1 = min(t.t0 + per, total);
    t.mask = mask;
    return t;
}

// Where lane's 16 bytes of a chunk's rows 2 pair, 2 pair + 1 lie in a ring, half a wave a row.  Asked for through a buffer resource: lanes
// past the last token ask beyond its end, which reads zeros and touches no memory.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ring_of(const uint16_t* ring, const Tokens& t) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(ring), 0, static_cast<int>((t.mask + 1) * (2 * kHd)), 0x00020000);
}
__device__ __forceinline__ int ring_place(const Tokens& t, uint32_t chunk, uint32_t pair, uint32_t lane) {
    const uint32_t token = chunk + 2 * pair + (lane >> 5);
    return token < t.t1 && token < t.n_ring ? static_cast<int>(((t.first + token) & t.mask) * (2 * kHd) + 16 * (lane & 31u)) : -1024;
}
// A worker's share of the first chunk: up to three of its 20 pairs of rows (ten of keys, ten of values).
struct Rows { uint4 v[3]; };
__device__ __forceinline__ void ask_rows(Rows& to, const uint16_t* ring_k, const uint16_t* ring_v, const Tokens& t, uint32_t wave, uint32_t lane) {
#pragma unroll
    for (uint32_t i = 0; i < 3; ++i) {
        const uint32_t pair = wave + kWorkers * i;
        const int at = pair < kChunk ? ring_place(t, t.t0, pair % (kChunk / 2), lane) : -1024;
        to.v[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(ring_of(pair < kChunk / 2 ? ring_k : ring_v, t), at, 0, 0));
    }
}
__device__ __forceinline__ void put_rows(Shared& sh, const Rows& from, uint32_t wave, uint32_t lane) {
#pragma unroll
    for (uint32_t i = 0; i < 3; ++i) {
        const uint32_t pair = wave + kWorkers * i, row = 2 * (pair % (kChunk / 2)) + (lane >> 5);
        if (pair < kChunk) *reinterpret_cast<uint4*>(&(pair < kChunk / 2 ? sh.k_s : sh.v_s)[0][row][8 * (lane & 31u)]) = from.v[i];
    }
}
// chunk `number` of the list (not the first) straight into its place in LDS, by one wave: kChunk requests.  (Requests into LDS want
// whole 16 bytes: rings that lie off them go through the wave's registers.)
__device__ __forceinline__ void ask_chunk(Shared& sh, const uint16_t* ring_k, const uint16_t* ring_v, const Tokens& t, uint32_t number, uint32_t lane) {
    const __amdgpu_buffer_rsrc_t keys = ring_of(ring_k, t), values = ring_of(ring_v, t);
    const uint32_t slot = number % kSlots;
    if ((reinterpret_cast<uintptr_t>(ring_k) | reinterpret_cast<uintptr_t>(ring_v)) & 15u) {
#pragma unroll 1
        for (uint32_t pair = 0; pair < kChunk / 2; ++pair) {
            const int at = ring_place(t, t.t0 + kChunk * number, pair, lane);
            const uint4 k = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(keys, at, 0, 0));
            const uint4 v = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(values, at, 0, 0));
            *reinterpret_cast<uint4*>(&sh.k_s[slot][2 * pair + (lane >> 5)][8 * (lane & 31u)]) = k;
            *reinterpret_cast<uint4*>(&sh.v_s[slot][2 * pair + (lane >> 5)][8 * (lane & 31u)]) = v;
        }
        return;
    }
#pragma unroll
    for (uint32_t pair = 0; pair < kChunk / 2; ++pair) {
        const int at = ring_place(t, t.t0 + kChunk * number, pair, lane);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(keys, (__attribute__((address_space(3))) void*)&sh.k_s[slot][2 * pair][0], 16, at, 0, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(values, (__attribute__((address_space(3))) void*)&sh.v_s[slot][2 * pair][0], 16, at, 0, 0, 0);
    }
}

// Head norm and rotation of 256 values, dimensions 2l, 2l+1, 128 + 2l, 128 + 2l + 1 a lane.
struct HeadNorm { float2 lo, hi; };
__device__ __forceinline__ HeadNorm load_head_norm(const float* p, uint32_t lane) {
    HeadNorm g;
    g.lo = make_float2(p[2 * lane], p[2 * lane + 1]); g.hi = make_float2(p[128 + 2 * lane], p[128 + 2 * lane + 1]);
    return g;
}
__device__ __forceinline__ void norm_rotate(float (&v)[4], const HeadNorm& gamma, const float2* rope, float eps, uint32_t lane) {
    const float ss = lanes_sum(fmaf(v[3], v[3], fmaf(v[2], v[2], fmaf(v[1], v[1], v[0] * v[0]))));
    const float inv = 1.0f / sqrtf(ss / 256.0f + eps);
    const float g[4] = {gamma.lo.x, gamma.lo.y, gamma.hi.x, gamma.hi.y};
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = v[k] * inv * g[k];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const float2 cs = rope[2 * lane + k];
        const float first = v[k], second = v[k + 2];
        v[k] = __fsub_rn(__fmul_rn(first, cs.x), __fmul_rn(second, cs.y));
        v[k + 2] = __fadd_rn(__fmul_rn(first, cs.y), __fmul_rn(second, cs.x));
    }
}

template <int G>
struct Pass {
    static constexpr uint32_t CW = (G + 2) * kHd, TA = 4 * G + 8;
    // Four waves attend, WPQ of them a query: one a SIMD (eight would share its issue slots).  Two more prepare the row's key and value.
    static constexpr uint32_t WPQ = 4 / G, ATTENDING = 4, PREPARING = 4;
    static constexpr uint32_t STEP = 4 * WPQ;                                  // tokens of a round
    const DArgs& a;
    Shared& sh;
    uint32_t lane;
    const uint32_t wave, slot, row;
    const float per_width;
    __amdgpu_buffer_rsrc_t exchange;

    // What another workgroup stored during this launch: past this CU's L1 (sc1), which nothing invalidates, from the L2.
    static constexpr int kPast = 16;
    __device__ __forceinline__ f4_t ld4(uint32_t at, uint32_t floats) const {
        return __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(exchange, static_cast<int>(4 * floats), static_cast<int>(at), kPast));
    }
    __device__ __forceinline__ float2 ld2(uint32_t at, uint32_t floats) const {
        return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(exchange, static_cast<int>(4 * floats), static_cast<int>(at), kPast));
    }
    // (a NaN of every bit, which a weight could bring, goes as the usual one: the others would wait for it)
    static __device__ __forceinline__ uint32_t sealed(float v) {
        const uint32_t bits = __float_as_uint(v);
        return bits == kEmpty ? 0x7FC00000u : bits;
    }
    __device__ __forceinline__ void st_bits(uint32_t at, uint32_t floats, uint32_t v) const {
        __builtin_amdgcn_raw_buffer_store_b32(v, exchange, static_cast<int>(4 * floats), static_cast<int>(at), 0);
    }
    __device__ __forceinline__ void st(uint32_t at, uint32_t floats, float v) const { st_bits(at, floats, sealed(v)); }
    __device__ __forceinline__ void st2(uint32_t at, uint32_t floats, float2 v) const {
        __builtin_amdgcn_raw_buffer_store_b64(u2_t{sealed(v.x), sealed(v.y)}, exchange, static_cast<int>(4 * floats), static_cast<int>(at), 0);
    }
    __device__ __forceinline__ void st4_bits(uint32_t at, uint32_t floats, u4_t v) const {
        __builtin_amdgcn_raw_buffer_store_b128(v, exchange, static_cast<int>(4 * floats), static_cast<int>(at), 0);
    }
    __device__ __forceinline__ void st4(uint32_t at, uint32_t floats, f4_t v) const {
        st4_bits(at, floats, u4_t{sealed(v.x), sealed(v.y), sealed(v.z), sealed(v.w)});
    }
    // whether a word of these is still to come, for any lane
    static __device__ __forceinline__ bool empty(float2 v) { return __any(max(__float_as_uint(v.x), __float_as_uint(v.y)) == kEmpty); }
    static __device__ __forceinline__ bool empty(f4_t v) {
        return __any(max(max(__float_as_uint(v.x), __float_as_uint(v.y)), max(__float_as_uint(v.z), __float_as_uint(v.w))) == kEmpty);
    }
    // after a look that found something missing: whether to look again
    __device__ __forceinline__ bool again(uint32_t& looks) const {
        asm volatile("" ::: "memory");
        if (sh.dead) return false;
        if (++looks <= a.spin_limit) return true;
        if (lane == 0) give_up();
        return false;
    }
    __device__ __forceinline__ uint32_t set_of(uint32_t l) const { return (l & 1u) * a.set_bytes; }

    __device__ __forceinline__ void enter() { lane = opaque(lane); }   // or every address that depends on the lane alone is kept in a register over the loop
    __device__ __forceinline__ void stamp(uint32_t l, uint32_t phase) const {
        if (a.stamps && row == 0 && slot == 0 && lane == 0) a.stamps[l * 16 + phase] = wall_clock64();
    }

    __device__ __forceinline__ void give_up() const { sh.dead = 1u; atomicOr(a.status, GUFFIN_STATUS_SYNC); }
    // The last wave, once a launch: its stores (both sets marked empty) are in the L2, then the arrival, then the wait for the other
    // workgroups.  A wait that gives up raises the status bit, and the workgroup waits no more for the rest of the launch.
    __device__ __forceinline__ void arrive_and_wait() const {
        __builtin_amdgcn_s_waitcnt(0);
        if (lane == 0 && !sh.dead) {
            uint32_t* counter = a.sync + row * kLine;
            __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            uint32_t spins = 0;
            while (__hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < kGroups)
                if (++spins > a.spin_limit) { give_up(); break; }
        }
        asm volatile("" ::: "memory");
    }
    __device__ __forceinline__ float workers_sum(int matrix) const {
        float s = sh.red[0][matrix][lane];
#pragma unroll
        for (uint32_t w = 1; w < kWorkers; ++w) s += sh.red[w][matrix][lane];
        return s;
    }

    // ---- rows of the same launch: the last wave hands keys and values on, 16 bytes a lane, keys in the lower half of the wave ----
    using Words = uint32_t __attribute__((ext_vector_type(4)));
    // (a copy of its own per block: a row may be blocks ahead of its readers, and the caller's rows need not lie on 8 bytes)
    __device__ __forceinline__ uint16_t* passed_on(uint32_t l, uint32_t r) const {
        return reinterpret_cast<uint16_t*>(a.exchange + size_t(r) * a.exchange_bytes + a.kv_at) + (size_t(l) * 64 + lane) * 8;
    }
    __device__ __forceinline__ uint16_t* staged(uint32_t i) const { return (lane < 32 ? sh.kp_s[i] : sh.vp_s[i]) + 8 * (lane & 31u); }
    // this row's, for the XCDs of later rows: past this L2 (sc1), then the flag
    __device__ __forceinline__ void hand_on(uint32_t l, uint32_t i) const {
        const uint2* from = reinterpret_cast<const uint2*>(staged(i));
        unsigned long long* to = reinterpret_cast<unsigned long long*>(passed_on(l, row));
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint2 w = from[h];
            __hip_atomic_store(to + h, w.x | static_cast<unsigned long long>(w.y) << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __builtin_amdgcn_s_waitcnt(0);
        asm volatile("" ::: "memory");
        if (lane == 0) __hip_atomic_store(a.sync + kFlagsAt + l * kRunRows + row, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // those of the private rows [from, to), counted from the first one attended, into their places in LDS
    __device__ __forceinline__ void take_over(uint32_t l, const Tokens& t, uint32_t from, uint32_t to) const {
        if (lane >= from && lane < to && !sh.dead) {
            const uint32_t* flag = a.sync + kFlagsAt + l * kRunRows + t.priv_first + lane;
            uint32_t spins = 0;
            while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
                if (++spins > a.spin_limit) { give_up(); break; }
        }
        asm volatile("" ::: "memory");
        for (uint32_t i0 = from; i0 < to; i0 += 4) {
            unsigned long long w[4][2];
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {   // past the last one the last again, unused
                const unsigned long long* p = reinterpret_cast<const unsigned long long*>(passed_on(l, t.priv_first + min(i0 + i, to - 1)));
                w[i][0] = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                w[i][1] = __hip_atomic_load(p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i)
                if (i0 + i < to) {
                    unsigned long long* p = reinterpret_cast<unsigned long long*>(staged(i0 + i));
                    p[0] = w[i][0]; p[1] = w[i][1];
                }
        }
    }

    // What a wave's part in a block's attention needs and does not depend on the pass, asked for a phase ahead.
    __device__ __forceinline__ HeadNorm ask_gamma(const DLayer& L) const {
        return load_head_norm(L.weights[wave == PREPARING ? 5 : 4], lane);
    }

    // Every query of the row against this workgroup's tokens; a token per 16 lanes, lane s of them with dimensions 8s .. 8s+7 and 128 +
    // 8s .. 128 + 8s + 7.  The first chunk's rows lie in LDS; the others are the last wave's to bring (LAST), which has nothing else under
    // way, three of them ahead of the one in work (position 4096, seven chunks: 9.2 us a block instead of 15.0 with one ahead through
    // registers of the workers, rounds one after the other; 4.9 of it would be the rows alone).
    template <bool LAST, typename First, typename Second>
    __device__ __forceinline__ void attend(uint32_t l, const DLayer& L, const Tokens& t, const HeadNorm& gamma, First first_request, Second second_request) {
        constexpr uint32_t ROUNDS = (kChunk + STEP - 1) / STEP;
        const uint32_t query = wave / WPQ, s16 = lane & 15u;
        const float2* rope = sh.rope[L.local ? 0 : 1];
        // private rows among this workgroup's tokens: this row's key and value are prepared here, a wave each, earlier rows' come
        // from their XCDs
        const uint32_t chunks = (t.t1 - t.t0 + kChunk - 1) / kChunk;
        if constexpr (LAST)
            for (uint32_t c = 1; c < min(chunks, kSlots); ++c) ask_chunk(sh, L.ring_k, L.ring_v, t, c, lane);
        const uint32_t own = t.priv_count - 1, priv_from = max(t.t0, t.n_ring) - t.n_ring, priv_to = max(t.t1, t.n_ring) - t.n_ring;
        const bool owner = priv_from <= own && own < priv_to, peers = min(priv_to, own) > priv_from;
        const bool prepares = owner && wave >= PREPARING && wave < PREPARING + 2, is_key = wave == PREPARING;
        float2 v0 = make_float2(0.f, 0.f), v1 = v0;
        if (wave < ATTENDING || prepares) {
            const uint32_t src = (wave < ATTENDING ? query : is_key ? G : G + 1) * kHd + 2 * lane, from = set_of(l) + a.qkv_at;
            uint32_t looks = 0;
            do { v0 = ld2(from, src); v1 = ld2(from, src + 128); } while ((empty(v0) || empty(v1)) && again(looks));
        }
        first_request();
        float* q_s = sh.head[wave];
        float v[4] = {v0.x, v0.y, v1.x, v1.y};
        if (wave < ATTENDING) {
            norm_rotate(v, gamma, rope, a.eps, lane);
            *reinterpret_cast<float2*>(q_s + 2 * lane) = make_float2(v[0] * a.scale, v[1] * a.scale);
            *reinterpret_cast<float2*>(q_s + 128 + 2 * lane) = make_float2(v[2] * a.scale, v[3] * a.scale);
        }
        if (prepares) {
            if (is_key) norm_rotate(v, gamma, rope, a.eps, lane);
            bool bad = false;
            uint32_t bits[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const _Float16 hv = static_cast<_Float16>(v[k]);
                bad |= !isfinite(static_cast<float>(hv));
                bits[k] = __builtin_bit_cast(uint16_t, hv);
            }
            uint16_t* to = (is_key ? sh.kp_s : sh.vp_s)[own];
            uint16_t* out = (is_key ? a.priv_k : a.priv_v) + (size_t(l) * a.rows + row) * kHd;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t d = (k >> 1) * 128 + 2 * lane + (k & 1);
                to[d] = static_cast<uint16_t>(bits[k]);
                out[d] = static_cast<uint16_t>(bits[k]);
            }
            if (bad) atomicOr(a.status, GUFFIN_STATUS_KV_NONFINITE);
        }
        if (owner) {
            meet();
            if (wave == kWorkers && row + 1 < a.rows) hand_on(l, own);
        }
        if (peers) {
            if (wave == kWorkers) take_over(l, t, priv_from, min(priv_to, own));
            meet();
        }
        if (!owner && !peers) own_lds();
        second_request();
        f4_t q[4];
        float m = -INFINITY, sum = 0.f, acc[16];
        if (wave < ATTENDING) {
#pragma unroll
            for (int k = 0; k < 4; ++k) q[k] = *reinterpret_cast<const f4_t*>(q_s + 128 * (k >> 1) + 8 * s16 + 4 * (k & 1));
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.f;
        for (uint32_t number = 0; number < chunks; ++number) {
            const uint32_t chunk = t.t0 + kChunk * number, chunk_end = min(chunk + kChunk, t.t1), in_work = number % kSlots;
            if (!LAST && wave < ATTENDING) {
                const uint32_t mine = 4 * (wave % WPQ) + (lane >> 4);   // this lane's token of a round, from the chunk's first
                // a token's row: a private one, or the chunk's (zeros past the last token)
                auto row_at = [&](uint32_t at, const uint16_t (*ring)[kHd], const uint16_t (*priv)[kHd]) {
                    return (chunk + at >= t.n_ring && chunk + at < t.t1 ? priv[chunk + at - t.n_ring] : ring[min(at, kChunk - 1)]) + 8 * s16;
                };
                // N rounds without a branch between them, each row asked for a round ahead, four chains a score: a round by itself
                // is 800 cycles, most of it waiting (position 4096, seven chunks: 9.2 us a block instead of 13.5)
                auto rounds = [&]<uint32_t N>() {
                    float s[N];
                    uint4 ahead[2];   // the next round's key or value
                    auto ask = [&](uint32_t at, const uint16_t (*ring)[kHd], const uint16_t (*priv)[kHd]) {
                        const uint16_t* from = row_at(at, ring, priv);
                        ahead[0] = *reinterpret_cast<const uint4*>(from);
                        ahead[1] = *reinterpret_cast<const uint4*>(from + 128);
                        asm volatile("" ::: "memory");   // here
                        lane = opaque(lane);             // no rounds' addresses kept: there are no registers for them
                    };
                    ask(mine, sh.k_s[in_work], sh.kp_s);
#pragma unroll
                    for (uint32_t u = 0; u < N; ++u) {
                        const uint32_t w[8] = {ahead[0].x, ahead[0].y, ahead[0].z, ahead[0].w, ahead[1].x, ahead[1].y, ahead[1].z, ahead[1].w};
                        if (u + 1 < N) ask(STEP * (u + 1) + mine, sh.k_s[in_work], sh.kp_s);
                        else ask(mine, sh.v_s[in_work], sh.vp_s);
                        float d[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int i = 0; i < 4; ++i)
#pragma unroll
                            for (int p = 0; p < 2; ++p) {
                                const half2_t h2 = __builtin_bit_cast(half2_t, w[4 * p + i]);
                                d[2 * p] = fmaf(static_cast<float>(h2.x), q[2 * p + (i >> 1)][2 * (i & 1)], d[2 * p]);
                                d[2 * p + 1] = fmaf(static_cast<float>(h2.y), q[2 * p + (i >> 1)][2 * (i & 1) + 1], d[2 * p + 1]);
                            }
                        const float dot = row16_sum((d[0] + d[1]) + (d[2] + d[3]));
                        s[u] = chunk + STEP * u + mine < chunk_end ? dot : -INFINITY;
                    }
                    float top = m;
#pragma unroll
                    for (uint32_t u = 0; u < N; ++u) top = fmaxf(top, s[u]);
                    const float base = top == -INFINITY ? 0.f : top;   // nothing attended so far: every weight is zero
                    if (number != 0) {
                        const float keep = expf(m - base);
                        sum *= keep;
#pragma unroll
                        for (int i = 0; i < 16; ++i) acc[i] *= keep;
                    }
                    m = top;
#pragma unroll
                    for (uint32_t u = 0; u < N; ++u) {
                        const float p = expf(s[u] - base);
                        sum += p;
                        const uint32_t w[8] = {ahead[0].x, ahead[0].y, ahead[0].z, ahead[0].w, ahead[1].x, ahead[1].y, ahead[1].z, ahead[1].w};
                        if (u + 1 < N) ask(STEP * (u + 1) + mine, sh.v_s[in_work], sh.vp_s);
#pragma unroll
                        for (int i = 0; i < 8; ++i) {
                            const half2_t h2 = __builtin_bit_cast(half2_t, w[i]);
                            acc[2 * i] = fmaf(static_cast<float>(h2.x), p, acc[2 * i]);
                            acc[2 * i + 1] = fmaf(static_cast<float>(h2.y), p, acc[2 * i + 1]);
                        }
                    }
                };
                if (chunk_end - chunk <= STEP * (ROUNDS / 2)) rounds.template operator()<ROUNDS / 2>();
                else rounds.template operator()<ROUNDS>();
            }
            if (number + 1 < chunks) {   // the next chunk has arrived, and this one's place is another's
                if constexpr (LAST) {
                    const uint32_t younger = min(chunks - 1, number + kSlots - 1) - (number + 1);   // chunks asked for behind the next
                    if (younger == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kChunk) : "memory");
                    else if (younger == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kChunk) : "memory");
                    else arrived();
                }
                meet();
                if constexpr (LAST)
                    if (number + kSlots < chunks) ask_chunk(sh, L.ring_k, L.ring_v, t, number + kSlots, lane);
            }
        }
        if (LAST || wave >= ATTENDING) return;
        // the four token groups of the wave: a common maximum, then halves of the values exchanged for halves of the lanes
        const float top = swap32_max(swap16_max(m)), base = top == -INFINITY ? 0.f : top, f = expf(m - base);
        sum = swap32_sum(swap16_sum(sum * f));
        float e[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const u2_t x = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[i] * f), __float_as_uint(acc[i + 8] * f), false, false);
            e[i] = __uint_as_float(x.x) + __uint_as_float(x.y);
        }
        f4_t o;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const u2_t x = __builtin_amdgcn_permlane16_swap(__float_as_uint(e[i]), __float_as_uint(e[i + 4]), false, false);
            o[i] = __uint_as_float(x.x) + __uint_as_float(x.y);
        }
        const uint32_t at = (lane >> 5) * 128 + 8 * s16 + ((lane >> 4) & 1u) * 4;
        if constexpr (WPQ == 1) {
            st4(set_of(l) + a.out_at, (slot * G + query) * kHd + at, o);
            if (lane == 0) st2(set_of(l) + a.ml_at, slot * kMl + query * 2, make_float2(top, sum));
        } else {
            own_lds();   // the query has been read
            *reinterpret_cast<f4_t*>(q_s + at) = o;
            if (lane == 0) sh.ml[wave] = make_float2(top, sum);
        }
    }

    // the last wave, where several share a query: the queries' outputs over this workgroup's tokens
    __device__ __forceinline__ void publish_attention(uint32_t l) {
#pragma unroll
        for (int n = 0; n < G; ++n) {
            float top = sh.ml[n * WPQ].x;
#pragma unroll
            for (uint32_t j = 1; j < WPQ; ++j) top = fmaxf(top, sh.ml[n * WPQ + j].x);
            const float base = top == -INFINITY ? 0.f : top;
            f4_t o = {0.f, 0.f, 0.f, 0.f};
            float sum = 0.f;
#pragma unroll
            for (uint32_t j = 0; j < WPQ; ++j) {
                const float2 mj = sh.ml[n * WPQ + j];
                const float f = expf(mj.x - base);
                const f4_t oj = *reinterpret_cast<const f4_t*>(&sh.head[n * WPQ + j][4 * lane]);
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = fmaf(oj[i], f, o[i]);
                sum = fmaf(mj.y, f, sum);
            }
            st4(set_of(l) + a.out_at, (slot * G + n) * kHd + 4 * lane, o);
            if (lane == 0) st2(set_of(l) + a.ml_at, slot * kMl + n * 2, make_float2(top, sum));
        }
    }

    // A worker's quads of a row: those of its own blocks, one a lane.
    struct Own { Share blocks; bool on; uint32_t at; };
    // ---- the eighth wave -------------------------------------------------------------------------------------
    // The row in this wave's registers, quads lane, lane + 64, lane + 128 of it (`mine`: the row has them).
    static constexpr int kQuads = kMaxWidth / 256 + 1;
    struct RowQuads { f4_t v[kQuads]; };
    __device__ __forceinline__ bool mine(int i) const { return lane + 64 * i < a.H / 4; }
    __device__ __forceinline__ uint32_t quad_at(int i) const { return 4 * min(lane + 64 * i, a.H / 4 - 1); }
    __device__ __forceinline__ void ask_row(RowQuads& to, const float* p) const {
#pragma unroll
        for (int i = 0; i < kQuads; ++i) { const float4 t = ldf4_a4(p + quad_at(i)); to.v[i] = f4_t{t.x, t.y, t.z, t.w}; }
    }
    // the sum of a projection's planes, once they are there
    __device__ __forceinline__ RowQuads gather(uint32_t planes) const {
        f4_t p[kQuads][kParts];
        uint32_t missing = (1u << (kQuads * kParts)) - 1, looks = 0;
        do {
#pragma unroll
            for (int i = 0; i < kQuads; ++i)
#pragma unroll
                for (uint32_t k = 0; k < kParts; ++k)
                    if (missing >> (kParts * i + k) & 1u) p[i][k] = ld4(planes, k * a.H + quad_at(i));
            uint32_t left = 0;
#pragma unroll
            for (int i = 0; i < kQuads; ++i)
#pragma unroll
                for (uint32_t k = 0; k < kParts; ++k)
                    if (empty(p[i][k])) left |= 1u << (kParts * i + k);
            missing = left;
        } while (missing && again(looks));
        RowQuads r;
#pragma unroll
        for (int i = 0; i < kQuads; ++i) r.v[i] = p[i][0] + p[i][1] + p[i][2];
        return r;
    }
    // 1 / rms of the row
    __device__ __forceinline__ float over_rms(const RowQuads& r) const {
        float ss[kQuads];
#pragma unroll
        for (int i = 0; i < kQuads; ++i) {
            const f4_t& v = r.v[i];
            ss[i] = mine(i) ? fmaf(v.w, v.w, fmaf(v.z, v.z, fmaf(v.y, v.y, v.x * v.x))) : 0.f;
        }
        float all = ss[0];
#pragma unroll
        for (int i = 1; i < kQuads; ++i) all += ss[i];
        return inverse_rms(lanes_sum(all), per_width, a.eps);
    }
    // x = x + rms(v, post), then rms(x, next) for the workers.  outputs: also written to memory (the state after the launch's last block).
    __device__ __forceinline__ void norm_pair(const RowQuads& v, const RowQuads& post, const RowQuads& next, RowQuads& x, bool outputs) const {
        const uint32_t H = a.H;
        float inv = over_rms(v);
#pragma unroll
        for (int i = 0; i < kQuads; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k) x.v[i][k] = fmaf(v.v[i][k] * inv, post.v[i][k], x.v[i][k]);
        inv = over_rms(x);
#pragma unroll
        for (int i = 0; i < kQuads; ++i) {
            const f4_t u = x.v[i] * inv * next.v[i];
            if (mine(i)) {
                *reinterpret_cast<f4_t*>(sh.u + quad_at(i)) = u;
                if (outputs) {
                    const size_t at = size_t(row) * H + quad_at(i);
                    *reinterpret_cast<f4_t*>(a.x_out + at) = x.v[i];
                    *reinterpret_cast<f4_t*>(a.u_out + at) = u;
                    if (a.u_last && row + 1 == a.rows) *reinterpret_cast<f4_t*>(a.u_last + quad_at(i)) = u;
                }
            }
        }
        if (outputs && a.u_receipt_out && (a.receipt_rows > 1 || row + 1 == a.rows)) {
            own_lds();
            for (uint32_t t = lane; t < H / 8; t += 64) {
                float y[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] = sh.u[8 * t + i];
                emit_receipt_values(y, 0, t, a.receipt_rows > 1 ? row : 0u, a.receipt_rows, H, a.u_receipt_out);
            }
        }
    }
    __device__ __forceinline__ void check(const RowQuads& x) const {
        bool bad = false;
#pragma unroll
        for (int i = 0; i < kQuads; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k) bad |= mine(i) && !isfinite(x.v[i][k]);
        if (bad) atomicOr(a.status, GUFFIN_STATUS_NONFINITE);
    }

    __device__ __forceinline__ void publisher() {
        const uint32_t tiles = a.H / 64, part = uniform(slot / tiles), column = (slot - part * tiles) * 64 + lane;
        // this workgroup's words of a set: q/k/v and the attention's, the others'
        auto mark_empty = [&](uint32_t set, bool attention, bool others) {
            if (attention) {
                if (slot < TA) st_bits(set + a.qkv_at, slot * 64 + lane, kEmpty);
#pragma unroll
                for (int n = 0; n < G; ++n) st4_bits(set + a.out_at, (slot * G + n) * kHd + 4 * lane, u4_t{kEmpty, kEmpty, kEmpty, kEmpty});
                if (lane < kMl) st_bits(set + a.ml_at, slot * kMl + lane, kEmpty);
            }
            if (others) {
                if (part < kParts) {
                    st_bits(set + a.o_at, part * a.H + column, kEmpty);
                    st_bits(set + a.d_at, part * a.H + column, kEmpty);
                }
                if (slot < a.F / 64) st_bits(set + a.h_at, slot * 64 + lane, kEmpty);
            }
        };
        mark_empty(0, true, true);
        mark_empty(a.set_bytes, true, true);
        RowQuads x, post, next;
        ask_row(x, a.x_in + size_t(row) * a.H);
        for (uint32_t l = 0; l < a.layers; ++l) {
            const DLayer& L = a.layer[l];
            const uint32_t set = set_of(l);
            enter();
            const Tokens t = tokens_of(sh, l, L.ring_mask, slot);
            const HeadNorm none {};
            stamp(l, 0);
            meet();
            if (slot < TA) st(set + a.qkv_at, slot * 64 + lane, workers_sum(0));
            if (l == 0) { arrive_and_wait(); meet(); }
            ask_row(post, L.weights[0]);
            ask_row(next, L.weights[1]);
            stamp(l, 1);
            attend<true>(l, L, t, none, [] {}, [] {});
            meet();
            if constexpr (WPQ > 1) publish_attention(l);
            stamp(l, 2);
            // o-projection, norm pair
            meet();
            stamp(l, 3);
            if (part < kParts) st(set + a.o_at, part * a.H + column, workers_sum(0));
            RowQuads v = gather(set + a.o_at);
            stamp(l, 4);
            norm_pair(v, post, next, x, false);
            meet();
            check(x);
            ask_row(post, L.weights[2]);
            ask_row(next, L.weights[3]);
            // gate and up
            meet();
            stamp(l, 5);
            if (slot < a.F / 64) st(set + a.h_at, slot * 64 + lane, geglu_value(workers_sum(0), workers_sum(1)));
            // Everybody has read what the block before left, and this block's q/k/v and attention (o says so, whose sums are all here).
            // The next block's words are marked empty here, where they stay in the L2 until they are wanted; those of its first two phases
            // were a block ago already: nobody knows there that this block's stores have been made, but the attention in between does.
            mark_empty(set ^ a.set_bytes, true, true);
            mark_empty(set, true, false);
            stamp(l, 6);
            // down, norm pair
            meet();
            arrived();
            if (part < kParts) st(set + a.d_at, part * a.H + column, workers_sum(2));
            v = gather(set + a.d_at);
            stamp(l, 7);
            norm_pair(v, post, next, x, l + 1 == a.layers && slot == 0);
            meet();
            check(x);
        }
    }

    // ---- the seven others ------------------------------------------------------------------------------------
    __device__ __forceinline__ void worker() {
        const uint32_t H = a.H, F = a.F, nb_h = H / 32, tiles = H / 64;
        Own own;
        own.blocks = share_of(nb_h, kWorkers, wave);             // blocks of the hidden width
        own.blocks.first = min(own.blocks.first, nb_h - 1);      // (no blocks: the last one's requests, unused)
        own.on = lane < 8 * own.blocks.count;
        own.at = 32 * own.blocks.first + (own.on ? 4 * lane : 0u);
        // q/k/v: a column tile a workgroup (workgroups past the last one repeat some tile's requests, unused)
        const uint32_t qt = slot % TA;
        const int qm = qt < 4 * G ? 0 : (qt < 4 * G + 4 ? 1 : 2);
        const uint32_t q_tile = qm == 0 ? qt : qm == 1 ? qt - 4 * G : qt - 4 * G - 4;
        const uint32_t q_at = uniform((q_tile * nb_h + own.blocks.first) * kTile);
        // o: a column tile and a part of K, blocks by pairs (64 elements lie in one head)
        const uint32_t row_part = uniform(slot / tiles), part = row_part < kParts ? row_part : 0, tile = slot - row_part * tiles;
        const Share o_part = share_of(4 * G, kParts, part);
        const bool o_on = wave < o_part.count;
        const bool merges = o_on && row_part < kParts;
        const uint32_t o_pair = uniform(o_part.first + (o_on ? wave : 0u));
        const uint32_t o_at = uniform((tile * (8 * G) + 2 * o_pair) * kTile);
        // gate and up: a tile pair a workgroup
        const uint32_t g_at = uniform(((slot % (F / 64)) * nb_h + own.blocks.first) * kTile);
        // down: a column tile and a part of K
        const Share d_part = share_of(F / 32, kParts, part), d_own = share_of(d_part.count, kWorkers, wave);
        const uint32_t d_first = uniform(min(d_part.first + d_own.first, F / 32 - 1)), d_at = uniform((tile * (F / 32) + d_first) * kTile);

        // Requests: a tile here and a tile there.  A wave's three to six at once, all waves at the same time, are 50 to 90 KB a
        // workgroup, which one XCD takes 1.1 to 2 us to fetch (1.3 TB/s); in front of a phase's products that is what the products
        // wait for, behind them what the last wave's store and poll do.
        Tile tq[kOwn], to[kOwnO], tg[kOwn], tu[kOwn], td[kOwnDown];
        Rows rows;
        HeadNorm gamma;
        auto ask_q = [&](const DLayer& from, int i) { ask_tile(tq[i], from.tiles[qm] + q_at, i, own.blocks.count, lane); };
        auto ask_o = [&](const DLayer& from, int i) { ask_tile(to[i], from.tiles[3] + o_at, i, 2, lane); };
        auto ask_gate = [&](const DLayer& from, int i) { ask_tile(tg[i], from.tiles[4] + g_at, i, own.blocks.count, lane); };
        auto ask_up = [&](const DLayer& from, int i) { ask_tile(tu[i], from.tiles[5] + g_at, i, own.blocks.count, lane); };
        auto ask_down = [&](const DLayer& from, int i) { ask_tile(td[i], from.tiles[6] + d_at, i, d_own.count, lane); };
        {
            const DLayer& L = a.layer[0];
#pragma unroll
            for (int i = 0; i < kOwn; ++i) ask_q(L, i);
            for (int i = 0; i < kOwnO; ++i) ask_o(L, i);
            for (int i = 0; i < kOwn; ++i) ask_gate(L, i);
            for (int i = 0; i < 1; ++i) ask_up(L, i);
            const Tokens t = tokens_of(sh, 0, L.ring_mask, slot);
            ask_rows(rows, L.ring_k, L.ring_v, t, wave, lane);
            gamma = ask_gamma(L);
        }
        // the operand that the launch starts from
        put_quad(*reinterpret_cast<const f4_t*>(a.u_in + size_t(row) * H + own.at), lane, own.on, sh.opnd[wave], sh.mult[wave]);
        own_lds();
        auto publish = [&](float acc, int matrix) { sh.red[wave][matrix][lane] = acc; };
        for (uint32_t l = 0; l < a.layers; ++l) {
            const DLayer& L = a.layer[l];
            const uint32_t ln = l + 1 < a.layers ? l + 1 : l;   // past the last block: this one's again, unused
            const DLayer& N = a.layer[ln];
            enter();
            // ---- q, k, v -----------------------------------------------------------------------------------
            {
                int op[2];
                i4_t D[kOwn];
                read_operand(op, sh.opnd[wave], lane);
                if (l != 0) {
                    ask_gate(L, 2);
                    ask_up(L, 0);
                }
                steps(tq, op, D);
                publish(fold(tq, own.blocks.count, D, sh.mult[wave]), 0);
            }
            put_rows(sh, rows, wave, lane);
            meet();
            const Tokens t = tokens_of(sh, l, L.ring_mask, slot);
            if (l == 0) meet();
            // ---- attention ---------------------------------------------------------------------------------
            attend<false>(l, L, t, gamma, [&] { ask_q(N, 0); ask_q(N, 1); ask_q(N, 2); }, [&] { ask_up(L, 1); ask_up(L, 2); });
            meet();
            // ---- merge of the partitions for this wave's 64 elements, o-projection ------------------------
            if (merges) {
                // 16 lanes hold the 64 elements, four each; lane group g the partitions 4 i + g
                const uint32_t head = (64 * o_pair) / kHd, dim = (64 * o_pair) % kHd, g = lane >> 4, s16 = lane & 15u;
                f4_t pv[kGroups / 4];
                float2 ml;
                // looked at until they are there, those that are missing only: all of them are 49 KB a workgroup
                uint32_t missing = (2u << (kGroups / 4)) - 1, looks = 0;
                do {
                    if (missing >> (kGroups / 4)) ml = ld2(set_of(l) + a.ml_at, (lane & 31u) * kMl + head * 2);
#pragma unroll
                    for (uint32_t i = 0; i < kGroups / 4; ++i)
                        if (missing >> i & 1u) pv[i] = ld4(set_of(l) + a.out_at + (4 * i * G * kHd + head * kHd + dim) * 4, g * (G * kHd) + 4 * s16);
                    uint32_t left = empty(ml) ? 1u << (kGroups / 4) : 0u;
#pragma unroll
                    for (uint32_t i = 0; i < kGroups / 4; ++i)
                        if (empty(pv[i])) left |= 1u << i;
                    missing = left;
                } while (missing && again(looks));
                float top = ml.y > 0.f ? ml.x : -INFINITY;
                top = swap16_max(row16_max(top));
                const float w = ml.y > 0.f ? expf(ml.x - top) : 0.f;
                const float den = swap16_sum(row16_sum(w * ml.y));
                if (lane < kGroups) sh.weight[wave][8 * (lane & 3u) + (lane >> 2)] = w;
                own_lds();
                const f4_t w0 = *reinterpret_cast<const f4_t*>(&sh.weight[wave][8 * g]), w1 = *reinterpret_cast<const f4_t*>(&sh.weight[wave][8 * g + 4]);
                f4_t e = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (uint32_t i = 0; i < kGroups / 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) e[j] = fmaf(i < 4 ? w0[i & 3] : w1[i & 3], pv[i][j], e[j]);
                // element 4 s16 + g is left in this lane
                const u2_t ex = __builtin_amdgcn_permlane32_swap(__float_as_uint(e.x), __float_as_uint(e.z), false, false);
                const u2_t ey = __builtin_amdgcn_permlane32_swap(__float_as_uint(e.y), __float_as_uint(e.w), false, false);
                const u2_t ez = __builtin_amdgcn_permlane16_swap(__float_as_uint(__uint_as_float(ex.x) + __uint_as_float(ex.y)),
                                                                 __float_as_uint(__uint_as_float(ey.x) + __uint_as_float(ey.y)), false, false);
                const float v = (__uint_as_float(ez.x) + __uint_as_float(ez.y)) / den;
                uint32_t m = magnitude(v);
                m = max(m, lane_cross_u32<0xB1, 0xF>(m));
                m = max(m, lane_cross_u32<0x4E, 0xF>(m));
                m = max(m, lane_cross_u32<0x141, 0xF>(m));
                const u2_t m16 = __builtin_amdgcn_permlane16_swap(m, m, false, false);
                m = max(m16.x, m16.y);
                const u2_t m32 = __builtin_amdgcn_permlane32_swap(m, m, false, false);
                const GroupScale scale = group_scale(max(m32.x, m32.y));
                sh.opnd[wave][4 * s16 + g] = digits(v, scale.scale);
                if ((lane & 0x37u) == 0) sh.mult[wave][s16 >> 3] = scale.mult;
                own_lds();
                int op[1];
                i4_t D[kOwnO];
                read_operand(op, sh.opnd[wave], lane);
                ask_down(L, 0);
                ask_down(L, 1);
                ask_down(L, 2);
                steps(to, op, D);
                publish(fold(to, 2u, D, sh.mult[wave]), 0);
                if (!isfinite(v)) atomicOr(a.status, GUFFIN_STATUS_NONFINITE);
            } else {
                publish(0.f, 0);
                ask_down(L, 0);
                ask_down(L, 1);
                ask_down(L, 2);
            }
            meet();
            // ---- x1 = x + rms(o, post_attention_norm), u = rms(x1, ffn_norm) by the last wave; gate and up ------------
            meet();
            {
                put_quad(*reinterpret_cast<const f4_t*>(sh.u + own.at), lane, own.on, sh.opnd[wave], sh.mult[wave]);
                own_lds();
                int op[2];
                i4_t D[kOwn], E[kOwn];
                read_operand(op, sh.opnd[wave], lane);
                ask_down(L, 3);
                ask_o(N, 0);
                ask_o(N, 1);
                steps(tg, op, D);
                steps(tu, op, E);
                publish(fold(tg, own.blocks.count, D, sh.mult[wave]), 0);
                publish(fold(tu, own.blocks.count, E, sh.mult[wave]), 1);
            }
            meet();
            // ---- down --------------------------------------------------------------------------------------
            {
                const uint32_t at = 32 * d_first + 4 * min(lane, 8 * max(d_own.count, 1u) - 1);
                f4_t hv;
                uint32_t looks = 0;
                do hv = ld4(set_of(l) + a.h_at, at); while (empty(hv) && again(looks));
                put_quad(hv, lane, lane < 8 * d_own.count, sh.opnd[wave], sh.mult[wave]);
                own_lds();
                int op[2];
                i4_t D[kOwnDown];
                read_operand(op, sh.opnd[wave], lane);
                ask_gate(N, 0);
                ask_gate(N, 1);
                steps(td, op, D);
                publish(fold(td, d_own.count, D, sh.mult[wave]), 2);
            }
            const Tokens tn = tokens_of(sh, ln, N.ring_mask, slot);
            ask_rows(rows, N.ring_k, N.ring_v, tn, wave, lane);
            gamma = ask_gamma(N);
            meet();
            // ---- x = x1 + rms(down, post_ffw_norm), u = rms(x, next block's attn_norm or the output norm) by the last wave ---
            meet();
            put_quad(*reinterpret_cast<const f4_t*>(sh.u + own.at), lane, own.on, sh.opnd[wave], sh.mult[wave]);
            own_lds();
        }
    }
};

template <int G>
__global__ void __launch_bounds__(kThreads) drafter_blocks_kernel(const DArgs a) {
    __shared__ __attribute__((aligned(256))) Shared sh;
    const uint32_t row = uniform(xcc_id());   // the model has one KV head: a row an XCD
    if (row >= a.rows) return;
    const uint32_t lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
    Pass<G> pass {a, sh, lane, wave, blockIdx.x / 8, row, 1.0f / static_cast<float>(a.H),
                  __builtin_amdgcn_make_buffer_rsrc(a.exchange + size_t(row) * a.exchange_bytes, 0, static_cast<int>(a.exchange_bytes), 0x00020000)};
    // The arguments' lines, once, all at a time: they come from far, and a block's pointers otherwise cost a wait at each first use.
    {
        uint64_t seen = 0;
        const uint64_t* words = reinterpret_cast<const uint64_t*>(&a);
#pragma unroll
        for (uint32_t i = 0; i < sizeof(DArgs) / 64; ++i) seen ^= words[8 * i];
        asm volatile("" ::"s"(seen));
    }
    // the rotations and the schedules
    if (threadIdx.x == 0) sh.dead = 0;
    for (uint32_t i = threadIdx.x; i < 2 * (kHd / 2); i += kThreads)
        (&sh.rope[0][0])[i] = (i < kHd / 2 ? a.rope_local : a.rope_global)[row * (kHd / 2) + i % (kHd / 2)];
    for (uint32_t i = threadIdx.x; i < 4 * a.layers; i += kThreads) sh.schedule[i / 4][i % 4] = a.schedule[4 * (i / 4 * a.rows + row) + i % 4];
    __syncthreads();
    if (wave == kWorkers) pass.publisher();
    else pass.worker();
}

}  // namespace

// Widths whose tiles a workgroup's waves hold: three blocks of the hidden width a worker, a gate / up pair a workgroup.  Heads are
// normalised here always: a model without head norms (null gammas) is the general resident pass's.
bool drafter_pass_fits(const guffin_model_desc& m) {
    if (m.kv_heads != 1 || m.head_dim != kHd || (m.q_heads != 1 && m.q_heads != 2 && m.q_heads != 4)) return false;
    if (uint64_t(std::max(m.ring_local, m.ring_global)) * 2 * kHd >= (uint64_t(1) << 31)) return false;   // 32-bit offsets into a ring
    if (m.hidden % 64 || m.hidden > kMaxWidth || m.ffn % 64 || m.ffn > kMaxFfn) return false;
    for (uint32_t l = 0; l < m.layer_count; ++l) {
        if (!m.layers[l].norm[1] || !m.layers[l].norm[2]) return false;
        for (int i = 0; i < 7; ++i)
            if (m.layers[l].dtype[i] != GUFFIN_Q8_0) return false;
    }
    return true;
}

// where the regions of a row's exchange buffers start; they start on cache lines of their own
static uint32_t lay_out(const guffin_model_desc& m, DArgs& a) {
    uint32_t used = 0;
    auto take = [&](uint32_t floats) {
        const uint32_t at = used;
        used += (floats * 4 + 255) & ~255u;
        return at;
    };
    a.qkv_at = take((m.q_heads + 2) * kHd);
    a.out_at = take(kGroups * m.q_heads * kHd);
    a.ml_at = take(kGroups * kMl);
    a.o_at = take(kParts * m.hidden);
    a.d_at = take(kParts * m.hidden);
    a.h_at = take(m.ffn);
    a.set_bytes = used;
    used += a.set_bytes;
    a.kv_at = take(std::min(m.layer_count, kLayers) * kHd);   // a key and a value a block, fp16
    return used;
}
uint64_t drafter_pass_bytes(const guffin_model_desc& m, uint32_t rows) {
    DArgs a {};
    return uint64_t(rows) * lay_out(m, a);
}
uint32_t drafter_pass_sync_words(const guffin_model_desc& m) { return (m.layer_count + kLayers - 1) / kLayers * kSyncWords; }

int drafter_pass(hipStream_t stream, const guffin_model_desc& m, uint32_t rows, const DrafterPass& p) {
    if (rows < 1 || rows > kRunRows) return fail(GUFFIN_E_SHAPE, "drafter pass: rows");
    DArgs a {};
    a.rows = rows; a.H = m.hidden; a.F = m.ffn; a.eps = m.eps; a.scale = 1.0f / std::sqrt(static_cast<float>(m.head_dim));
    a.exchange = p.exchange;
    a.exchange_bytes = lay_out(m, a);
    a.rope_local = reinterpret_cast<const float2*>(p.rope_local); a.rope_global = reinterpret_cast<const float2*>(p.rope_global);
    a.status = p.status; a.spin_limit = g_spin_limit;
    for (uint32_t first = 0, n = 0; first < m.layer_count; first += kLayers, ++n) {
        a.layers = std::min(kLayers, m.layer_count - first);
        for (uint32_t i = 0; i < a.layers; ++i) {
            const uint32_t l = first + i;
            const guffin_layer_desc& L = m.layers[l];
            DLayer& d = a.layer[i];
            for (int k = 0; k < 7; ++k) d.tiles[k] = static_cast<const uint8_t*>(L.tiles[k]);
            for (int k = 0; k < 3; ++k) d.weights[k] = L.norm[3 + k];
            d.weights[3] = l + 1 == m.layer_count ? m.out_norm : m.layers[l + 1].norm[0];
            d.weights[4] = L.norm[1]; d.weights[5] = L.norm[2];
            d.ring_k = static_cast<const uint16_t*>(L.ring_k); d.ring_v = static_cast<const uint16_t*>(L.ring_v);
            d.local = layer_is_local(m.global_period, l) ? 1u : 0u;
            d.ring_mask = (d.local ? m.ring_local : m.ring_global) - 1;
        }
        const bool last = first + a.layers == m.layer_count;
        a.sync = p.sync + n * kSyncWords;
        a.schedule = p.schedule + size_t(first) * rows * 4;
        a.priv_k = static_cast<uint16_t*>(p.priv_k) + size_t(first) * rows * kHd;
        a.priv_v = static_cast<uint16_t*>(p.priv_v) + size_t(first) * rows * kHd;
        a.x_in = p.x; a.u_in = p.u; a.x_out = p.x;
        a.u_out = last ? p.out_hidden : p.u;
        a.u_last = last ? p.last_hidden : nullptr;
        a.u_receipt_out = last ? p.out_sums : nullptr;
        a.receipt_rows = p.receipt_rows;
        a.stamps = g_resident_stamps ? g_resident_stamps + size_t(first) * 16 : nullptr;
        switch (m.q_heads) {
            case 1: launch(drafter_blocks_kernel<1>, dim3(kGrid), dim3(kThreads), 0, stream, a); break;
            case 2: launch(drafter_blocks_kernel<2>, dim3(kGrid), dim3(kThreads), 0, stream, a); break;
            case 4: launch(drafter_blocks_kernel<4>, dim3(kGrid), dim3(kThreads), 0, stream, a); break;
            default: return fail(GUFFIN_E_SHAPE, "drafter pass: unsupported head grouping");
        }
        if (int rc = check_launch("drafter_blocks")) return rc;
    }
    return GUFFIN_OK;
}

}  // namespace guffin
