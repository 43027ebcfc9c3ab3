// Prefill GEMM on the matrix core (gfx950): M activation rows times quantised weights.
//
// Replaces the reference's prefill matrix path (src/tensor/backends/metal/metal_kernels.mm:1031-1199, dispatch rules
// metal_command_context.mm:384-401).
//
// Operands.  Weights come as the wave tiles of the decode GEMV (64 columns x one block), activations as the image of
// prefill_image.hpp: fp16 hi and lo halves of x 2^-E.  Both halves of a row meet the same B operand and accumulate in
// the same fp32 accumulator, so one 16x16x32 matrix instruction covers 16 rows.  B is exact: Q4_K sc * q (<= 945) as one
// fused multiply-add of the biased quant, Q8_0 the signed quant, Q6_K s * (q - 32) as the nearest fp16 and the exact
// rest of that rounding (at most one unit of 2049 or more; it meets the hi half only, its product with lo lies below
// the image's own 22 bits).  A block's sums accumulate inside the matrix instruction; its d and the span's
// multiplier are applied in fp32, and Q4_K's -dmin m is one more instruction on the block's group sums.
//
// Precision.  A matrix instruction rounds at the size its accumulator has grown to (some 4.7 times, going by the error), so
// the order of a chain counts: Q4_K takes a group's lo half ahead of its hi half and ends a chain after half a block.  rms
// error against 64 bits in 1e-7 of the result's rms, 333 rows, K = 3840 (Q4_K), 15360 (Q6_K), 2048 (Q8_0): normal activations
// 1.51, 2.16, 1.61; of a 512-fold range 1.57, 2.20, 1.65; every 97th 200-fold 1.63, 2.29, 1.68; all positive 0.87, 2.16, 1.59.
// Those of Q8_0 are three and four row tiles'; up to two add a span up under d alone: 1.06, 1.11, 1.17, 1.05.
// (Kernels of 8 rows, hi and lo in accumulators of their own and Q6_K's -32 a term by itself: 1.56, 3.80, 2.68; 2.24, 4.10,
// 2.74; 3.31, 12.7, 2.88; 0.88, 6.34, 5.21.  Q4_K hi before lo over whole blocks: 1.78, 1.84, 1.87, 0.78, and 4 % faster.  Its
// minima or quants as denormal halves need no bias, but the instruction then drops the places they lack: 1.59 on normal ones.)
//
// A workgroup is four waves on the same R * 16 rows and four neighbouring column tiles.  The A operand of a 64-element
// chunk goes from memory to LDS without passing registers, two chunks ahead in three rotating buffers, one barrier per
// chunk; weights are private to a wave and requested half a block ahead.  A barrier waits for the chunk it opens and leaves everything younger
// on its way, weights too: waits are counts of requests, so requests have a fixed order (in_order()).  Waiting for the weights as well, with the
// first of them asked for behind the first barrier, blocks of 12B shapes took, us, so / as it is: 16 rows 95.9 / 93.4, 37 rows 123.4 / 121.3, 96 rows
// 169.9 / 168.4, 333 rows 428.8 / 424.1; of Q4_K alone 16 rows 88.8 / 86.6, 100 rows 190.4 / 183.0, 192 rows 246.6 / 242.4.
//
// What bounds it: the instructions that form B.  A loop of one matrix and V packed vector instructions (sixteen independent chains of the one, eight
// of the other, two waves a SIMD) takes 8.9, 10.2, 10.6, 12.2 and 13.6 ns of a SIMD for V = 0 to 4, 1.4 more for each further one; a
// block of four row tiles is 272 (Q6_K 384) of the one and 780 (920) of the other, 3.2 (4.3) us by that, and takes 3.7 (4.9) at 2048 rows.  So
// scales are widened for two column groups at once, Q6_K's quants put together as bytes, operands change places instead of being
// copied, and addresses are immediates.  us before / after: 2048 rows gate + up 855 / 839, down (Q6_K) 571 / 552, q/k/v 250 / 243, o 121 /
// 119; 333 rows 180 / 174, 129 / 119, 64.7 / 61.0, 29.1 / 28.4; 37 rows 31.9 / 30.7, 26.9 / 25.1, 14.8 / 13.9, 10.2 / 9.8.
#include "common.hpp"
#include "prefill_image.hpp"
#include "prefill_run.hpp"
#include "receipt.hpp"

#include <algorithm>

namespace guffin {
namespace {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));
typedef uint32_t uint2_t __attribute__((ext_vector_type(2)));

constexpr uint32_t kCols = 64;       // columns per wave tile

__host__ __device__ constexpr uint32_t block_bytes(int dtype) {
    return dtype == GUFFIN_Q8_0 ? 34u : dtype == GUFFIN_Q4_K ? 144u : 210u;
}
__host__ __device__ constexpr uint32_t block_elems(int dtype) { return dtype == GUFFIN_Q8_0 ? 32u : 256u; }

// one thread per 8 elements of a row
__global__ void __launch_bounds__(256)
prefill_pack_kernel(const float* __restrict__ x, uint8_t* __restrict__ blob, uint32_t M, uint32_t K) {
    const ImageLayout L = image_layout(M, K);
    const uint32_t per_row = K / 8;
    const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= uint64_t(M) * per_row) return;   // whole spans leave together: a span is 4 or 32 aligned threads
    const uint32_t row = static_cast<uint32_t>(i / per_row), t = static_cast<uint32_t>(i % per_row);
    const float* src = x + size_t(row) * K + 8 * t;
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = src[k];
    emit_image_values(v, t, row, L, blob);
}

__device__ __forceinline__ half8_t as_half8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(half8_t, make_uint4(a, b, c, d));
}
__device__ __forceinline__ half2_t h2(uint32_t v) { return __builtin_bit_cast(half2_t, v); }
__device__ __forceinline__ uint32_t u2(half2_t v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ half2_t splat(float f) { const _Float16 h = static_cast<_Float16>(f); return half2_t{h, h}; }
// one half for both places: a modifier of the packed instruction that takes it
template <int I>
__device__ __forceinline__ half2_t both(half2_t v) { return __builtin_shufflevector(v, v, I, I); }

// two bytes of w under the bias 1024, which comes off exactly, as a pair of halves; sel: their
// places with 0x04 (the bias byte) in between
__device__ __forceinline__ uint32_t bytes_as_halves(uint32_t w, uint32_t sel, float bias = 1024.f) {
    return u2(h2(__builtin_amdgcn_perm(0x64646464u, w, sel)) - splat(bias));
}

// (w & mask) | c is one instruction if it needs no literal (it takes none) and at most one scalar register: the mask is kept
// in a scalar, c in a vector register.  (Empty asm statements pin them; the instruction itself is the compiler's, whose
// hazard handling around matrix instructions does not look into an asm statement.)
// the bytes of a pair of groups' scale word that belong to the first (second) group, under a bias byte each
constexpr uint32_t pair_bytes(int second) { return second ? 0x04030402u : 0x04010400u; }
__device__ __forceinline__ uint32_t scalar(uint32_t v) { asm("" : "+s"(v)); return v; }
__device__ __forceinline__ uint32_t and_or(uint32_t w, uint32_t mask, uint32_t c) { return (w & mask) | c; }
// a value the compiler takes as it is (it would turn two of the above into two ands and an or3)
__device__ __forceinline__ uint32_t kept(uint32_t v) { asm("" : "+v"(v)); return v; }
__device__ __forceinline__ uint32_t vector_bias(uint32_t c = 0x64006400u) {
    asm("" : "+v"(c));
    return c;
}

// memory is read through buffer resources: an address is the resource and a wave-uniform offset (scalar registers)
// plus the lane's 32-bit offset; reads past the end give zeros
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_resource(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000);
}
__device__ __forceinline__ uint4 ld16(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t uniform_off) {
    const uint4_t v = __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(lane_off), static_cast<int>(uniform_off), 0);
    return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ uint2 ld8(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t uniform_off) {
    const uint2_t v = __builtin_amdgcn_raw_buffer_load_b64(r, static_cast<int>(lane_off), static_cast<int>(uniform_off), 0);
    return make_uint2(v[0], v[1]);
}
__device__ __forceinline__ uint32_t ld4(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t uniform_off) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, static_cast<int>(lane_off), static_cast<int>(uniform_off), 0);
}
// 64 lanes x 16 (4) bytes straight into LDS at `to` (+ 16 (4) per lane)
// (and AT further on both sides: an immediate of the instruction)
template <int AT = 0>
__device__ __forceinline__ void to_lds16(__amdgpu_buffer_rsrc_t r, uint8_t* to, uint32_t lane_off, uint32_t uniform_off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)to, 16, static_cast<int>(lane_off),
                                             static_cast<int>(uniform_off), AT, 0);
}
__device__ __forceinline__ void to_lds4(__amdgpu_buffer_rsrc_t r, uint8_t* to, uint32_t lane_off, uint32_t uniform_off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)to, 4, static_cast<int>(lane_off),
                                             static_cast<int>(uniform_off), 0, 0);
}
// LDS reads of 16 and 8 bytes through the compiler's vector types.  Copied as an object of HIP's, a read carries no type, and
// before such a read the compiler waits for all of the wave's requests into LDS (once or twice a block; with them 128 rows of the
// 12B shapes take 10290 us instead of 9940, 1000 rows 53.5 ms instead of 52.7); for the others the waits stand here.
__device__ __forceinline__ uint4_t from_lds16(const uint8_t* at) { return *reinterpret_cast<const uint4_t*>(at); }
__device__ __forceinline__ uint2_t from_lds8(const uint8_t* at) { return *reinterpret_cast<const uint2_t*>(at); }
// the wave's requests but the N youngest have arrived and its LDS accesses are done, and so have every wave's
template <int N>
__device__ __forceinline__ void arrive() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory"); }

// requests on either side keep their order, which the counts above rely on
__device__ __forceinline__ void in_order() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// What a launch brings.  A kernel takes it as words and pointers in this order: the first fourteen words of a launch's arguments
// are in registers when a wave starts (a build flag), as long as no struct stands among them.
struct GemmArgs {
    const uint8_t* tiles[3];
    const uint8_t* blob;
    uint32_t M, K, columns[3];   // column tiles of 64 of each matrix, 0: no such matrix
    uint32_t form;               // k-slices, and the matrices' formats in the upper bytes
    float* y[3];
};
// the matrix of a workgroup and its first column tile there
struct GemmSegment { const uint8_t* tiles; float* y; uint32_t columns, dtype, first; };
__device__ __forceinline__ GemmSegment segment_of(uint32_t group, const uint8_t* t0, const uint8_t* t1, const uint8_t* t2, uint32_t n0, uint32_t n1,
                                                  uint32_t n2, uint32_t form, float* y0, float* y1, float* y2) {
    const uint32_t g1 = (n0 + 3) / 4, g2 = g1 + (n1 + 3) / 4;
    if (group < g1) return {t0, y0, n0, (form >> 8) & 0xFFu, 4 * group};
    if (group < g2) return {t1, y1, n1, (form >> 16) & 0xFFu, 4 * (group - g1)};
    return {t2, y2, n2, form >> 24, 4 * (group - g2)};
}

// Where a workgroup works: row chunk, column group of 256 over all segments, k-slice (past the last one: nothing to do).
constexpr uint32_t kSliceBits = 5;   // of `form`; above them, up to its matrices' formats: 0, or 1 + log2(row_ways)
struct GemmPlace { uint32_t chunk, group, slice; };
template <int R>
__device__ __forceinline__ GemmPlace place_of(uint32_t M, uint32_t n0, uint32_t n1, uint32_t n2, uint32_t form) {
    const uint32_t cut = (form >> kSliceBits) & 7u;
    if (cut == 0) return {blockIdx.x, blockIdx.y, blockIdx.z};
    const uint32_t chunks = (M + 16 * R - 1) / (16 * R), groups = (n0 + 3) / 4 + (n1 + 3) / 4 + (n2 + 3) / 4;
    const uint32_t lc = cut - 1, ways = 1u << lc, own = (chunks + ways - 1) >> lc;
    const uint32_t x = blockIdx.x & 7u, k = blockIdx.x >> 3, turn = k / own;
    const uint32_t chunk = (x & (ways - 1)) + ways * (k - turn * own), unit = (x >> lc) + (8u >> lc) * turn, slice = unit / groups;
    return {chunk, unit - slice * groups, chunk < chunks ? slice : ~0u};
}

// what the workgroup keeps in LDS, R row tiles of 16
template <int R>
struct Stage {
    static constexpr uint32_t kChunk = 4096 * R;              // 2 groups x R tiles x {hi, lo} x 1 KB; three of them
    static constexpr uint32_t kSums = 3 * kChunk;             // the block's sums image
    static constexpr uint32_t kMult = kSums + 2048;           // and its multipliers
    static constexpr uint32_t kHead = kMult + 256;            // the waves' block headers (scales), two blocks
    static constexpr uint32_t kBytes = kHead + 2 * 4 * 1280;
};

// The chunk's share of one wave: R of its 4R records.
template <int R>
struct Feed {
    __amdgpu_buffer_rsrc_t img;
    uint8_t* stage;
    uint32_t lane16, base, group_stride, wv, last;   // base: this wave's first record of group 0
    __device__ __forceinline__ void ask(uint32_t chunk, uint32_t buffer) const {
        const uint32_t c = chunk < last ? chunk : last;   // past the end: the last chunk again, never read
        const uint32_t from = base + (2 * c + (wv >> 1)) * group_stride;
        uint8_t* to = stage + buffer * Stage<R>::kChunk + (wv >> 1) * (2048 * R) + (wv & 1) * (1024 * R);
        to_lds16<0>(img, to, lane16, from);
        if constexpr (R > 1) to_lds16<1024>(img, to, lane16, from);
        if constexpr (R > 2) to_lds16<2048>(img, to, lane16, from);
        if constexpr (R > 3) to_lds16<3072>(img, to, lane16, from);
    }
};

template <int R>
__device__ __forceinline__ void read_half(const uint8_t* group, uint32_t half, uint32_t lane16, half8_t (&a)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r) a[r] = __builtin_bit_cast(half8_t, from_lds16(group + r * 2048 + half * 1024 + lane16));
}
// the schedule of a region of N matrix instructions: V vector instructions and, at first, an LDS read behind each
template <int N, int V, int D>
__device__ __forceinline__ void weave() {
#pragma unroll
    for (int i = 0; i < N; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (i < D) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, V, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
}

// the lane's number, worked out where it stands
__device__ __forceinline__ uint32_t lane_again() {
    uint32_t none = 0;
    asm volatile("" : "+s"(none));
    return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, none));
}

// ---- Q4_K ------------------------------------------------------------------------------------------------
// The B operands of group G (0..7) of a block for column groups 2P, 2P + 1, from its half block's quants and scale words.
template <int G, int P>
__device__ __forceinline__ void q4_operands(const uint4 (&q)[4], const uint32_t (&scw)[4], half8_t (&b)[4]) {
    constexpr bool HIGH = G & 1;
    constexpr int WORD = (G >> 1) & 1;
    // the quant under a bias whose last place is the quant's: 1024 + q, or 64 + q where the high nibbles stay in bits 4-7
    const uint32_t bias = vector_bias(HIGH ? 0x54005400u : 0x64006400u), mask = scalar(HIGH ? 0x00F000F0u : 0x000F000Fu);
    // both column groups' scales under the bias: 1024 + sc, then sc and -bias sc (all exact in fp16)
    const half2_t sc = h2(__builtin_amdgcn_perm(0x64646464u, scw[2 * P + WORD], pair_bytes(G & 1))) - splat(1024.f);
    const half2_t off = sc * splat(HIGH ? -64.f : -1024.f);
    auto column = [&]<int I>() {
        const uint4 v = q[2 * P + I];
        const uint32_t w0 = WORD ? v.z : v.x, w1 = WORD ? v.w : v.y;
        auto piece = [&](uint32_t w) { return u2(__builtin_elementwise_fma(h2(and_or(w, mask, bias)), both<I>(sc), both<I>(off))); };
        b[2 * P + I] = as_half8(piece(w0), piece(w0 >> 8), piece(w1), piece(w1 >> 8));
    };
    column.template operator()<0>();
    column.template operator()<1>();
}

template <int R, bool FIRST, int C0 = 0, int C1 = 4>
__device__ __forceinline__ void products(const half8_t (&a)[R], const half8_t (&b)[4], float4_t (&D)[4][R]) {
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int cg = C0; cg < C1; ++cg)
#pragma unroll
        for (int r = 0; r < R; ++r) D[cg][r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[r], b[cg], FIRST ? zero : D[cg][r], 0, 0, 0);
}

// A group is two regions of 4R matrix instructions, the hi and the lo halves of A against the same B.  While they run, the
// next region's A operands come from LDS and the next group's B operands are formed, so a wave by itself keeps the matrix
// pipe and the vector pipe busy together.  A chunk's last lo half is in registers when its last region starts: there the
// workgroup meets, the next chunk has arrived and the one after the next but one is asked for in place of the old.
template <int R>
__device__ __forceinline__ void q4_walk(const ImageLayout& L, Feed<R> feed, uint8_t* stage, const uint8_t* tile_base,
                                        uint32_t rt0, uint32_t b0, uint32_t b1, float (&acc)[4][R][4]) {
    constexpr uint32_t TB = kCols * block_bytes(GUFFIN_Q4_K);
    constexpr int kHalf = 4;                        // requests of a half block's quants
    constexpr int V = (26 + 4 * R - 1) / (4 * R);   // vector instructions behind each matrix instruction
    // Up to three row tiles the fold is woven in as well: a tile's beside the next tile's products, the last one's beside the
    // second half's first products.  Four leave no registers for that (2048 x 3840 x 15360: 446 us against 440 by itself).
    constexpr bool WOVEN = R < 4;
    constexpr int VA = (26 + 32 * (R - 1) + 4 * R - 1) / (4 * R), VB = (58 + 4 * R - 1) / (4 * R);
    using S = Stage<R>;
    const uint32_t wv = feed.wv;
    uint32_t lane = lane_again(), j = lane & 15, lg = lane >> 4, lane16 = lane * 16;
    const __amdgpu_buffer_rsrc_t tile = make_resource(tile_base, b1 * TB);
    uint8_t* const heads = stage + S::kHead + wv * 1280;
    uint4 q[2][4];
    uint32_t sc[4];
    half8_t hi[R], lo[R], operands[2][4];   // B of a group and of the next, by turns
    float4_t D[4][R];
    auto ask_half = [&](uint32_t blk, int h, uint4 (&to)[4]) {
#pragma unroll
        for (int cg = 0; cg < 4; ++cg) to[cg] = ld16(tile, lane16, blk * TB + 2048 * cg + 1024 * h);
    };
    auto ask_head = [&](uint32_t blk) { to_lds16(tile, heads + (blk & 1) * 5120, lane16, blk * TB + 8192); };
    // the block's small operands: two waves bring the sums image, one the multipliers
    auto ask_block = [&](uint32_t blk) {
        if (wv < 2) to_lds16(feed.img, stage + S::kSums + 1024 * wv, lane16, static_cast<uint32_t>(L.sums_off) + (blk * (L.mpad / 16) + rt0) * 512 + 1024 * wv);
        else if (wv == 2) to_lds4(feed.img, stage + S::kMult, lane * 4, static_cast<uint32_t>(L.mult_off) + (blk * L.mpad + rt0 * 16) * 4);
    };
    // a word holds the scales of two column groups for two groups of the half: [column pair][groups 0, 1 | 2, 3]
    auto scales = [&](uint32_t blk, int half) {
        uint32_t four[4];   // a column's four groups
#pragma unroll
        for (int cg = 0; cg < 4; ++cg) {
            const uint32_t* h = reinterpret_cast<const uint32_t*>(heads + (blk & 1) * 5120 + 256 * cg + j * 16);
            four[cg] = half ? (h[3] & 0x0F0F0F0Fu) | ((h[1] >> 2) & 0x30303030u) : h[1] & 0x3F3F3F3Fu;
        }
#pragma unroll
        for (int p = 0; p < 4; p += 2) {
            sc[p] = __builtin_amdgcn_perm(four[p + 1], four[p], 0x05010400u);
            sc[p + 1] = __builtin_amdgcn_perm(four[p + 1], four[p], 0x07030602u);
        }
    };
    ask_half(b0, 0, q[0]);
    ask_head(b0);
    feed.ask(4 * b0, 0);
    in_order();
    feed.ask(4 * b0 + 1, 1);
    in_order();
    ask_half(b0, 1, q[1]);
    in_order();
    feed.ask(4 * b0 + 2, 2);
    arrive<2 * R + kHalf>();
    scales(b0, 0);
    read_half<R>(stage, 1, lane16, lo);
    q4_operands<0, 0>(q[0], sc, operands[0]);
    q4_operands<0, 1>(q[0], sc, operands[0]);
    uint32_t rd = 0;   // the buffer of the chunk in work
    uint32_t blk = b0;   // (no test ahead of the first block: behind one, the first weights would be asked for after the first meeting)
    do {
        if constexpr (!WOVEN) { lane = lane_again(); j = lane & 15; lg = lane >> 4; lane16 = feed.lane16 = lane * 16; }   // no register to keep addresses in
        const uint32_t next = blk + 1 < b1 ? blk + 1 : blk;   // the last block asks for itself again
        float dh[4];   // the first half's sums leave their chain for acc (no bias term yet)
        auto fold_scales = [&] {
#pragma unroll
            for (int cg = 0; cg < 4; ++cg)
                dh[cg] = h2f(*reinterpret_cast<const uint16_t*>(heads + (blk & 1) * 5120 + 256 * cg + j * 16));
        };
        auto fold = [&](int r) {
            const float4_t mult = *reinterpret_cast<const float4_t*>(stage + S::kMult + 64 * r + 16 * lg);
#pragma unroll
            for (int cg = 0; cg < 4; ++cg)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[cg][r][i] = fmaf(dh[cg] * mult[i], D[cg][r][i], acc[cg][r][i]);
        };
        auto group = [&]<int G>() {
            half8_t (&b)[4] = operands[G & 1], (&bn)[4] = operands[(G + 1) & 1];
            const uint8_t* now = stage + rd * S::kChunk + (G & 1) * (2048 * R);
            if constexpr (G == 3) ask_half(next, 0, q[0]);   // the half's last operands were formed beside the group before
            if constexpr (G == 7) ask_half(next, 1, q[1]);
            if constexpr ((G & 3) == 3) in_order();
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (G == 3) scales(blk, 1);
            if constexpr (WOVEN && G == 3) fold_scales();
            if constexpr (G == 7) scales(next, 0);
            read_half<R>(now, 0, lane16, hi);
            q4_operands<(G + 1) & 7, 0>(q[G == 7 ? 0 : (G + 1) >> 2], sc, bn);
            if constexpr (WOVEN && G == 4) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    if (r + 1 == R) fold(r);
#pragma unroll
                    for (int cg = 0; cg < 4; ++cg) D[cg][r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[r], b[cg], float4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                }
                weave<4 * R, VB, R>();
            } else {
                products<R, (G & 3) == 0>(lo, b, D);
                weave<4 * R, V, R>();
            }
            if constexpr (G & 1) {
                // What may still be on its way: the chunk asked for at the last meeting and half a block of weights, asked for a group
                // before this meeting (3, 7) or the last one (1, 5); at 3 the next header as well (the fold wants the multipliers).
                arrive<R + kHalf + (G == 3 ? 1 : 0)>();
                if constexpr (G == 1) { ask_block(blk); in_order(); }
                feed.ask(4 * blk + (G >> 1) + 3, rd);
                if constexpr (G == 1) { in_order(); ask_head(next); }
                rd = rd == 2 ? 0 : rd + 1;
            }
            const uint8_t* then = stage + rd * S::kChunk + ((G + 1) & 1) * (2048 * R);
            __builtin_amdgcn_sched_barrier(0);
            read_half<R>(then, 1, lane16, lo);
            q4_operands<(G + 1) & 7, 1>(q[G == 7 ? 0 : (G + 1) >> 2], sc, bn);
            if constexpr (WOVEN && G == 3) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
#pragma unroll
                    for (int cg = 0; cg < 4; ++cg) D[cg][r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[r], b[cg], D[cg][r], 0, 0, 0);
                    if (r > 0) fold(r - 1);
                }
                weave<4 * R, VA, R>();
            } else {
                products<R, false>(hi, b, D);
                weave<4 * R, V, R>();
            }
        };
        group.template operator()<0>();
        group.template operator()<1>();
        group.template operator()<2>();
        group.template operator()<3>();
        if constexpr (!WOVEN) {
            fold_scales();
#pragma unroll
            for (int r = 0; r < R; ++r) fold(r);
        }
        group.template operator()<4>();
        group.template operator()<5>();
        group.template operator()<6>();
        group.template operator()<7>();
        // block done: -dmin sum_g m_g (sum of group g) as one more instruction per tile, then one scale step
        half8_t bm[4];
        float d[4], dmin[4];
#pragma unroll
        for (int cg = 0; cg < 4; ++cg) {
            const uint4_t h = from_lds16(heads + (blk & 1) * 5120 + 256 * cg + j * 16);
            d[cg] = h2f(h.x & 0xFFFFu);
            dmin[cg] = -16.0f * h2f(h.x >> 16);   // the group sums are in units of 32, and twice in dm
            // minima against the sums' hi (k-slices 0 and 2) and lo (1 and 3) halves
            const uint32_t mn_a = h.z & 0x3F3F3F3Fu, mn_b = ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u);
            bm[cg] = as_half8(bytes_as_halves(mn_a, 0x04020400u), bytes_as_halves(mn_a, 0x04030401u),
                              bytes_as_halves(mn_b, 0x04020400u), bytes_as_halves(mn_b, 0x04030401u));
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const half8_t as = __builtin_bit_cast(half8_t, from_lds16(stage + S::kSums + 512 * r + (lane & 31) * 16));
            const float4_t mult = *reinterpret_cast<const float4_t*>(stage + S::kMult + 64 * r + 16 * lg);
#pragma unroll
            for (int cg = 0; cg < 4; ++cg) {
                const float4_t dm = __builtin_amdgcn_mfma_f32_16x16x32_f16(as, bm[cg], float4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[cg][r][i] = fmaf(mult[i], fmaf(dmin[cg], dm[i], d[cg] * D[cg][r][i]), acc[cg][r][i]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    } while (++blk < b1);
}

// ---- Q6_K ------------------------------------------------------------------------------------------------
// Group QD (0..3) of a half block: the quants q - 32 of column groups C0 .. C1 - 1 as halves.  Put together as bytes, four at
// a time, and widened under the bias: 14.5 instructions for a column group's eight quants instead of 18.5 on pairs of halves.
template <int QD, int C0 = 0, int C1 = 4>
__device__ __forceinline__ void q6_quants(const uint4 (&ql)[4], const uint2 (&qh)[4], half8_t (&q)[4]) {
    const uint32_t low = scalar(0x0F0F0F0Fu), high = scalar(0x30303030u);
#pragma unroll
    for (int cg = C0; cg < C1; ++cg) {
        const uint32_t w[2] = {(QD & 1) ? ql[cg].z : ql[cg].x, (QD & 1) ? ql[cg].w : ql[cg].y};
        const uint32_t h[2] = {qh[cg].x, qh[cg].y};
        uint32_t o[4];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            constexpr int up = 4 - 2 * QD;   // the two high bits go to bits 4-5
            const uint32_t wk = QD >= 2 ? w[k] >> 4 : w[k];
            const uint32_t hk = up >= 0 ? h[k] << (up >= 0 ? up : 0) : h[k] >> (up < 0 ? -up : 0);
            const uint32_t bytes = and_or(wk, low, kept(hk & high));
            o[2 * k] = bytes_as_halves(bytes, 0x04020400u, 1056.f);
            o[2 * k + 1] = bytes_as_halves(bytes, 0x04030401u, 1056.f);
        }
        q[cg] = as_half8(o[0], o[1], o[2], o[3]);
    }
}
// both column groups' scales of the pair P (a scale covers 16 elements; a word holds those of two column groups for two groups, int8 + 128)
template <int QD, int P>
__device__ __forceinline__ half2_t q6_scales(const uint32_t (&scw)[4]) {
    return h2(__builtin_amdgcn_perm(0x64646464u, scw[2 * P + (QD >> 1)], pair_bytes(QD & 1))) - splat(1152.f);
}
// times the lane's scale: q becomes the nearest half of the product, rest what that rounding left
__device__ __forceinline__ void q6_times(half2_t s, half8_t& q, half8_t& rest) {
    const uint4 v = __builtin_bit_cast(uint4, q);
    const uint32_t x[4] = {v.x, v.y, v.z, v.w};
    uint32_t p[4], r[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const half2_t prod = s * h2(x[k]);
        p[k] = u2(prod);
        r[k] = u2(__builtin_elementwise_fma(s, h2(x[k]), -prod));
    }
    q = as_half8(p[0], p[1], p[2], p[3]);
    rest = as_half8(r[0], r[1], r[2], r[3]);
}
template <int QD>
__device__ __forceinline__ void q6_scaled(const uint32_t (&scw)[4], half8_t (&q)[4], half8_t (&rest)[4]) {
    auto two = [&]<int P>() {
        const half2_t pair = q6_scales<QD, P>(scw);
        q6_times(both<0>(pair), q[2 * P], rest[2 * P]);
        q6_times(both<1>(pair), q[2 * P + 1], rest[2 * P + 1]);
    };
    two.template operator()<0>();
    two.template operator()<1>();
}
// a half block's scale words from the waves' headers: lanes of k-slices 0, 1 take a group's first scale, of 2, 3 its second
__device__ __forceinline__ void q6_scale_words(const uint8_t* head, int half, uint32_t j, uint32_t sel, uint32_t (&sc)[4]) {
#pragma unroll
    for (int p = 0; p < 4; p += 2) {
        const uint2_t a = from_lds8(head + 256 * p + j * 16 + 8 * half), b = from_lds8(head + 256 * p + 256 + j * 16 + 8 * half);
        sc[p] = __builtin_amdgcn_perm(b.x, a.x, sel) ^ 0x80808080u;   // int8 -> + 128
        sc[p + 1] = __builtin_amdgcn_perm(b.y, a.y, sel) ^ 0x80808080u;
    }
}

// Three regions per group: hi against the rest, hi and lo against the products; while they run, the next group's operands
// are formed (its quants beside the first region, its products and rests beside the second, in place of the rests that are
// done) and the halves of A that the next region wants are read.  Otherwise as the Q4_K walk.
template <int R>
__device__ __forceinline__ void q6_walk(const ImageLayout& L, const Feed<R>& feed, uint8_t* stage, const uint8_t* tile_base,
                                        uint32_t rt0, uint32_t b0, uint32_t b1, float (&acc)[4][R][4]) {
    constexpr uint32_t TB = kCols * block_bytes(GUFFIN_Q6_K);
    constexpr int kHalf = 8;   // requests of a half block's quants
    constexpr int V0 = (60 + 4 * R - 1) / (4 * R), V1 = (38 + 4 * R - 1) / (4 * R);
    using S = Stage<R>;
    const uint32_t lane = threadIdx.x & 63, wv = feed.wv, j = lane & 15, lg = lane >> 4, lane16 = lane * 16;
    const __amdgpu_buffer_rsrc_t tile = make_resource(tile_base, b1 * TB);
    const uint32_t sel = lane >= 32 ? 0x07030501u : 0x06020400u;
    uint8_t* const heads = stage + S::kHead + wv * 1280;
    uint4 ql[2][4];
    uint2 qh[2][4];
    uint32_t sc[4];
    half8_t hi[R], lo[R], operands[2][4], rest[4];
    float4_t D[4][R];
    auto ask_half = [&](uint32_t blk, int h) {
#pragma unroll
        for (int cg = 0; cg < 4; ++cg) {
            ql[h][cg] = ld16(tile, lane16 + 2048 * (cg & 1) + 1024 * h, blk * TB + 4096 * (cg >> 1));
            qh[h][cg] = ld8(tile, lane16 + 8 * h + 1024 * (cg & 3), blk * TB + 8192);
        }
    };
    auto ask_head = [&](uint32_t blk) {   // the 16 scales of every column, then the columns' d (read beyond the tile: zeros)
        to_lds16(tile, heads + (blk & 1) * 5120, lane16, blk * TB + 12288);
        to_lds4(tile, heads + (blk & 1) * 5120 + 1024, lane < 32 ? lane * 4 : 0, blk * TB + 13312);
    };
    auto scales = [&](uint32_t blk, int half) { q6_scale_words(heads + (blk & 1) * 5120, half, j, sel, sc); };
    ask_half(b0, 0);
    ask_head(b0);
    feed.ask(4 * b0, 0);
    in_order();
    feed.ask(4 * b0 + 1, 1);
    in_order();
    ask_half(b0, 1);
    in_order();
    feed.ask(4 * b0 + 2, 2);
    arrive<2 * R + kHalf>();
    scales(b0, 0);
    read_half<R>(stage, 0, lane16, hi);
    q6_quants<0>(ql[0], qh[0], operands[0]);
    q6_scaled<0>(sc, operands[0], rest);
    uint32_t rd = 0, blk = b0;
    do {
        const uint32_t next = blk + 1 < b1 ? blk + 1 : blk;   // the last block asks for itself again
        auto group = [&]<int G>() {
            constexpr int H = ((G + 1) & 7) >> 2, QD = (G + 1) & 3;   // the next group's half block and place
            half8_t (&b)[4] = operands[G & 1], (&bn)[4] = operands[(G + 1) & 1];
            const uint8_t* now = stage + rd * S::kChunk + (G & 1) * (2048 * R);
            if constexpr (G == 3) ask_half(next, 0);
            if constexpr (G == 7) ask_half(next, 1);
            if constexpr ((G & 3) == 3) in_order();
            __builtin_amdgcn_sched_barrier(0);
            read_half<R>(now, 1, lane16, lo);
            q6_quants<QD>(ql[H], qh[H], bn);
            products<R, G == 0>(hi, rest, D);
            weave<4 * R, V0, R>();
            if constexpr (G == 3) scales(blk, 1);
            if constexpr (G == 7) scales(next, 0);
            q6_scaled<QD>(sc, bn, rest);
            products<R, false>(hi, b, D);
            weave<4 * R, V1, 0>();
            if constexpr (G & 1) {
                arrive<R + kHalf + (G == 3 ? 2 : 0)>();   // as the Q4_K walk, a header being two requests
                if constexpr (G == 1) {
                    if (wv == 2) to_lds4(feed.img, stage + S::kMult, lane * 4, static_cast<uint32_t>(L.mult_off) + (blk * L.mpad + rt0 * 16) * 4);
                    in_order();
                }
                feed.ask(4 * blk + (G >> 1) + 3, rd);
                if constexpr (G == 1) { in_order(); ask_head(next); }
                rd = rd == 2 ? 0 : rd + 1;
            }
            __builtin_amdgcn_sched_barrier(0);
            read_half<R>(stage + rd * S::kChunk + ((G + 1) & 1) * (2048 * R), 0, lane16, hi);
            products<R, false>(lo, b, D);
            __builtin_amdgcn_sched_barrier(0);
        };
        group.template operator()<0>();
        group.template operator()<1>();
        group.template operator()<2>();
        group.template operator()<3>();
        group.template operator()<4>();
        group.template operator()<5>();
        group.template operator()<6>();
        group.template operator()<7>();
        float d[4];
#pragma unroll
        for (int cg = 0; cg < 4; ++cg)
            d[cg] = h2f(*reinterpret_cast<const uint16_t*>(heads + (blk & 1) * 5120 + 1024 + 32 * cg + 2 * j));
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float4_t mult = *reinterpret_cast<const float4_t*>(stage + S::kMult + 64 * r + 16 * lg);
#pragma unroll
            for (int cg = 0; cg < 4; ++cg)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[cg][r][i] = fmaf(d[cg] * mult[i], D[cg][r][i], acc[cg][r][i]);
        }
        __builtin_amdgcn_sched_barrier(0);
    } while (++blk < b1);
}

// The same for four row tiles, where the accumulators leave no registers for a whole group's operands formed ahead: a region takes one
// column group, its rest and its products with hi and lo, while the next column group's operands are formed; the compiler's order
// inside a region and the second wave of the SIMD fill the gaps.  2048 x 15360 x 3840, us, two column groups' operands formed ahead of their
// products / so: 521 / 504 (575 / 560 on a part whose clock falls further); 25.8 clocks a matrix instruction at 2.45 vector instructions.
template <int R>
__device__ __forceinline__ void q6_walk_wide(const ImageLayout& L, Feed<R> feed, uint8_t* stage, const uint8_t* tile_base,
                                             uint32_t rt0, uint32_t b0, uint32_t b1, float (&acc)[4][R][4]) {
    constexpr uint32_t TB = kCols * block_bytes(GUFFIN_Q6_K);
    constexpr int kHalf = 8;   // requests of a half block's quants
    using S = Stage<R>;
    const uint32_t wv = feed.wv;
    uint32_t lane = lane_again(), j = lane & 15, lg = lane >> 4, lane16 = lane * 16;
    const __amdgpu_buffer_rsrc_t tile = make_resource(tile_base, b1 * TB);
    uint32_t sel = lane >= 32 ? 0x07030501u : 0x06020400u;
    uint8_t* const heads = stage + S::kHead + wv * 1280;
    uint4 ql[2][4];
    uint2 qh[2][4];
    uint32_t sc[4];
    half8_t hi[R], lo[R], b[4], rest[4];
    float4_t D[4][R];
    auto ask_half = [&](uint32_t blk, int h) {
#pragma unroll
        for (int cg = 0; cg < 4; ++cg) {
            ql[h][cg] = ld16(tile, lane16 + 2048 * (cg & 1) + 1024 * h, blk * TB + 4096 * (cg >> 1));
            qh[h][cg] = ld8(tile, lane16 + 8 * h + 1024 * (cg & 3), blk * TB + 8192);
        }
    };
    auto ask_head = [&](uint32_t blk) {
        to_lds16(tile, heads + (blk & 1) * 5120, lane16, blk * TB + 12288);
        to_lds4(tile, heads + (blk & 1) * 5120 + 1024, lane < 32 ? lane * 4 : 0, blk * TB + 13312);
    };
    auto scales = [&](uint32_t blk, int half) { q6_scale_words(heads + (blk & 1) * 5120, half, j, sel, sc); };
    auto form = [&]<int G, int CG>() {
        q6_quants<G & 3, CG, CG + 1>(ql[(G & 7) >> 2], qh[(G & 7) >> 2], b);
        q6_times(both<CG & 1>(q6_scales<G & 3, (CG >> 1)>(sc)), b[CG], rest[CG]);
    };
    ask_half(b0, 0);
    ask_head(b0);
    feed.ask(4 * b0, 0);
    in_order();
    feed.ask(4 * b0 + 1, 1);
    in_order();
    ask_half(b0, 1);
    in_order();
    feed.ask(4 * b0 + 2, 2);
    arrive<2 * R + kHalf>();
    scales(b0, 0);
    read_half<R>(stage, 0, lane16, hi);
    form.template operator()<0, 0>();
    uint32_t rd = 0, blk = b0;
    do {
        lane = lane_again(); j = lane & 15; lg = lane >> 4; lane16 = feed.lane16 = lane * 16;   // no register to keep addresses in
        sel = lane >= 32 ? 0x07030501u : 0x06020400u;
        const uint32_t next = blk + 1 < b1 ? blk + 1 : blk;   // the last block asks for itself again
        auto group = [&]<int G>() {
            const uint8_t* now = stage + rd * S::kChunk + (G & 1) * (2048 * R);
            auto column = [&]<int CG>() {
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (CG == 0) read_half<R>(now, 1, lane16, lo);
                form.template operator()<G, CG + 1>();
                products<R, G == 0, CG, CG + 1>(hi, rest, D);
                products<R, false, CG, CG + 1>(hi, b, D);
                products<R, false, CG, CG + 1>(lo, b, D);
            };
            column.template operator()<0>();
            column.template operator()<1>();
            column.template operator()<2>();
            if constexpr (G == 3) ask_half(next, 0);   // the half's last operands are formed
            if constexpr (G == 7) ask_half(next, 1);
            if constexpr ((G & 3) == 3) in_order();
            if constexpr (G == 3) scales(blk, 1);
            if constexpr (G == 7) scales(next, 0);
            __builtin_amdgcn_sched_barrier(0);
            form.template operator()<G + 1, 0>();
            products<R, G == 0, 3, 4>(hi, rest, D);
            products<R, false, 3, 4>(hi, b, D);
            if constexpr (G & 1) {
                arrive<R + kHalf + (G == 3 ? 2 : 0)>();   // as the walk above
                if constexpr (G == 1) {
                    if (wv == 2) to_lds4(feed.img, stage + S::kMult, lane * 4, static_cast<uint32_t>(L.mult_off) + (blk * L.mpad + rt0 * 16) * 4);
                    in_order();
                }
                feed.ask(4 * blk + (G >> 1) + 3, rd);
                if constexpr (G == 1) { in_order(); ask_head(next); }
                rd = rd == 2 ? 0 : rd + 1;
            }
            __builtin_amdgcn_sched_barrier(0);
            read_half<R>(stage + rd * S::kChunk + ((G + 1) & 1) * (2048 * R), 0, lane16, hi);
            products<R, false, 3, 4>(lo, b, D);
            __builtin_amdgcn_sched_barrier(0);
        };
        group.template operator()<0>();
        group.template operator()<1>();
        group.template operator()<2>();
        group.template operator()<3>();
        group.template operator()<4>();
        group.template operator()<5>();
        group.template operator()<6>();
        group.template operator()<7>();
        float d[4];
#pragma unroll
        for (int cg = 0; cg < 4; ++cg)
            d[cg] = h2f(*reinterpret_cast<const uint16_t*>(heads + (blk & 1) * 5120 + 1024 + 32 * cg + 2 * j));
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float4_t mult = *reinterpret_cast<const float4_t*>(stage + S::kMult + 64 * r + 16 * lg);
#pragma unroll
            for (int cg = 0; cg < 4; ++cg)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[cg][r][i] = fmaf(d[cg] * mult[i], D[cg][r][i], acc[cg][r][i]);
        }
        __builtin_amdgcn_sched_barrier(0);
    } while (++blk < b1);
}

// grid (row chunks, column groups of 256 over all segments, k-slices), so that an XCD's L2 keeps its share of the image, or as
// row_ways has it; 256 threads a team.
// Two teams take half a slice each on operands of their own and add up through LDS: where a compute unit has one workgroup, a second wave a
// SIMD issues beside the first, and a slice rounds as two while its planes, and the next operator's reads of them, are those of one.  (R = 1, one
// wave a SIMD 5840 clocks a block, two 8170 for both.  One team taking both halves one after the other, and twice the slices where that was
// faster, blocks of 12B shapes, us, so / by teams: 10 rows 92.5 / 89.0, 20 rows 105.2 / 102.6, 96 rows 168.5 / 165.8, 128 rows 199.0 / 196.2; of
// Q4_K alone 37 rows 116.8 / 113.8, 100 rows 183.0 / 174.0.  52 to 64 rows lose a little, 140.3 / 141.4; without halves they take 0.3-1.1 % more
// again.)
template <int R, int KINDS, int TEAMS = 1>
__global__ void __launch_bounds__(256 * TEAMS, 2)
prefill_gemm_kernel(const uint8_t* __restrict__ t0, const uint8_t* __restrict__ t1, const uint8_t* __restrict__ t2, const uint8_t* __restrict__ blob,
                    uint32_t M, uint32_t K, uint32_t n0, uint32_t n1, uint32_t n2, uint32_t form, float* __restrict__ y0,
                    float* __restrict__ y1, float* __restrict__ y2) {
    // (two stages pass what a kernel may declare for itself)
    __shared__ __attribute__((aligned(16))) uint8_t one[TEAMS == 1 ? Stage<R>::kBytes : 16];
    extern __shared__ __attribute__((aligned(16))) uint8_t two[];
    uint8_t* const stages = TEAMS == 1 ? one : two;
    const ImageLayout L = image_layout(M, K);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wv = wave & 3, team = TEAMS == 1 ? 0u : wave >> 2;
    uint8_t* const stage = stages + team * Stage<R>::kBytes;
    const GemmPlace at = place_of<R>(M, n0, n1, n2, form);
    const uint32_t slices = form & ((1u << kSliceBits) - 1);
    if (at.slice >= slices) return;
    const GemmSegment seg = segment_of(at.group, t0, t1, t2, n0, n1, n2, form, y0, y1, y2);
    const uint32_t tile_index = seg.first + wv, nblk = K / 256, rt0 = at.chunk * R;
    const bool valid = tile_index < seg.columns;   // a wave past the last tile works on tile 0 and stores nothing
    const uint32_t part = TEAMS * at.slice + team, parts = TEAMS * slices;
    const uint32_t b0 = part * nblk / parts, b1 = (part + 1) * nblk / parts;
    Feed<R> feed;
    feed.img = make_resource(blob, static_cast<uint32_t>(L.bytes));
    feed.stage = stage;
    feed.lane16 = lane_again() * 16;
    feed.group_stride = (L.mpad / 16) * 2048;
    feed.base = rt0 * 2048 + (wv & 1) * (1024 * R);
    feed.wv = wv;
    feed.last = 4 * b1 - 1;
    // a whole form per format: what they share would have to lie in the same registers for both
    auto run = [&](auto walk, uint32_t bytes) {
        float acc[4][R][4];
#pragma unroll
        for (int cg = 0; cg < 4; ++cg)
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[cg][r][i] = 0.f;
        walk(L, feed, stage, seg.tiles + size_t(valid ? tile_index : 0) * nblk * (kCols * bytes), rt0, b0, b1, acc);
        // the chunks asked for past the end are still on their way into this workgroup's LDS
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const uint32_t N = seg.columns * kCols;
        float* y = seg.y + at.slice * (uint64_t(M) * N);
        const uint32_t lane = lane_again(), col = tile_index * kCols + (lane & 15), row0 = rt0 * 16 + 4 * (lane >> 4);
        auto store = [&]<int C0, int C1>() {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t row = row0 + 16 * r + i;
                    if (row < M)
#pragma unroll
                        for (int cg = C0; cg < C1; ++cg) y[size_t(row) * N + col + 16 * cg] = acc[cg][r][i];
                }
        };
        if constexpr (TEAMS == 1) {
            if (valid) store.template operator()<0, 4>();
        } else {
            // the team with a block less meets as often as the other one
            const uint32_t other = part ^ 1u, others = (other + 1) * nblk / parts - other * nblk / parts;
            for (uint32_t n = 4 * (b1 - b0); n < 4 * others; ++n) asm volatile("s_barrier" ::: "memory");
            arrive<0>();
            // a team's sums of two column groups to the other one, which finishes and stores them
            float4_t* const swap = reinterpret_cast<float4_t*>(stages) + wv * 64 + lane;   // [team][column group][row tile][256]
            auto finish = [&]<int OWN>() {
                constexpr int GIVEN = 2 - OWN;
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const float(&give)[4] = acc[GIVEN + c][r];
                        swap[(GIVEN * R + c * R + r) * 256] = float4_t{give[0], give[1], give[2], give[3]};
                    }
                arrive<0>();
                if (!valid) return;
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const float4_t more = swap[(OWN * R + c * R + r) * 256];
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[OWN + c][r][i] += more[i];
                    }
                store.template operator()<OWN, OWN + 2>();
            };
            if (team == 0) finish.template operator()<0>(); else finish.template operator()<2>();
        }
    };
    if (KINDS == 1 || (KINDS == 3 && seg.dtype == GUFFIN_Q4_K)) run(q4_walk<R>, block_bytes(GUFFIN_Q4_K));
    else if constexpr (KINDS != 1 && R == 4) run(q6_walk_wide<R>, block_bytes(GUFFIN_Q6_K));
    else if constexpr (KINDS != 1) run(q6_walk<R>, block_bytes(GUFFIN_Q6_K));
}

// ---- Q8_0 ------------------------------------------------------------------------------------------------
// The same stages; a 32-element block is one group, so its d and the span's multiplier are applied after the two matrix
// instructions (hi, lo) of a tile: eight vector instructions to one of the matrix unit's, half of them here.  SPAN (spans of 256, up to two row
// tiles): blocks add up under d alone and a span's sum takes the multiplier, a third of the instructions less and no less exact (rms error
// against 64 bits, 1e-7 of the result's, K = 1024 and 2048, a multiplier a block / so: 1.25 / 0.98, 1.61 / 1.06; of a 512-fold range 1.30 / 1.05, 1.65
// / 1.12); three row tiles have no registers for it.  us before / after it and the walk without branches: 2048 rows o 16.8 / 14.9, down 27.4 /
// 25.1, q/k/v 19.5 / 18.7; 1000 rows o 12.0 / 10.8, down 15.7 / 14.9, gate + up 25.2 / 23.9.  Chunks [c0, c1) of two blocks; WAVES share the chunk's records, the waves of a pair (wv, wv + 4) by turns.
template <int R>
constexpr uint32_t kQ8Slot = Stage<R>::kChunk + 512;   // chunk, its two groups' multipliers
template <int R, int WAVES, bool SPAN>
__device__ __forceinline__ void q8_walk(const ImageLayout& L, __amdgpu_buffer_rsrc_t img, __amdgpu_buffer_rsrc_t tile, uint8_t* stage, uint32_t lane,
                                        uint32_t wv, uint32_t rt0, uint32_t nblk, uint32_t c0, uint32_t c1, float (&acc)[4][R][4]) {
    constexpr uint32_t TB = kCols * block_bytes(GUFFIN_Q8_0), kSlot = kQ8Slot<R>;
    constexpr int kOwn = WAVES == 4 ? R : R / 2;   // records that every wave asks for at least
    const uint32_t j = lane & 15, lg = lane >> 4;
    const uint32_t lane16 = lane * 16, group_stride = (L.mpad / 16) * 2048, shift = L.span == 256 ? 3 : 0, quarter = wv & 3;
    const uint32_t base = rt0 * 2048 + (quarter & 1) * (1024 * R), mult_off = static_cast<uint32_t>(L.mult_off) + rt0 * 64;
    auto ask = [&](uint32_t chunk, uint32_t buffer) {
        const uint32_t c = chunk < c1 ? chunk : c1 - 1;
        uint8_t* to = stage + buffer * kSlot;
#pragma unroll
        for (int i = 0; i < R; ++i)
            if (WAVES == 4 || uint32_t(i & 1) == wv >> 2)
                to_lds16(img, to + (quarter >> 1) * (2048 * R) + (quarter & 1) * (1024 * R) + 1024 * i, lane16,
                         base + min(2 * c + (quarter >> 1), nblk - 1) * group_stride + 1024 * i);
        if (wv < 2) to_lds4(img, to + Stage<R>::kChunk + 256 * wv, lane * 4, mult_off + (min(2 * c + wv, nblk - 1) >> shift) * L.mpad * 4);
    };
    uint4 q[2][2][2];       // [buffer][group][piece]
    uint32_t dw[2][2][4];
    auto ask_weights = [&](uint32_t chunk, int to) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t at = min(2 * chunk + h, nblk - 1) * TB;   // past the end: the last block again, never used
            q[to][h][0] = ld16(tile, lane16, at);
            q[to][h][1] = ld16(tile, lane16, at + 1024);
#pragma unroll
            for (int cg = 0; cg < 4; ++cg) dw[to][h][cg] = ld4(tile, (j >> 1) * 4, at + 2048 + 32 * cg);
        }
    };
#pragma unroll
    for (int cg = 0; cg < 4; ++cg)
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[cg][r][i] = 0.f;
    float t[SPAN ? 4 : 1][R][4];
    if constexpr (SPAN) {
#pragma unroll
        for (int cg = 0; cg < 4; ++cg)
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int i = 0; i < 4; ++i) t[cg][r][i] = 0.f;
    }
    ask_weights(c0, 0);
    ask(c0, 0);
    asm volatile("" ::: "memory");   // in this order
    ask(c0 + 1, 1);
    uint32_t rd = 0, wr = 2;
    auto chunk = [&]<bool BOTH>(uint32_t c, int now) {
        arrive<kOwn>();
        ask_weights(c + 1, now ^ 1);
        ask(c + 2, wr);
        const uint8_t* from = stage + rd * kSlot;
#pragma unroll
        for (int h = 0; h < (BOTH || R == 4 ? 2 : 1); ++h) {
            if (R == 4 && 2 * c + h >= nblk) break;
            half8_t hi[R], lo[R];
            read_half<R>(from + h * (2048 * R), 0, lane16, hi);
            read_half<R>(from + h * (2048 * R), 1, lane16, lo);
            half8_t b[4];
            float d[4];
#pragma unroll
            for (int cg = 0; cg < 4; ++cg) {
                const uint4 piece = q[now][h][cg >> 1];
                const uint32_t w0 = ((cg & 1) ? piece.z : piece.x) ^ 0x80808080u, w1 = ((cg & 1) ? piece.w : piece.y) ^ 0x80808080u;
                b[cg] = as_half8(bytes_as_halves(w0, 0x04020400u, 1152.f), bytes_as_halves(w0, 0x04030401u, 1152.f),
                                 bytes_as_halves(w1, 0x04020400u, 1152.f), bytes_as_halves(w1, 0x04030401u, 1152.f));
                d[cg] = h2f((dw[now][h][cg] >> (16 * (j & 1u))) & 0xFFFFu);
            }
            float4_t D[4][R];
            products<R, true>(hi, b, D);
            products<R, false>(lo, b, D);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float4_t mult = *reinterpret_cast<const float4_t*>(from + Stage<R>::kChunk + 256 * h + 64 * r + 16 * lg);
#pragma unroll
                for (int cg = 0; cg < 4; ++cg)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if constexpr (SPAN) t[cg][r][i] = fmaf(d[cg], D[cg][r][i], t[cg][r][i]);
                        else acc[cg][r][i] = fmaf(d[cg] * mult[i], D[cg][r][i], acc[cg][r][i]);
                    }
            }
        }
        if constexpr (SPAN) {
            if (((c + 1) & 3u) == 0 || c + 1 >= c1) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float4_t mult = *reinterpret_cast<const float4_t*>(from + Stage<R>::kChunk + 64 * r + 16 * lg);
#pragma unroll
                    for (int cg = 0; cg < 4; ++cg)
#pragma unroll
                        for (int i = 0; i < 4; ++i) { acc[cg][r][i] = fmaf(mult[i], t[cg][r][i], acc[cg][r][i]); t[cg][r][i] = 0.f; }
                }
            }
        }
        rd = rd == 2 ? 0 : rd + 1;
        wr = wr == 2 ? 0 : wr + 1;
    };
    // A branch around a block has the sums copied from register to register, and keeps its products from the next block's: only four row
    // tiles, which have no registers for two blocks' products, have one.
    const uint32_t both = R == 4 ? c1 : min(c1, nblk / 2);   // an odd number of blocks: the last chunk has one
    uint32_t c = c0;
    if constexpr (R == 4) {
        for (; c < c1; c += 2) {
            chunk.template operator()<true>(c, 0);
            if (c + 1 < c1) chunk.template operator()<true>(c + 1, 1);
        }
    }
    for (; c + 2 <= both; c += 2) {
        chunk.template operator()<true>(c, 0);
        chunk.template operator()<true>(c + 1, 1);
    }
    if (R == 4) {
    } else if (c < both) {
        chunk.template operator()<true>(c, 0);
        if (c + 1 < c1) chunk.template operator()<false>(c + 1, 1);
    } else if (c < c1) {
        chunk.template operator()<false>(c, 0);
    }
    // the chunks asked for past the end are still on their way into this workgroup's LDS
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// grid as prefill_gemm_kernel's, k-slices in chunks of two blocks.
template <int R>
__global__ void __launch_bounds__(256, 2)
prefill_gemm_q8_kernel(const uint8_t* __restrict__ t0, const uint8_t* __restrict__ t1, const uint8_t* __restrict__ t2, const uint8_t* __restrict__ blob,
                    uint32_t M, uint32_t K, uint32_t n0, uint32_t n1, uint32_t n2, uint32_t form, float* __restrict__ y0,
                    float* __restrict__ y1, float* __restrict__ y2) {
    constexpr uint32_t TB = kCols * block_bytes(GUFFIN_Q8_0);
    __shared__ __attribute__((aligned(16))) uint8_t stage[3 * kQ8Slot<R>];
    const ImageLayout L = image_layout(M, K);
    const uint32_t lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 15, lg = lane >> 4;
    const uint32_t slices = form & ((1u << kSliceBits) - 1);
    const GemmSegment seg = segment_of(blockIdx.y, t0, t1, t2, n0, n1, n2, form, y0, y1, y2);
    const uint32_t tile_index = seg.first + wv, nblk = K / 32, rt0 = blockIdx.x * R;
    const bool valid = tile_index < seg.columns;
    const uint32_t chunks = (nblk + 1) / 2, c0 = blockIdx.z * chunks / slices, c1 = (blockIdx.z + 1) * chunks / slices;
    const __amdgpu_buffer_rsrc_t img = make_resource(blob, static_cast<uint32_t>(L.bytes));
    const __amdgpu_buffer_rsrc_t tile = make_resource(seg.tiles + size_t(valid ? tile_index : 0) * nblk * TB, nblk * TB);
    float acc[4][R][4];
    if (R < 3 && L.span == 256) q8_walk<R, 4, (R < 3)>(L, img, tile, stage, lane, wv, rt0, nblk, c0, c1, acc);
    else q8_walk<R, 4, false>(L, img, tile, stage, lane, wv, rt0, nblk, c0, c1, acc);
    if (!valid) return;
    const uint32_t N = seg.columns * kCols;
    float* y = seg.y + blockIdx.z * (uint64_t(M) * N);
    const uint32_t col = tile_index * kCols + j, row0 = rt0 * 16 + 4 * lg;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t row = row0 + 16 * r + i;
            if (row < M)
#pragma unroll
                for (int cg = 0; cg < 4; ++cg) y[size_t(row) * N + col + 16 * cg] = acc[cg][r][i];
        }
}

// Gate, up and GeGLU: the next GEMM's operand straight from the products.  grid (row chunks, F / 256), eight waves: four gate tiles and the four
// up tiles of the same columns, 256 of them -- one span of the operand.  A gate wave takes the first 32 columns of the tile pair over, its
// up wave the others; values go through LDS from a column a lane to eight columns a lane, and the span's largest from wave to wave.
// Bound by its first trips and the twenty vector instructions a column group costs (as above); 1000 rows of the drafter: 20.0 + 7.2 us as
// two launches.
template <int R>
struct GatedStage {
    static constexpr uint32_t kSwap = 8 * R * 2048;                           // half an accumulator of every wave
    static constexpr uint32_t kPitch = 36, kTurn = 8 * 16 * R * kPitch * 4;    // rows of 32 columns of every wave
    static constexpr uint32_t kWalk = 3 * kQ8Slot<R>;
    static constexpr uint32_t kMost = kTurn > kSwap ? (kTurn > kWalk ? kTurn : kWalk) : (kSwap > kWalk ? kSwap : kWalk);
    static constexpr uint32_t kBytes = kMost + 8 * 16 * R * 4;                 // and its rows' largest
};
template <int R>
__global__ void __launch_bounds__(512)
prefill_gateup_q8_kernel(const uint8_t* __restrict__ gate, const uint8_t* __restrict__ up, const uint8_t* __restrict__ blob, uint32_t M, uint32_t K,
                         uint32_t F, uint8_t* __restrict__ out) {
    constexpr uint32_t TB = kCols * block_bytes(GUFFIN_Q8_0);
    using G = GatedStage<R>;
    extern __shared__ __attribute__((aligned(16))) uint8_t stage[];
    const ImageLayout L = image_layout(M, K), O = image_layout(M, F);
    const uint32_t lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 15, lg = lane >> 4;
    const uint32_t pair = wv & 3, nblk = K / 32, rt0 = blockIdx.x * R;
    const bool is_up = wv >= 4;
    const __amdgpu_buffer_rsrc_t img = make_resource(blob, static_cast<uint32_t>(L.bytes));
    const __amdgpu_buffer_rsrc_t tile = make_resource((is_up ? up : gate) + size_t(4 * blockIdx.y + pair) * nblk * TB, nblk * TB);
    float acc[4][R][4];
    q8_walk<R, 8, false>(L, img, tile, stage, lane, wv, rt0, nblk, 0, (nblk + 1) / 2, acc);
    __syncthreads();
    // the other half of the tile pair's products
    float4_t* swap = reinterpret_cast<float4_t*>(stage);
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float(&give)[4] = acc[is_up ? c : 2 + c][r];
            swap[((wv * 2 + c) * R + r) * 64 + lane] = float4_t{give[0], give[1], give[2], give[3]};
        }
    __syncthreads();
    float h[2][R][4];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float4_t other = swap[(((wv ^ 4) * 2 + c) * R + r) * 64 + lane];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float own = is_up ? acc[2 + c][r][i] : acc[c][r][i];
                h[c][r][i] = is_up ? geglu_value(other[i], own) : geglu_value(own, other[i]);
            }
        }
    __syncthreads();
    float* turn = reinterpret_cast<float*>(stage) + wv * (16 * R * G::kPitch);   // this wave's [row][32 columns]
    float* largest = reinterpret_cast<float*>(stage + G::kMost);                 // [wave][row]
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i) turn[(16 * r + 4 * lg + i) * G::kPitch + 16 * c + j] = h[c][r][i];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the wave's own
    // lane (row j, k-slice lg) of a record
    float v[R][8];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float* from = turn + (16 * r + j) * G::kPitch + 8 * lg;
        const float4_t a = *reinterpret_cast<const float4_t*>(from), b = *reinterpret_cast<const float4_t*>(from + 4);
        float m = 0.f;
#pragma unroll
        for (int k = 0; k < 8; ++k) { v[r][k] = k < 4 ? a[k & 3] : b[k & 3]; m = fmaxf(m, fabsf(v[r][k])); }
        m = fmaxf(m, __shfl_xor(m, 16, kWave));
        m = fmaxf(m, __shfl_xor(m, 32, kWave));
        if (lg == 0) largest[wv * (16 * R) + 16 * r + j] = m;
    }
    __syncthreads();
    const uint32_t group = 8 * blockIdx.y + 2 * pair + (is_up ? 1u : 0u);   // of 32 columns
#pragma unroll
    for (int r = 0; r < R; ++r) {
        float m = 0.f;
#pragma unroll
        for (int w = 0; w < 8; ++w) m = fmaxf(m, largest[w * (16 * R) + 16 * r + j]);
        const uint32_t row = 16 * (rt0 + r) + j;
        if (row >= M) continue;
        emit_image_record(v[r], m, group, lg, row, O, out);
        if (wv == 0 && lg == 0) reinterpret_cast<float*>(out + O.mult_off)[size_t(blockIdx.y) * O.mpad + row] = image_multiplier(m);
    }
}

// How many ways the XCDs cut the row chunks of a launch between them, the column groups of all slices (`units`) being dealt over the others;
// 0: the grid's own order.  Consecutive workgroups go to different XCDs, so where the rows run fastest the workgroups that share weights sit in
// different L2s and each fetches them, while an L2 keeps its share of the image; dealt, the workgroups of a unit share an L2 and the
// weights are fetched once (one way) or twice.  The lines are by the number of chunks alone: as many XCDs fetch a weight as there are chunks, up to
// eight.  Passes of the 12B shapes, us, grid's order / one way / two ways: 160 rows 12207 / 11861 / 13439, 333 21035 / 20486 / 20563, 448 25888 /
// 25270 / 24869, 640 34744 / 35441 / 33996, 704 38435 / 40628 / 39683, 2048 100656 / 104727 / 102185.  Single launches of other widths, 288 / 448 /
// 640 / 1024 rows, grid's order / so: K = 2048, N = 16384 Q4_K 49.4 / 46.2, 62.7 / 60.3, 91.2 / 88.6, the same; K = 8192, N = 2048 Q6_K 37.1 / 34.6, 47.2
// / 42.7, the same, the same; K = 5120, N = 27648 182.9 / 173.8, 241.8 / 256.6 (seven chunks by fours leave XCDs uneven), 358.5 / 344.6, the same.
// Not where the uneven shares take an XCD one more turn of two workgroups a compute unit: 288 rows of K = 13824, N = 5120, five chunks, 65
// workgroups instead of 63, 93.9 / 119.2.  The drafter's weights are small beside its image: 333 rows 1302 / 1417 / 1375.
uint32_t row_ways(uint32_t chunks, uint32_t units, bool q8) {
    if (q8 || chunks < 2 || chunks > 10) return 0;
    const uint32_t ways = chunks <= 6 ? 1 : 2, others = 8 / ways, turn = std::max(1u, 2 * compute_units() / 8);
    const uint32_t dealt = (chunks + ways - 1) / ways * ((units + others - 1) / others), even = (chunks * units + 7) / 8;
    return (dealt + turn - 1) / turn > (even + turn - 1) / turn ? 0 : ways;
}

// (columns come by 64, planes lie in arenas of 256 bytes)
__global__ void __launch_bounds__(256) zero_planes_kernel(float* planes, uint64_t quads) {
    const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i < quads) reinterpret_cast<float4_t*>(planes)[i] = float4_t{0.f, 0.f, 0.f, 0.f};
}

int gemm_launch(hipStream_t s, const PrefillMatrix* m, uint32_t count, const uint8_t* image, float* const* y, uint32_t M, uint32_t K,
                uint32_t slices, uint32_t R, bool halves) {
    if (count > 3 || slices >= 1u << kSliceBits) return fail(GUFFIN_E_SHAPE, "prefill_gemm: at most three matrices and 31 slices");
    GemmArgs a {};
    a.blob = image; a.M = M; a.K = K; a.form = slices;
    uint32_t groups = 0, kinds = 0;
    for (uint32_t i = 0; i < count; ++i) {
        a.tiles[i] = static_cast<const uint8_t*>(m[i].tiles); a.y[i] = y[i];
        a.columns[i] = m[i].N / kCols;
        a.form |= static_cast<uint32_t>(m[i].dtype) << (8 * (i + 1));
        groups += (a.columns[i] + 3) / 4;
        kinds |= m[i].dtype == GUFFIN_Q4_K ? 1u : m[i].dtype == GUFFIN_Q6_K ? 2u : 4u;
    }
    if (halves && (kinds != 1 || 2 * slices > K / 256)) return fail(GUFFIN_E_SHAPE, "prefill_gemm: a slice in halves is two blocks of Q4_K at least");
    if (kinds != 4 && slices > K / 256) return fail(GUFFIN_E_SHAPE, "prefill_gemm: a slice of a K-quant is a block at least");   // its walk begins with one unasked
    const uint32_t chunks = (M + 16 * R - 1) / (16 * R);
    dim3 grid(chunks, groups, slices), block(halves ? 512 : 256);
    const uint32_t units = groups * slices;
    if (const uint32_t ways = row_ways(chunks, units, kinds == 4u)) {
        const uint32_t others = 8 / ways;
        a.form |= (ways == 1 ? 1u : 2u) << kSliceBits;
        grid = dim3(8 * ((chunks + ways - 1) / ways) * ((units + others - 1) / others));
    }
#define GUFFIN_PG_ARGS a.tiles[0], a.tiles[1], a.tiles[2], a.blob, a.M, a.K, a.columns[0], a.columns[1], a.columns[2], a.form, a.y[0], a.y[1], a.y[2]
#define GUFFIN_PG(R_) \
    do { \
        if (halves) launch((prefill_gemm_kernel<R_, 1, 2>), grid, block, 2 * Stage<R_>::kBytes, s, GUFFIN_PG_ARGS); \
        else if (kinds == 1) launch(prefill_gemm_kernel<R_, 1>, grid, block, 0, s, GUFFIN_PG_ARGS); \
        else if (kinds == 2) launch(prefill_gemm_kernel<R_, 2>, grid, block, 0, s, GUFFIN_PG_ARGS); \
        else if (kinds == 3) launch(prefill_gemm_kernel<R_, 3>, grid, block, 0, s, GUFFIN_PG_ARGS); \
        else launch(prefill_gemm_q8_kernel<R_>, grid, block, 0, s, GUFFIN_PG_ARGS); \
    } while (0)
    if (R == 1) GUFFIN_PG(1); else if (R == 2) GUFFIN_PG(2); else if (R == 3) GUFFIN_PG(3); else GUFFIN_PG(4);
#undef GUFFIN_PG
#undef GUFFIN_PG_ARGS
    return check_launch("prefill_gemm");
}

// Time of a launch by a model of the chip, in microseconds: `start` from the launch to the first product and from the last one
// to the end, then every compute unit works off its share of the workgroups, each `workgroup` of its own and `unit` per slice unit -- 256
// elements of K, 64 for Q8_0 --, one workgroup by itself on a compute unit `alone` of that (it leaves gaps that a second one fills); a plane
// costs a write here and a read in the next operator.  Constants fitted to sweeps over 4 to 1000 rows of both models' shapes.
//
// K-quant launches of up to kShortRun rows have a set of their own, fitted to whole passes over every pair of 5 to 150 rows after the
// kernels had lost a tenth of their instructions: what a workgroup costs by itself counts there, and one workgroup a compute unit beats twice as
// many half as long.  It chooses among the cuts whose sums round no more than those of the other set's cut, see rounding().  A pass of the 12B
// shapes, us, by the other set / so: 5 rows 4568 / 4550, 20 rows 5430 / 5374, 37 rows 6429 / 6293, 55 rows 7430 / 7137, 64 rows 7701 / 7302, 100 rows
// 10453 / 10121, 128 rows 10671 / 10406; what planes cost differs from machine to machine, on another one 37 rows 6198 / 6215, 64 rows 7381 / 7131, 100
// rows 9901 / 9909.  Past the line it finds nothing in most runs and loses some: 200 rows 14528 / 14638, 512 rows 26588 / 26793.
struct SplitCosts { float start[4], unit[3][4], alone[4], workgroup, plane_bytes; };   // unit: Q8_0, Q4_K, Q6_K
constexpr uint32_t kShortRun = 192;   // whole row tiles
constexpr SplitCosts kShort = {{4.6f, 6.7f, 8.2f, 9.3f}, {{}, {2.27f, 2.61f, 3.19f, 4.08f}, {2.92f, 3.62f, 4.73f, 5.61f}}, {1.21f, 1.19f, 1.17f, 1.11f}, 5.1f, 14.4e6f};
constexpr SplitCosts kLong = {{5.0f, 6.2f, 7.5f, 8.5f}, {{0.6f, 0.82f, 1.0f, 1.35f}, {2.3f, 2.7f, 3.2f, 3.8f}, {2.8f, 3.3f, 4.0f, 4.8f}},
                              {1.22f, 1.22f, 1.22f, 1.22f}, 0.0f, 5.0e6f};

// The part of a sum's squared error that its cut decides: an addition rounds at the size its chain has reached, so a chain of
// units / S blocks (half as many in halves) counts by its length and the one over S planes by its own, weighted by what a block's other
// roundings leave of it.  rms error from 64 bits, 1e-7 of the result's rms, of 1, 2, 4, 8 and all slices: Q4_K, K = 3840 1.52, 1.38, 1.33, 1.33,
// 1.40, K = 15360 2.30, 1.85, 1.59, 1.49, (16) 1.50; Q6_K, K = 3840 1.79, 1.74, 1.73, 1.75, 1.82, K = 15360 2.17, 1.96, 1.85, 1.82, (16)
// 1.86; Q4_K in halves, 1, 2 and 4 slices: K = 3840 1.38, 1.33, 1.32, K = 15360 1.86, 1.59, 1.47.
constexpr float kPlaneRounding[3] = {0.f, 0.54f, 1.2f};
constexpr float rounding(uint32_t units, uint32_t S, uint32_t halves, float plane) { return float(units) / float(S << halves) + plane * float(S + halves); }

constexpr float kHalvesCost = 2.0f;   // us: twice the first trips at once, sums from team to team
struct SplitShape { uint32_t units, groups, width, most; bool q8; float unit[4]; };   // units: what a slice is made of; unit: of a workgroup, the mean over the launch
SplitShape split_shape(const PrefillMatrix* m, uint32_t count, uint32_t K, uint32_t most, const SplitCosts& costs) {
    SplitShape s {};
    for (uint32_t i = 0; i < count; ++i) {
        const uint32_t n = (m[i].N / kCols + 3) / 4;
        s.q8 |= m[i].dtype == GUFFIN_Q8_0;
        s.groups += n;
        s.width += m[i].N;
        for (int r = 0; r < 4; ++r) s.unit[r] += float(n) * costs.unit[m[i].dtype][r];
    }
    s.units = s.q8 ? (K + 63) / 64 : K / 256;
    // A Q8_0 slice has two units at least: a single one is a workgroup's first trips and little else, and leaves twice the planes (q/k/v of the
    // 640-wide drafter: ten, which the next operator asks for in two goes).  A pass, us, with slices of one unit / so: 16 rows 786 / 756, 30 rows
    // 836 / 795, 48 rows 884 / 838, 57 rows 989 / 930; from 64 rows on, where the model cuts less, 865 / 852 and 0.3-0.9 % less.
    s.most = std::max(1u, std::min(most, s.q8 ? s.units / 2 : s.units));
    return s;
}

template <typename Allowed>
PrefillSplit cheapest_split(const SplitShape& s, const SplitCosts& costs, uint32_t M, Allowed allowed, uint32_t most_halves = 0) {
    const uint32_t cus = compute_units();
    const float plane = 8.0f * float(M) * float(s.width) / costs.plane_bytes;
    PrefillSplit best {};
    float least = 0.f;
    for (uint32_t R = 1; R <= 4; ++R) {
        const uint32_t chunks = (M + 16 * R - 1) / (16 * R);
        for (uint32_t S = 1; S <= s.most; ++S) {
            const float fixed = costs.start[R - 1] + float(S) * plane;
            if (best.slices && fixed >= least) break;   // grows with S
            for (uint32_t halves = 0; halves <= most_halves; ++halves) {
                const uint32_t n = chunks * s.groups * S;
                // (halves: two teams are what a compute unit takes)
                if (!allowed(R, S, halves) || (halves && n > cus)) continue;
                // the last, partly filled turn overlaps the one before it: half of it counts
                const float turns = halves ? 1.f : std::max(costs.alone[R - 1], 0.5f * (float((n + cus - 1) / cus) + float(n) / float(cus)));
                const uint32_t units = halves ? 2 * ((s.units + 2 * S - 1) / (2 * S)) : (s.units + S - 1) / S;   // a team's, each beside the other's
                const float cost = fixed + float(halves) * kHalvesCost + turns * (costs.workgroup + float(units) * s.unit[R - 1] / float(s.groups));
                if (!best.slices || cost < least) { best = {R, S, halves}; least = cost; }
            }
        }
    }
    return best;
}

PrefillSplit split_for(const PrefillMatrix* m, uint32_t count, uint32_t M, uint32_t K, uint32_t most) {
    const SplitShape shape = split_shape(m, count, K, most, kLong);
    auto any = [](uint32_t, uint32_t, uint32_t) { return true; };
    if (shape.q8 || M > kShortRun) return cheapest_split(shape, kLong, M, any);
    // one cut for all runs of as many row tiles, by the costs in their middle: it holds against the other set's for the shortest and the longest
    const uint32_t last = (M + 15) & ~15u;
    const PrefillSplit bar[2] = {cheapest_split(shape, kLong, last - 15, any), cheapest_split(shape, kLong, last, any)};
    bool q4 = true;
    for (uint32_t i = 0; i < count; ++i) q4 &= m[i].dtype == GUFFIN_Q4_K;
    auto close = [&](uint32_t, uint32_t S, uint32_t halves) {
        if (halves && 2 * S > std::max(bar[0].slices, bar[1].slices)) return false;   // halves stand for two of its slices
        for (uint32_t i = 0; i < count; ++i)
            for (const PrefillSplit& b : bar)
                if (rounding(shape.units, S, halves, kPlaneRounding[m[i].dtype]) > rounding(shape.units, b.slices, 0, kPlaneRounding[m[i].dtype])) return false;
        return true;
    };
    const PrefillSplit best = cheapest_split(split_shape(m, count, K, most, kShort), kShort, last - 8, close, q4 && most > 1 ? 1u : 0u);
    return best.slices ? best : bar[1];
}

}  // namespace

int prefill_gemm_init() {
    return allow_lds(prefill_gateup_q8_kernel<4>, GatedStage<4>::kBytes) && allow_lds((prefill_gemm_kernel<2, 1, 2>), 2 * Stage<2>::kBytes)
        && allow_lds((prefill_gemm_kernel<3, 1, 2>), 2 * Stage<3>::kBytes) && allow_lds((prefill_gemm_kernel<4, 1, 2>), 2 * Stage<4>::kBytes) ? 0 : -1;
}

// The fewest row tiles a workgroup with which every workgroup has a compute unit, as long as more than half of them have work: a
// launch, a write and a read of both products less.  A pass of the drafter (640 x 2048, 18 blocks), us, as two launches / so: 270 rows 1256 /
// 1214, 512 1523 / 1461, 1024 2009 / 1896, 1536 2624 / 2491, 2048 3035 / 2905; fewer rows leave the chip idle (240: 1182 / 1185; 64: 912 /
// 979), two row tiles where one is enough cost more (512: 1556).  Wider models form B too often so: 768 x 2304 1923 / 1855 at 700 rows, but
// 1024 x 4096 1708 / 1762 at 300 and 2048 x 8192 1800 / 2003 at 100.
uint32_t prefill_gateup_tiles(int gate_dtype, int up_dtype, uint32_t rows, uint32_t K, uint32_t F) {
    if (gate_dtype != GUFFIN_Q8_0 || up_dtype != GUFFIN_Q8_0 || F % 256 != 0 || K > 768) return 0;
    const uint32_t cus = compute_units();
    for (uint32_t R = 1; R <= 4; ++R)
        if ((rows + 16 * R - 1) / (16 * R) * (F / 256) <= cus) return R > 1 || (rows + 15) / 16 * (F / 256) > cus / 2 ? R : 0;
    return 0;
}

int prefill_gateup(hipStream_t s, const void* gate, const void* up, const uint8_t* image, uint32_t M, uint32_t K, uint32_t F, uint32_t R, uint8_t* out) {
    if (K % 32 != 0 || F % 256 != 0) return fail(GUFFIN_E_SHAPE, "prefill_gateup: need K % 32 == 0 and F % 256 == 0");
    if ((reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(up)) & 15u) return fail(GUFFIN_E_ALIGN, "prefill_gateup: tiles need 16-byte alignment");
    if (image_layout(M, K).bytes >= (size_t(1) << 31)) return fail(GUFFIN_E_SHAPE, "prefill_gateup: the image of M x K exceeds 2 GiB, split the rows");
    const dim3 grid((M + 16 * R - 1) / (16 * R), F / 256), block(512);
    const uint8_t *g = static_cast<const uint8_t*>(gate), *u = static_cast<const uint8_t*>(up);
#define GUFFIN_PG(R_) launch(prefill_gateup_q8_kernel<R_>, grid, block, GatedStage<R_>::kBytes, s, g, u, image, M, K, F, out)
    if (R == 1) GUFFIN_PG(1); else if (R == 2) GUFFIN_PG(2); else if (R == 3) GUFFIN_PG(3); else GUFFIN_PG(4);
#undef GUFFIN_PG
    return check_launch("prefill_gateup");
}

constexpr uint32_t kMostSlices = 16;
PrefillSplit prefill_split(const PrefillMatrix* m, uint32_t count, uint32_t M, uint32_t K) { return split_for(m, count, M, K, kMostSlices); }

// Runs of as many row tiles differ in what a plane costs alone, so the shortest of them has the most slices and the longest the most rows.
uint64_t prefill_most_rows(const PrefillMatrix* m, uint32_t count, uint32_t rows, uint32_t K, uint64_t least) {
    const uint32_t most = split_shape(m, count, K, kMostSlices, kLong).most;
    for (uint32_t last = rows; last > 0 && uint64_t(most) * last > least; last = (last - 1) & ~15u)
        least = std::max(least, uint64_t(prefill_split(m, count, ((last - 1) & ~15u) + 1, K).slices) * last);
    return least;
}

int prefill_gemm_planes(hipStream_t s, const PrefillMatrix* m, uint32_t count, const uint8_t* image, float* const* y, uint32_t M,
                        uint32_t K, PrefillSplit split) {
    bool q8 = false, k = false;
    for (uint32_t i = 0; i < count; ++i) {
        if (K % block_elems(m[i].dtype) != 0 || m[i].N % kCols != 0) return fail(GUFFIN_E_SHAPE, "prefill_gemm: need K % block == 0 and N % 64 == 0");
        if (reinterpret_cast<uintptr_t>(m[i].tiles) & 15u) return fail(GUFFIN_E_ALIGN, "prefill_gemm: tiles need 16-byte alignment");
        (m[i].dtype == GUFFIN_Q8_0 ? q8 : k) = true;
    }
    if (image_layout(M, K).bytes >= (size_t(1) << 31)) return fail(GUFFIN_E_SHAPE, "prefill_gemm: the image of M x K exceeds 2 GiB, split the rows");
    if (q8 && k) {   // the formats' workgroups walk K in different units: a launch each
        for (uint32_t i = 0; i < count; ++i) {
            // The cut is by Q8_0's finer units.  Where it has more slices than a K-quant has blocks, each block is a slice of its own, in order,
            // and the planes behind them are zeros: so the kernels, whose walks have a block at least, need no test of their own.
            const uint32_t blocks = m[i].dtype == GUFFIN_Q8_0 ? split.slices : std::min(split.slices, K / 256);
            if (int rc = prefill_gemm_planes(s, m + i, 1, image, y + i, M, K, {split.row_tiles, blocks, split.halves})) return rc;
            const uint64_t plane = uint64_t(M) * m[i].N, quads = (split.slices - blocks) * plane / 4;
            if (quads) launch(zero_planes_kernel, dim3(static_cast<uint32_t>((quads + 255) / 256)), dim3(256), 0, s, y[i] + blocks * plane, quads);
            if (int rc = check_launch("prefill_gemm planes")) return rc;
        }
        return GUFFIN_OK;
    }
    return gemm_launch(s, m, count, image, y, M, K, split.slices, split.row_tiles, split.halves);
}
}  // namespace guffin

using namespace guffin;

extern "C" uint64_t guffin_hip_prefill_image_bytes(uint32_t M, uint32_t K) {
    if (M == 0 || K == 0 || K % 32 != 0) return 0;
    return image_layout(M, K).bytes;
}

extern "C" int guffin_hip_prefill_pack(void* stream, const float* x, void* image, uint32_t M, uint32_t K) {
    if (!x || !image) return fail(GUFFIN_E_ARG, "prefill_pack: null pointer");
    if (M == 0 || K == 0 || K % 32 != 0) return fail(GUFFIN_E_SHAPE, "prefill_pack: K must be a positive multiple of 32");
    if (reinterpret_cast<uintptr_t>(image) & 255u) return fail(GUFFIN_E_ALIGN, "prefill_pack: the image must be 256-byte aligned");
    const uint64_t threads = uint64_t(M) * (K / 8);
    launch(prefill_pack_kernel, dim3(static_cast<uint32_t>((threads + 255) / 256)), dim3(256), 0,
                       as_stream(stream), x, static_cast<uint8_t*>(image), M, K);
    return check_launch("prefill_pack");
}

extern "C" int guffin_hip_prefill_gemm(void* stream, int dtype, const void* tiles, const void* image, float* y,
                                       uint32_t M, uint32_t K, uint32_t N) {
    if (!tiles || !image || !y) return fail(GUFFIN_E_ARG, "prefill_gemm: null pointer");
    if (dtype < GUFFIN_Q8_0 || dtype > GUFFIN_Q6_K) return fail(GUFFIN_E_ARG, "prefill_gemm: unknown dtype");
    if (M == 0 || K == 0 || N == 0 || K % block_elems(dtype) != 0 || N % kCols != 0)
        return fail(GUFFIN_E_SHAPE, "prefill_gemm: need K % block == 0 and N % 64 == 0");
    if ((reinterpret_cast<uintptr_t>(tiles) & 15u) || (reinterpret_cast<uintptr_t>(image) & 255u))
        return fail(GUFFIN_E_ALIGN, "prefill_gemm: tiles need 16-byte, the image 256-byte alignment");
    // the kernels address the image with 32-bit offsets
    if (image_layout(M, K).bytes >= (size_t(1) << 31)) return fail(GUFFIN_E_SHAPE, "prefill_gemm: the image of M x K exceeds 2 GiB, split the rows");
    const PrefillMatrix m {dtype, tiles, N};
    return gemm_launch(as_stream(stream), &m, 1, static_cast<const uint8_t*>(image), &y, M, K, 1, split_for(&m, 1, M, K, 1).row_tiles, false);
}
