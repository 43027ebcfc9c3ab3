// The streaming product for 3 and 4 rows (verify trees, the shortest prompt runs).
//
// Same tiles, operands and arithmetic as the kernels of gemv_packed.hip, the K-quants through the same code with a second set of
// four variants: a weight byte is fetched and unpacked once for four rows where two passes of two rows do it twice.  A split that
// leaves every wave one block holds one tile a lane and runs up to sixteen waves a workgroup; otherwise a lane holds two tiles and
// the operands of two blocks, which is more than the 128 registers sixteen waves would leave it, and eight run.  Q8_0 keeps the
// 16x16x32 instruction, whose 16 rows hold the 8 variants twice: lane (j, g) has the sums of rows 2 (g % 2) and + 1, columns
// 32 (g / 2) + j and + 16.
// Blocks of a 12B-shaped stack, four rows, with the operand staged in LDS for the 16x16x32 form / now / two launches of two rows
// (us): q/k/v 8.7 / 8.4 / 14.3, o 4.8 / 5.7 / 9.1, gate + up 19.3 / 17.2 / 29.8, down 15.1 / 12.2 / 21.5.  (The block's multipliers
// and sums brought to scalar registers ahead of the tile, which 64 to 96 words do not fit: down 14.1, q/k/v 11.2.)
// Three rows leave the last pair of variants zero and its row unwritten.
#include "common.hpp"
#include "receipt.hpp"
#include "gemv_tiles.hpp"

namespace guffin {
namespace {

constexpr uint32_t kWideWaves = 8;
constexpr int kWideMixed = 3;   // Q4_K and Q6_K matrices in one launch

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

// One wave: blocks [b0, b1) of column tile `ct` against the receipt of four rows of K activations; the sums go to red[row][64 columns].
template <int DTYPE, int WALK = kWalkAhead>
__device__ __forceinline__ void run_wide(const uint8_t* __restrict__ wt, const float* __restrict__ xsums, uint32_t K, uint32_t nblk,
                                         uint32_t ct, uint32_t b0, uint32_t b1, float* red, uint32_t lane) {
    constexpr uint32_t TB = kTileCols * block_bytes(DTYPE);
    if constexpr (DTYPE != GUFFIN_Q8_0) {
        float acc[kWideRows];
        run_blocks<DTYPE, kWideRows, WALK>(wt, xsums, K, nblk, ct, b0, b1, acc);
#pragma unroll
        for (uint32_t r = 0; r < kWideRows; ++r) red[r * 64 + lane] = acc[r];
    } else {
        const ReceiptLayout L = receipt_layout(kWideRows, K);
        const uint8_t* tp = wt + (size_t(ct) * nblk + b0) * TB + lane * 16;
        const uint32_t n16 = K / 16, n32 = K / 32, per_row = n16 + n32, pair = (lane >> 4) & 1u;
        const uint8_t* base = reinterpret_cast<const uint8_t*>(xsums);
        const float* mult = reinterpret_cast<const float*>(base + L.mult_off) + 2 * pair * size_t(n32);
        const float* xs = xsums + 2 * pair * size_t(per_row) + n16;
        const uint8_t* image = base + L.image_off + (lane & 7u) * 64u + (lane >> 4) * 16u;
        float acc[2][2] = {};
        Q8Wide cur, nxt;
        if (b0 < b1) load_tile(cur, tp, lane);
        for (uint32_t b = b0; b < b1; ++b, tp += TB) {
            const half8_t a = __builtin_bit_cast(half8_t, *reinterpret_cast<const uint4*>(image + size_t(b) * 512u));
            const float m[2] = {mult[b], mult[n32 + b]}, x[2] = {xs[b], xs[per_row + b]};
            if (b + 1 < b1) load_tile(nxt, tp + TB, lane);
            compute_tile(cur, a, m, x, lane, acc);
            cur = nxt;
        }
#pragma unroll
        for (uint32_t c = 0; c < 2; ++c)
#pragma unroll
            for (uint32_t r = 0; r < 2; ++r) red[(2 * pair + r) * 64 + 32 * (lane >> 5) + 16 * c + (lane & 15u)] = acc[c][r];
    }
}

// Up to three matrices of the same rows, their column tiles side by side along grid x; grid y: planes.  (The arguments' order: as
// for the kernels of gemv_packed.hip.)  end0, end1: the tiles of the first matrix, of the first two; dtypes: a byte each.
template <int MODE, uint32_t WAVES>
__global__ void __launch_bounds__(64 * WAVES)
gemv_wide_kernel(const uint8_t* __restrict__ t0, const uint8_t* __restrict__ t1, const uint8_t* __restrict__ t2, const float* __restrict__ xsums,
                 uint32_t end0, uint32_t end1, uint32_t dtypes, uint32_t K, uint32_t bps, uint32_t W, uint32_t rows, uint32_t n0, uint32_t n1,
                 uint32_t n2, float* __restrict__ p0, float* __restrict__ p1, float* __restrict__ p2) {
    __shared__ float red[WAVES * kWideRows * 64];
    const uint32_t which = blockIdx.x >= end1 ? 2u : blockIdx.x >= end0 ? 1u : 0u;
    const uint8_t* wt = which == 0 ? t0 : which == 1 ? t1 : t2;
    float* part = which == 0 ? p0 : which == 1 ? p1 : p2;
    const uint32_t N = which == 0 ? n0 : which == 1 ? n1 : n2, nblk = K / block_elems(MODE == kWideMixed ? GUFFIN_Q4_K : MODE);
    [[maybe_unused]] const uint32_t dtype = (dtypes >> (8 * which)) & 0xFFu;
    const uint32_t ct = blockIdx.x - (which == 0 ? 0u : which == 1 ? end0 : end1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t slice = blockIdx.y * W + wave, b0 = min(slice * bps, nblk), b1 = min(b0 + bps, nblk);
    float* own = red + wave * kWideRows * 64;
    if constexpr (MODE == kWideMixed) {
        if (dtype == GUFFIN_Q4_K) run_wide<GUFFIN_Q4_K, (WAVES > kWideWaves ? kWalkOne : kWalkAhead)>(wt, xsums, K, nblk, ct, b0, b1, own, lane);
        else run_wide<GUFFIN_Q6_K, (WAVES > kWideWaves ? kWalkOne : kWalkAhead)>(wt, xsums, K, nblk, ct, b0, b1, own, lane);
    } else {
        run_wide<MODE, (WAVES > kWideWaves ? kWalkOne : kWalkAhead)>(wt, xsums, K, nblk, ct, b0, b1, own, lane);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < rows * 64; i += 64 * W) {
        const float t = sum_of_waves<WAVES>(red + i, kWideRows * 64, W);
        part[(size_t(blockIdx.y) * rows + (i >> 6)) * N + ct * kTileCols + (i & 63u)] = t;
    }
}

// gate and up of one column tile and GeGLU, as gateup_geglu_kernel: waves [0, W) gate, [W, 2W) up
template <int DTYPE>
__global__ void __launch_bounds__(64 * kWideWaves)
gateup_wide_kernel(const uint8_t* __restrict__ gate_tiles, const uint8_t* __restrict__ up_tiles, const float* __restrict__ xsums,
                   uint32_t K, uint32_t bps, uint32_t W, uint32_t F, uint32_t rows, float* __restrict__ h,
                   void* __restrict__ h_receipt) {
    __shared__ float red[kWideWaves * kWideRows * 64];
    __shared__ float vals[kWideRows * 64];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t nblk = K / block_elems(DTYPE);
    const bool is_up = wave >= W;
    const uint32_t slice = is_up ? wave - W : wave, b0 = min(slice * bps, nblk), b1 = min(b0 + bps, nblk);
    run_wide<DTYPE>(is_up ? up_tiles : gate_tiles, xsums, K, nblk, blockIdx.x, b0, b1, red + wave * kWideRows * 64, lane);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < rows * 64; i += 128 * W) {
        const float v = geglu_value(sum_of_waves<kWideWaves / 2>(red + i, kWideRows * 64, W),
                                    sum_of_waves<kWideWaves / 2>(red + W * kWideRows * 64 + i, kWideRows * 64, W));
        h[size_t(i >> 6) * F + blockIdx.x * kTileCols + (i & 63u)] = v;
        vals[i] = v;
    }
    lds_barrier();   // h is on its way out and nobody here reads it
    // a wave a row; a tile of one k-slice has two waves for up to four rows
    for (uint32_t r = wave; r < rows; r += 2 * W) emit_receipt(vals + r * 64, blockIdx.x * kTileCols, kTileCols, r, rows, F, h_receipt, lane, 64);
}

__global__ void wide_reduce_kernel(const float* __restrict__ part, float* __restrict__ y, uint32_t planes, uint32_t count) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) y[i] = load_planes(part + i, planes, count);
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
    // a split that leaves every wave one block runs with a tile in registers at a time, and sixteen waves
    const uint32_t nblk = K / block_elems(dtypes[0]);
    *split = gemv_split(nblk, tiles, 16, 16);
    if (split->bps != 1) *split = gemv_split(nblk, tiles, kWideWaves, kWideWaves);
    return GUFFIN_OK;
}

}  // namespace

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
    const uint8_t* t[3];
    float* p[3];
    uint32_t n[3], ends[3], end = 0, formats = 0;
    for (uint32_t i = 0; i < 3; ++i) {
        const uint32_t k = i < count ? i : 0;
        if (i < count) end += N[i] / kTileCols;
        t[i] = static_cast<const uint8_t*>(tiles[k]); p[i] = partials[k]; n[i] = N[k]; ends[i] = end;
        formats |= static_cast<uint32_t>(dtypes[k]) << (8 * i);
    }
    if (y && sp.planes == 1) p[0] = y;   // one plane is the result
    const dim3 grid(end, sp.planes), block(64 * sp.W);
#define GUFFIN_WIDE(M_) do { if (sp.bps == 1) launch((gemv_wide_kernel<M_, 16>), grid, block, 0, s, GUFFIN_WIDE_ARGS); \
        else launch((gemv_wide_kernel<M_, kWideWaves>), grid, block, 0, s, GUFFIN_WIDE_ARGS); } while (0)
#define GUFFIN_WIDE_ARGS t[0], t[1], t[2], xsums, ends[0], ends[1], formats, K, sp.bps, sp.W, rows, n[0], n[1], n[2], p[0], p[1], p[2]
    if (mode == GUFFIN_Q4_K) GUFFIN_WIDE(GUFFIN_Q4_K);
    else if (mode == GUFFIN_Q6_K) GUFFIN_WIDE(GUFFIN_Q6_K);
    else if (mode == GUFFIN_Q8_0) GUFFIN_WIDE(GUFFIN_Q8_0);
    else GUFFIN_WIDE(kWideMixed);
#undef GUFFIN_WIDE_ARGS
#undef GUFFIN_WIDE
    if (int rc = check_launch("gemv_wide")) return rc;
    if (!y || sp.planes == 1) return GUFFIN_OK;
    const uint32_t elements = rows * N[0];
    launch(wide_reduce_kernel, dim3((elements + 255) / 256), dim3(256), 0, s, partials[0], y, sp.planes, elements);
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
    const dim3 grid(F / kTileCols), block(2 * sp.W * 64);
    const uint8_t *g = static_cast<const uint8_t*>(gate_tiles), *u = static_cast<const uint8_t*>(up_tiles);
    if (dtype == GUFFIN_Q4_K) launch(gateup_wide_kernel<GUFFIN_Q4_K>, grid, block, 0, s, g, u, xsums, K, sp.bps, sp.W, F, rows, h, static_cast<void*>(h_sums));
    else launch(gateup_wide_kernel<GUFFIN_Q8_0>, grid, block, 0, s, g, u, xsums, K, sp.bps, sp.W, F, rows, h, static_cast<void*>(h_sums));
    return check_launch("gateup_wide");
}

}  // namespace guffin
