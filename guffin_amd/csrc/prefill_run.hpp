// What the prefill pass (plan.hip) asks of the files that hold its kernels.
#pragma once
#include "common.hpp"

namespace guffin {

// ---- GEMM (prefill_gemm.hip) ---------------------------------------------------------------
struct PrefillMatrix { int dtype; const void* tiles; uint32_t N; };
// rows per workgroup in tiles of 16, and k-slices: every slice leaves a plane of partial sums; halves (Q4_K alone): a workgroup adds up its
// slice as two
struct PrefillSplit { uint32_t row_tiles, slices, halves; };
// the split for `count` matrices (at most 3) over the same K that run as one launch
PrefillSplit prefill_split(const PrefillMatrix* m, uint32_t count, uint32_t M, uint32_t K);
// the most plane rows (slices times rows) that the launch keeps in any run of up to `rows` rows, or `least` if that is more
uint64_t prefill_most_rows(const PrefillMatrix* m, uint32_t count, uint32_t rows, uint32_t K, uint64_t least);
// y[i]: split.slices planes of [M][N_i], one behind the other
int prefill_gemm_planes(hipStream_t s, const PrefillMatrix* m, uint32_t count, const uint8_t* image, float* const* y, uint32_t M,
                        uint32_t K, PrefillSplit split);

// gate, up and GeGLU of a Q8_0 block as one launch: out is the down projection's operand (not the memory of image)
// row_tiles: of a workgroup; prefill_gateup_tiles has them, 0: the launches apart
uint32_t prefill_gateup_tiles(int gate_dtype, int up_dtype, uint32_t rows, uint32_t K, uint32_t F);
int prefill_gateup(hipStream_t s, const void* gate, const void* up, const uint8_t* image, uint32_t M, uint32_t K, uint32_t F, uint32_t row_tiles, uint8_t* out);

// ---- attention (prefill.hip) -----------------------------------------------------------------
struct ValueSpan { uint32_t first_visible, base32, T; };
// virtual tokens whose values a run of `rows` rows at `position` can see, padded to whole 32-token tiles
inline ValueSpan value_span(uint32_t rows, uint32_t position, uint32_t window) {
    const uint32_t first = (window && position + 1 > window) ? position + 1 - window : 0;
    const uint32_t base32 = first & ~31u;
    return {first, base32, (position + rows - base32 + 31u) & ~31u};
}
// Element e of k-slice lg of a dimension's 32 tokens in V^T: the tokens whose probabilities lane group lg has (four of either half).
__host__ __device__ constexpr uint32_t value_token(uint32_t lg, uint32_t e) { return (e < 4 ? 0u : 12u) + 4 * lg + e; }
// The matrix-core path wants one, two or four query heads per KV head, and K/V rows and queries at 16-byte addresses.
bool prefill_attention_on_matrix_core(const void* q, const void* ring_k, const void* ring_v, const void* run_k, const void* run_v,
                                      uint32_t q_heads, uint32_t kv_heads);
// the workspace of a run of `rows` rows that sees at most T tokens; the largest of any run of up to `rows` rows
uint64_t prefill_attention_bytes(uint32_t rows, uint32_t T, uint32_t q_heads, uint32_t kv_heads);
uint64_t prefill_attention_most_bytes(uint32_t rows, uint32_t T, uint32_t q_heads, uint32_t kv_heads);
// workspace: the transposed values of the span (already there) and room for the parts' states behind them; image: the
// operand of the o projection
int prefill_attention_run(hipStream_t s, const float* q, const void* ring_k, const void* run_k, float* out, uint8_t* image, uint32_t rows,
                          uint32_t position, uint32_t window, uint32_t ring_mask, uint32_t q_heads, uint32_t kv_heads, float scale,
                          void* workspace);

// ---- between the GEMMs (prefill_ops.hip) -------------------------------------------------------
constexpr uint32_t kPrefillMaxWidth = 8192;   // widest row the norm kernels hold (8 columns per thread)
// K/V rows of the run on their way to the ring; run_k null: none.  Rows before first_row would be overwritten anyway.
struct RunRows { const void *run_k, *run_v; void *ring_k, *ring_v; uint32_t first_row, position, ring_mask, row_vec; };
struct QkvRun {
    const float *q_planes, *k_planes, *v_planes;   // planes of [rows][heads * 256]
    const float *q_norm, *k_norm, *rope_table;     // table [rows][128] of cos, sin
    float* q_out; uint16_t *k_out, *v_out;         // [rows][heads * 256]
    const uint16_t* ring_v; uint16_t* vt;          // vt [kv_heads][T / 32][256][32], tokens as value_token has them
    uint32_t planes, rows, q_heads, kv_heads, position, ring_mask, first_visible, base32, T, head_groups;
    float eps;
    uint32_t* status;
};
int prefill_norm(hipStream_t s, const float* x, const float* gamma, uint8_t* image, uint32_t rows, uint32_t width, float eps, uint32_t* status);
int prefill_joint(hipStream_t s, const float* x, uint32_t planes, const float* gamma_post, const float* residual, float* out_residual,
                  const float* gamma_next, float* out_norm, uint8_t* image, uint32_t rows, uint32_t width, float eps, const RunRows& run,
                  uint32_t* status);
int prefill_geglu(hipStream_t s, const float* gate, const float* up, uint32_t planes, uint8_t* image, uint32_t rows, uint32_t width);
int prefill_qkv(hipStream_t s, QkvRun a);

}  // namespace guffin
