// Shared device helpers for the gfx950 kernels of the H1 step.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/guffin_hip.h"
#include "chain.hpp"

namespace guffin {

constexpr int kWave = 64;

// ---- error plumbing (host) -------------------------------------------------
void set_last_error(const char* message);
int fail(int code, const char* message);
int check_launch(const char* what);

// Lets `kernel` ask for more than 64 KB of dynamic LDS on the current device.  The permission is a device's own, so this runs in
// the init functions that guffin_hip_init calls, once per device, and nowhere else.
template <typename Kernel>
inline bool allow_lds(Kernel* kernel, uint32_t bytes) {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)) == hipSuccess;
}

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// Layer policy of src/engine/model.cpp:607-610: with a period above one, every layer but the last of
// each period uses the sliding window (local ring, local rotation base); otherwise every layer is global.
__host__ __device__ inline bool layer_is_local(uint32_t global_period, uint32_t layer) {
    return global_period > 1 && (layer % global_period) != global_period - 1;
}

// ---- resident forward pass (resident.hip), used by the block graph of plan.hip ------------------
constexpr uint32_t kResidentLayers = 6;   // blocks per launch (their pointers travel as kernel arguments)
extern uint32_t g_spin_limit;
extern unsigned long long* g_resident_stamps;
extern int g_forward_mode;
bool resident_fits(const guffin_model_desc& m, uint32_t rows);
// Whether forward_rows runs the resident pass for this model now: the model fits, the mode asks for it (2) or leaves
// the choice open (0) for a model with one KV head, and no earlier pass of this process gave up a wait.
bool resident_chosen(const guffin_model_desc& m, uint32_t rows);
// Host code that reads a device status word reports it here: GUFFIN_STATUS_SYNC switches the automatic choice of
// the resident pass off for the rest of the process (a device shared with other work, or one whose dispatcher does
// not place the workgroups as the pass assumes, would raise it on every pass).
void resident_note_status(uint32_t status_word);
int resident_init(int cu_count);
uint64_t resident_scratch_bytes(const guffin_model_desc& m, uint32_t rows);
uint32_t resident_sync_words(const guffin_model_desc& m);
int resident_launch(hipStream_t stream, const guffin_model_desc& m, uint32_t rows, uint32_t first, uint32_t count,
                    uint8_t* exchange, uint32_t* sync_words, const float* rope_local, const float* rope_global,
                    const uint32_t* schedule, const uint32_t* ancestors, void* priv_k, void* priv_v, const float* x_in,
                    const void* u_receipt_in, float* x_out, float* u_out, void* u_receipt_out, uint32_t max_ring_tokens,
                    uint32_t* status);

// Up to kRunRows contiguous rows of a model that the drafter's pass covers (plan.hip): every row's final state to row_states (or null),
// the last one's with its receipt to last_state / last_receipt as well.  scratch: forward_run_bytes, 256-byte aligned; priv_k,
// priv_v: [block][rows][kv width].  A row's results are those of a pass by itself, bit for bit.
constexpr uint32_t kRunRows = 8;          // XCDs of the part
bool forward_run_chosen(const guffin_model_desc& m);
uint64_t forward_run_bytes(const guffin_model_desc& m);
int forward_run(hipStream_t stream, const guffin_model_desc& m, const uint32_t* tokens, uint32_t rows, uint32_t position, void* scratch,
                void* priv_k, void* priv_v, float* row_states, float* last_state, float* last_receipt, uint32_t* status);

// ---- streaming products of 3 and 4 rows (gemv_wide.hip) -------------------------------------------------------
constexpr uint32_t kWideRows = 4;
// The work split of a streaming product over `tiles` column tiles of `nblk` blocks (gemv_packed.hip): blocks per wave, waves per
// workgroup (at most max_w) and planes left to the consumer; waves_per_cu waves are assumed to fit a CU.
struct GemvSplit { uint32_t bps, W, planes; };
uint32_t compute_units();   // of the device the library was initialised on (256 before that)
GemvSplit gemv_split(uint32_t nblk, uint32_t tiles, uint32_t max_w, uint32_t waves_per_cu);
uint32_t gemv_wide_planes(uint32_t count, const int* dtypes, const uint32_t* N, uint32_t K);
// partials[i]: [planes][rows][N[i]]; y (one matrix): the planes' sum [rows][N]
int gemv_wide(hipStream_t s, uint32_t count, const int* dtypes, const void* const* tiles, const uint32_t* N, float* const* partials,
              const float* xsums, float* y, uint32_t rows, uint32_t K);
int gateup_wide(hipStream_t s, int dtype, const void* gate_tiles, const void* up_tiles, const float* xsums, float* h, float* h_sums,
                uint32_t rows, uint32_t K, uint32_t F);

// ---- K/V rows of every block of a model between its rings and a flat block of rows (prefill.hip) ---------------
// flat_k / flat_v: [layer][flat_rows][kv width], position p in row p & (flat_rows - 1), flat_rows a power of two.  Save and
// Restore copy positions [first, first + count); Publish saves them and then puts row path[i] of the private rows
// [layer][priv_rows][kv width] at position first + i; Put does that without saving (no flat block).
enum class KvMove { Save, Restore, Publish, Put };
constexpr uint32_t kMovePath = 8;   // rows a Publish or Put may take
int kv_move_rows(hipStream_t s, const guffin_model_desc& m, KvMove move, void* flat_k, void* flat_v, uint32_t flat_rows, uint32_t first,
                 uint32_t count, const void* priv_k = nullptr, const void* priv_v = nullptr, uint32_t priv_rows = 0,
                 const uint32_t* path = nullptr);

// ---- a whole verify tree of up to 4 rows in one pass (plan.hip) -----------------------------------------------------
bool tree_pass_fits(const guffin_model_desc& m);
uint64_t tree_pass_bytes(const guffin_model_desc& m, uint32_t position);   // scratch of a tree at that position
int forward_tree_pass(hipStream_t stream, const guffin_model_desc& m, const uint32_t* tokens, uint32_t rows, uint32_t position,
                      const uint32_t* depths, const uint32_t* parents, void* scratch, uint64_t scratch_bytes, void* priv_k, void* priv_v,
                      float* out_hidden, float* out_hidden_sums, uint32_t* status);

// guffin_hip_commit_rows of every row, with the rows' final states kept: kept[row] = hidden[row] unless kept is null (plan.hip)
int commit_rows_keeping(void* stream, const guffin_model_desc& m, const void* priv_k, const void* priv_v, void* const* ring_k_table,
                        void* const* ring_v_table, const uint32_t* accepted, uint32_t position, uint32_t rows, const float* hidden, float* kept);

// ---- attention with a host-known schedule (attention.hip), used by the block graph of plan.hip --------
int qkv_attention_scheduled(void* stream, const float* q_raw, const float* k_raw, const float* v_raw, uint32_t planes,
                            uint64_t q_plane_stride, uint64_t k_plane_stride, uint64_t v_plane_stride, const float* q_norm,
                            const float* k_norm, const float* rope_table, float eps, const void* ring_k, const void* ring_v,
                            void* priv_k, void* priv_v, const uint32_t* schedule, const uint32_t* ancestors,
                            const uint32_t* host_schedule, const uint32_t* host_amask, float* out, float* out_sums,
                            float* partial_out, float* partial_ml, uint32_t rows, uint32_t max_tokens, uint32_t ring_mask,
                            uint32_t q_heads, uint32_t kv_heads, uint32_t head_dim, float scale, uint32_t* status);

// ---- typed loads at the alignment a GGUF block stream guarantees ------------
struct __attribute__((packed, aligned(4))) U4a4 { uint32_t x, y, z, w; };
struct __attribute__((packed, aligned(2))) U4a2 { uint32_t x, y, z, w; };
struct __attribute__((packed, aligned(2))) U2a2 { uint32_t x, y; };
struct __attribute__((packed, aligned(4))) F4a4 { float x, y, z, w; };
struct __attribute__((packed, aligned(4))) F2a4 { float x, y; };

__device__ __forceinline__ uint4 ld16_a4(const uint8_t* p) {
    const U4a4 t = *reinterpret_cast<const U4a4*>(p);
    return make_uint4(t.x, t.y, t.z, t.w);
}
__device__ __forceinline__ uint4 ld16_a2(const uint8_t* p) {
    const U4a2 t = *reinterpret_cast<const U4a2*>(p);
    return make_uint4(t.x, t.y, t.z, t.w);
}
__device__ __forceinline__ uint2 ld8_a2(const uint8_t* p) {
    const U2a2 t = *reinterpret_cast<const U2a2*>(p);
    return make_uint2(t.x, t.y);
}
__device__ __forceinline__ float4 ldf4_a4(const float* p) {
    const F4a4 t = *reinterpret_cast<const F4a4*>(p);
    return make_float4(t.x, t.y, t.z, t.w);
}
__device__ __forceinline__ uint32_t ld_u16(const uint8_t* p) { return *reinterpret_cast<const uint16_t*>(p); }

// fp16 bits -> fp32, exact (IEEE widening, subnormals included)
__device__ __forceinline__ float h2f(uint32_t bits) {
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<unsigned short>(bits)));
}

// Hides a value from the optimiser so that a following (v >> 8k) & 0xFF selects
// v_cvt_f32_ubyteK instead of being re-derived from the unmasked source.
__device__ __forceinline__ uint32_t opaque(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}
__device__ __forceinline__ float ub0(uint32_t v) { return static_cast<float>(v & 0xFFu); }
__device__ __forceinline__ float ub1(uint32_t v) { return static_cast<float>((v >> 8) & 0xFFu); }
__device__ __forceinline__ float ub2(uint32_t v) { return static_cast<float>((v >> 16) & 0xFFu); }
__device__ __forceinline__ float ub3(uint32_t v) { return static_cast<float>(v >> 24); }
__device__ __forceinline__ float sb0(uint32_t v) { return static_cast<float>(static_cast<int8_t>(v)); }
__device__ __forceinline__ float sb1(uint32_t v) { return static_cast<float>(static_cast<int8_t>(v >> 8)); }
__device__ __forceinline__ float sb2(uint32_t v) { return static_cast<float>(static_cast<int8_t>(v >> 16)); }
__device__ __forceinline__ float sb3(uint32_t v) { return static_cast<float>(static_cast<int8_t>(v >> 24)); }

// Sums and maxima over the 16 lanes of a row on the vector unit's lane-crossing modifiers (two quad permutations,
// then the mirror of 8 and of 16 lanes: every lane ends with the row's total), and over the wave with two more
// steps that swap neighbouring rows and halves of the wave.  A shuffle through the LDS crossbar would cost a wave that is
// alone on its SIMD more than a hundred cycles, and the reductions sit in dependent chains; every lane of the wave must be
// active.
template <int CTRL>
__device__ __forceinline__ float lane_cross(float v) {   // a lane outside the modifier's reach reads 0
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float row16_sum(float v) {
    v += lane_cross<0xB1>(v);    // quad_perm [1,0,3,2]
    v += lane_cross<0x4E>(v);    // quad_perm [2,3,0,1]
    v += lane_cross<0x141>(v);   // row_half_mirror
    v += lane_cross<0x140>(v);   // row_mirror
    return v;
}
// the values of this lane's row and of the row beside it (xor 16 lanes), the even row's first; the same for the wave's halves
struct Both { uint32_t a, b; };
__device__ __forceinline__ Both rows_beside(uint32_t v) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return {r[0], r[1]};
}
__device__ __forceinline__ Both halves_beside(uint32_t v) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return {r[0], r[1]};
}
__device__ __forceinline__ float both_sum(Both p) { return __uint_as_float(p.a) + __uint_as_float(p.b); }
__device__ __forceinline__ float both_max(Both p) { return fmaxf(__uint_as_float(p.a), __uint_as_float(p.b)); }
__device__ __forceinline__ float row16_max(float v) {
    v = fmaxf(v, lane_cross<0xB1>(v));
    v = fmaxf(v, lane_cross<0x4E>(v));
    v = fmaxf(v, lane_cross<0x141>(v));
    v = fmaxf(v, lane_cross<0x140>(v));
    return v;
}
// Inclusive prefix sum over the 64 lanes, the same way: four shifts inside the rows of 16 (a lane past the row's
// start reads 0), then lane 15's total into the next row and lane 31's into the upper half.
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t lane_cross_u32(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, ROWS, 0xF, ROWS == 0xF));
}
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v) {
    v += lane_cross_u32<0x111, 0xF>(v);   // row_shr:1
    v += lane_cross_u32<0x112, 0xF>(v);   // row_shr:2
    v += lane_cross_u32<0x114, 0xF>(v);   // row_shr:4
    v += lane_cross_u32<0x118, 0xF>(v);   // row_shr:8
    v += lane_cross_u32<0x142, 0xA>(v);   // row_bcast:15 into rows 1 and 3
    v += lane_cross_u32<0x143, 0xC>(v);   // row_bcast:31 into rows 2 and 3
    return v;
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    v = max(v, lane_cross_u32<0xB1, 0xF>(v));
    v = max(v, lane_cross_u32<0x4E, 0xF>(v));
    v = max(v, lane_cross_u32<0x141, 0xF>(v));
    v = max(v, lane_cross_u32<0x140, 0xF>(v));
    const Both rows = rows_beside(v);
    const Both halves = halves_beside(max(rows.a, rows.b));
    return max(halves.a, halves.b);
}

__device__ __forceinline__ float wave_sum(float v) {
    v = both_sum(rows_beside(__float_as_uint(row16_sum(v))));
    return both_sum(halves_beside(__float_as_uint(v)));
}
__device__ __forceinline__ float wave_max(float v) {
    v = both_max(rows_beside(__float_as_uint(row16_max(v))));
    return both_max(halves_beside(__float_as_uint(v)));
}

// A workgroup barrier for data that moves through LDS: it waits for this wave's LDS operations only.  (__syncthreads() also
// waits for every load and store to memory under way: for operands of later steps that were requested ahead, and for results on
// their way out, a trip to memory in the middle of a chain.)  What waves exchange through memory needs the other.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Sum of one word of each of `count` waves in LDS, `stride` words apart, in wave order.  All of up to MOST words are read ahead of the
// first add: a loop over a count known at run time waits for the words it is left with (up to seven) one after the other, 0.04 us
// each at the end of a launch.  MOST words have to lie there; -0 leaves a sum as it is.
template <int MOST>
__device__ __forceinline__ float sum_of_waves(const float* at, uint32_t stride, uint32_t count) {
    float v[MOST];
#pragma unroll
    for (int w = 0; w < MOST; ++w) v[w] = at[w * stride];
    float t = v[0];
#pragma unroll
    for (int w = 1; w < MOST; ++w) t += uint32_t(w) < count ? v[w] : -0.f;
    return t;
}

// 1 / sqrt(mean + eps) of a sum of squares, per_width = 1 / width.  The root's reciprocal (an ulp) and one step of Newton's: no
// further off than a division, a root and a division, which are 40 instructions behind each other where a norm waits for them.
// The instruction takes a denormal for zero; a row of zeros with an epsilon as small as that goes 2^24 times as large, beside the other.
// (A value meets this factor ahead of its gamma: the row's values by it are at most the root of its width, where a value times a gamma can
// pass either end of the floats.)
__device__ __forceinline__ float inverse_rms(float sum, float per_width, float eps) {
    const float mean = fmaf(sum, per_width, eps);
    const float y = mean < 0x1p-126f ? __builtin_amdgcn_rsqf(mean * 0x1p24f) * 0x1p12f : __builtin_amdgcn_rsqf(mean);
    const float better = fmaf(0.5f * y, fmaf(-(mean * y), y, 1.0f), y);
    return mean == INFINITY ? 0.f : better;
}

// Sum of `planes` partial planes in plane order; loads are issued four at a time so that the
// adds, not the memory latency, form the dependent chain.
__device__ __forceinline__ float load_planes(const float* p, uint32_t planes, size_t plane_stride) {
    float v = p[0];
    uint32_t s = 1;
    for (; s + 4 <= planes; s += 4) {
        const float a = p[s * plane_stride], b = p[(s + 1) * plane_stride], c = p[(s + 2) * plane_stride],
                    d = p[(s + 3) * plane_stride];
        v += a; v += b; v += c; v += d;
    }
    for (; s < planes; ++s) v += p[s * plane_stride];
    return v;
}

// Reduces NV per-lane values across the 64 lanes with NV-1 + (6 - log2 NV) exchanges
// instead of 6*NV: at each level the upper half-wave keeps one half of the values and
// the lower half-wave the other.  Afterwards v[0] on lane l holds the wave total of
// value index l >> (6 - log2 NV); the summation order is fixed, so results repeat.
template <int NV>
__device__ __forceinline__ void wave_reduce_multi(float (&v)[NV], int lane) {
    static_assert(NV >= 1 && NV <= 64 && (NV & (NV - 1)) == 0, "NV must be a power of two");
    int stride = 32;
#pragma unroll
    for (int m = NV; m > 1; m >>= 1) {
        const int half = m >> 1;
        const bool upper = (lane & stride) != 0;
#pragma unroll
        for (int i = 0; i < half; ++i) {
            const float send = upper ? v[i] : v[i + half];
            const float keep = upper ? v[i + half] : v[i];
            v[i] = keep + __shfl_xor(send, stride, kWave);
        }
        stride >>= 1;
    }
#pragma unroll
    for (; stride > 0; stride >>= 1) v[0] += __shfl_xor(v[0], stride, kWave);
}

template <int NV>
__device__ __forceinline__ constexpr int reduce_multi_shift() {
    int s = 6, n = NV;
    while (n > 1) { n >>= 1; --s; }
    return s;
}

// cos and sin of the NeoX rotation of (position, pair)
__device__ __forceinline__ void rope_sincos(uint32_t position, uint32_t pair, uint32_t rope_dim, float base,
                                            float scale, float& c, float& s) {
    // angle in double, as the CPU operator forms it (rope.cpp:109-117), times the layer's frequency scale
    const double exponent = static_cast<double>(2u * pair) / static_cast<double>(rope_dim);
    const double angle = static_cast<double>(position) / pow(static_cast<double>(base), exponent)
        * static_cast<double>(scale);
    c = static_cast<float>(cos(angle));
    s = static_cast<float>(sin(angle));
}

}  // namespace guffin
