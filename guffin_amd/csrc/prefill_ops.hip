// The operators between the GEMMs of a prefill pass (gfx950), each reading the k-slice planes the GEMM before left and
// writing the operand image the GEMM after reads (prefill_image.hpp), so that no activation crosses memory a second time:
//
//   first norm   rms(x)                                       reference: encode_rms_norm
//   qkv          head norms, NeoX rotation, fp16 narrowing, and the values of every visible token transposed for the
//                attention                                    gemma_target_runtime.cpp:88-133, metal_kernels.mm:2406-2486
//   joint        residual + rms(a), then rms of that          gemma_target_runtime.cpp:156-173, 201-213; the joint after the
//                attention also publishes the run's K/V       attention, when nobody reads the ring rows they replace
//   geglu        gelu_tanh(gate) * up                         metal_kernels.mm:1827-1843
#include "common.hpp"
#include "prefill_image.hpp"
#include "prefill_run.hpp"
#include "receipt.hpp"

namespace guffin {
namespace {

// scratch: 16 floats, nobody else's, and used once; waves: of the workgroup
__device__ __forceinline__ float block_total(float v, float* scratch, uint32_t waves) {
    v = wave_sum(v);
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) scratch[wv] = v;
    lds_barrier();
    return waves <= 8 ? sum_of_waves<8>(scratch, 1, waves) : sum_of_waves<16>(scratch, 1, waves);  // same order on every thread
}

// 8 consecutive floats of `planes` planes, summed in plane order; up to B planes are requested before the first add
template <int B>
__device__ __forceinline__ void sum_planes8(const float* p, uint32_t planes, size_t stride, float (&v)[8]) {
    for (uint32_t s0 = 0; s0 < planes; s0 += B) {
        float4 a[B], b[B];
#pragma unroll
        for (int s = 0; s < B; ++s)
            if (s0 + s < planes) {
                a[s] = *reinterpret_cast<const float4*>(p + (s0 + s) * stride);
                b[s] = *reinterpret_cast<const float4*>(p + (s0 + s) * stride + 4);
            }
#pragma unroll
        for (int s = 0; s < B; ++s)
            if (s0 + s < planes) {
                const float w[8] = {a[s].x, a[s].y, a[s].z, a[s].w, b[s].x, b[s].y, b[s].z, b[s].w};
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = s0 + s == 0 ? w[i] : v[i] + w[i];
            }
    }
}
__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
    const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void store8(float* p, const float (&v)[8]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
// the same where the caller's pointer may start at any word
__device__ __forceinline__ void load8_words(const float* p, float (&v)[8]) {
    const float4 a = ldf4_a4(p), b = ldf4_a4(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void store8_words(float* p, const float (&v)[8]) {
    *reinterpret_cast<F4a4*>(p) = F4a4 {v[0], v[1], v[2], v[3]};
    *reinterpret_cast<F4a4*>(p + 4) = F4a4 {v[4], v[5], v[6], v[7]};
}

// The row of a workgroup.  Eight rows of a record's k-slice share a 128-byte line of the image, and consecutive workgroups go to
// different XCDs: the eight go to one, whose L2 puts the line together.  (2048 x 3840: the joints 44.7 -> 32.0 and 50.1 -> 35.1 us, the
// first norm 34.4 -> 16.5; 333 rows 10.6 -> 10.0 and 10.3 -> 9.4.)
__device__ __forceinline__ uint32_t row_of(uint32_t b, uint32_t rows) {
    const uint32_t x = b & 7u, k = b >> 3;
    return b < (rows & ~63u) ? (k & ~7u) * 8 + x * 8 + (k & 7u) : b;
}

// one workgroup per row, a thread owns 8 consecutive columns
__global__ void __launch_bounds__(1024)
prefill_norm_kernel(const float* __restrict__ x, const float* __restrict__ gamma, uint8_t* __restrict__ image, uint32_t rows,
                    uint32_t width, float eps, uint32_t* __restrict__ status) {
    __shared__ __attribute__((aligned(16))) float scratch[16];
    const uint32_t r = row_of(blockIdx.x, rows), t = threadIdx.x;
    const bool active = t < width / 8;
    float v[8] = {}, g[8] = {};
    if (active) { load8(x + size_t(r) * width + 8 * t, v); load8_words(gamma + 8 * t, g); }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) ss = fmaf(v[i], v[i], ss);
    const float inv = inverse_rms(block_total(ss, scratch, (width + 511) / 512), 1.0f / static_cast<float>(width), eps);
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 8; ++i) { v[i] = v[i] * inv * g[i]; bad |= !isfinite(v[i]); }
    if (active) emit_image_values(v, t, r, image_layout(rows, width), image);
    if (bad && status) atomicOr(status, GUFFIN_STATUS_NONFINITE);
}

// Workgroups [0, rows): one row each.  The rest copy the run's fp16 K/V rows to their ring slots, 16 bytes per thread.
// B planes are requested at a time: a short run has up to 16 and few workgroups, and is bound by the trips (37 rows, 15 planes:
// 8.4 us by eights, 8.1 at once; 12 rows 8.0 and 7.5); THREADS: the widest row's.
template <int B, int THREADS>
__global__ void __launch_bounds__(THREADS)
prefill_joint_kernel(const float* __restrict__ x, const float* __restrict__ residual, const float* __restrict__ gamma_post,
                     const float* __restrict__ gamma_next, size_t plane_stride, uint32_t planes, uint32_t width, uint32_t rows, float eps,
                     float* __restrict__ out_residual, float* __restrict__ out_norm, uint8_t* __restrict__ image, RunRows run,
                     uint32_t* __restrict__ status) {
    if (blockIdx.x >= rows) {
        const uint64_t i = uint64_t(blockIdx.x - rows) * ((width + 511) / 512 * 64) + threadIdx.x;
        if (i >= uint64_t(rows - run.first_row) * run.row_vec) return;
        const uint32_t row = run.first_row + static_cast<uint32_t>(i / run.row_vec), c = static_cast<uint32_t>(i % run.row_vec);
        const size_t dst = size_t((run.position + row) & run.ring_mask) * run.row_vec + c;
        static_cast<U4a4*>(run.ring_k)[dst] = static_cast<const U4a4*>(run.run_k)[size_t(row) * run.row_vec + c];
        static_cast<U4a4*>(run.ring_v)[dst] = static_cast<const U4a4*>(run.run_v)[size_t(row) * run.row_vec + c];
        return;
    }
    __shared__ __attribute__((aligned(16))) float scratch[2][16];
    const uint32_t r = row_of(blockIdx.x, rows), t = threadIdx.x;
    const bool active = t < width / 8;
    const size_t at = size_t(r) * width + 8 * t;
    float v[8] = {}, gp[8] = {}, gn[8] = {}, res[8] = {};
    if (active) {
        load8_words(gamma_post + 8 * t, gp);
        load8(residual + at, res);
        load8_words(gamma_next + 8 * t, gn);
        sum_planes8<B>(x + at, planes, plane_stride, v);
    }
    // what only the stores need, asked for beside the operands (see rms_norm_add_norm_regs_kernel)
    asm volatile("" ::"s"(out_residual), "s"(out_norm), "s"(image), "s"(status));
    const float per_width = 1.0f / static_cast<float>(width);
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) ss = fmaf(v[i], v[i], ss);
    float inv = inverse_rms(block_total(ss, scratch[0], (width + 511) / 512), per_width, eps);
    ss = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        v[i] = fmaf(v[i] * inv, gp[i], res[i]);
        ss = fmaf(v[i], v[i], ss);
    }
    inv = inverse_rms(block_total(ss, scratch[1], (width + 511) / 512), per_width, eps);
    if (active) store8(out_residual + at, v);
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        bad |= !isfinite(v[i]);
        v[i] = v[i] * inv * gn[i];
    }
    if (active) {
        if (image) emit_image_values(v, t, r, image_layout(rows, width), image);
        else store8_words(out_norm + at, v);
    }
    if (bad && status) atomicOr(status, GUFFIN_STATUS_NONFINITE);
}

// grid (width / 256, ceil(rows / 8)): 8 rows of 256 columns, a thread 8 of them; the rows' operand pieces leave together, whole
// 128-byte lines.  (With every thread's 16 bytes written where they belong, into lines shared by workgroups of several XCDs,
// 2048 x 15360 took 145 us instead of 65.)
__global__ void __launch_bounds__(256)
prefill_geglu_kernel(const float* __restrict__ gate, const float* __restrict__ up, uint32_t planes, size_t plane_stride,
                     uint8_t* __restrict__ image, uint32_t rows, uint32_t width) {
    __shared__ __attribute__((aligned(16))) uint8_t records[8 * 2048];
    const ImageLayout L = image_layout(rows, width);
    const uint32_t t0 = blockIdx.x * 32, c = threadIdx.x & 31, valid = min(32u, width / 8 - t0), row = blockIdx.y * 8 + (threadIdx.x >> 5);
    if (row < rows && c < valid) {
        float g[8], u[8];
        const size_t at = size_t(row) * width + 8 * (t0 + c);
        sum_planes8<4>(gate + at, planes, plane_stride, g);
        sum_planes8<4>(up + at, planes, plane_stride, u);
#pragma unroll
        for (int k = 0; k < 8; ++k) g[k] = geglu_value(g[k], u[k]);
        emit_image_values(g, t0 + c, row, L, image, records);
    }
    lds_barrier();   // what went to memory already is read by nobody here
    // 8 rows of a record's k-slice are 128 contiguous bytes; padding rows' places hold what they held: nobody looks at them
    const uint32_t tile = blockIdx.y >> 1, half = (blockIdx.y & 1) * 128;
    for (uint32_t k = threadIdx.x; k < (valid / 4) * 64; k += 256) {
        const uint32_t g = k >> 6, at = ((k >> 3) & 7) * 256 + half + (k & 7) * 16;   // hi or lo and k-slice, row
        *reinterpret_cast<uint4*>(image + (size_t(t0 / 4 + g) * (L.mpad / 16) + tile) * 2048 + at) = *reinterpret_cast<const uint4*>(records + g * 2048 + at);
    }
}

// Workgroups [0, head_groups): sixteen (row, query or key head) pairs, a wave each.  The rest: 32 visible tokens of one KV
// head's values each, from the ring or (the run's own, narrowed and kept on the way) from the planes, written transposed.
// Bound by its trips in a short run, so a thread has eight elements of one token and asks for eight planes at a time (with four
// tokens one behind the other, by fours, 15 planes were sixteen trips: 12 rows at position 100 9.1 us, 37 at 1500 11.8, 2048 at 0 30.0; now
// 6.4, 7.5 and 29.0).
constexpr uint32_t kQkvThreads = 1024;
__global__ void __launch_bounds__(kQkvThreads)
prefill_qkv_kernel(const float* __restrict__ q_planes, const float* __restrict__ k_planes, const float* __restrict__ v_planes,
                   const uint16_t* __restrict__ ring_v, uint32_t rows, uint32_t head_groups, uint32_t planes, uint32_t kv_heads, uint32_t position,
                   uint32_t base32, QkvRun a) {
    // (the struct holds them as well, but arrives a trip later: see the kernels of gemv_packed.hip)
    constexpr uint32_t HD = 256, PITCH = HD + 8;
    __shared__ __attribute__((aligned(16))) uint16_t tile[32][PITCH];
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    bool bad = false;
    if (blockIdx.x < head_groups) {
        const uint32_t per_row = a.q_heads + kv_heads, p = blockIdx.x * (kQkvThreads / 64) + wv;
        if (p >= rows * per_row) return;
        const uint32_t r = p / per_row, h = p % per_row;
        const bool is_q = h < a.q_heads;
        const uint32_t hh = is_q ? h : h - a.q_heads, heads = is_q ? a.q_heads : kv_heads;
        const size_t off = (size_t(r) * heads + hh) * HD;
        const size_t stride = size_t(rows) * heads * HD;
        const float* src = (is_q ? q_planes : k_planes) + off;
        const float* gamma = is_q ? a.q_norm : a.k_norm;
        // lane: columns 2 lane, 2 lane + 1 of either half, the pairs that rotate together
        const float4 rot = reinterpret_cast<const float4*>(a.rope_table)[size_t(r) * (HD / 4) + lane];   // cos, sin of two pairs
        float2 g0 = make_float2(1.f, 1.f), g1 = g0;   // null: no head norm
        if (gamma) {
            g0 = make_float2(gamma[2 * lane], gamma[2 * lane + 1]);
            g1 = make_float2(gamma[HD / 2 + 2 * lane], gamma[HD / 2 + 2 * lane + 1]);
        }
        float v[4];
        for (uint32_t s0 = 0; s0 < planes; s0 += 8) {
            float2 x[8], y[8];
#pragma unroll
            for (int s = 0; s < 8; ++s)
                if (s0 + s < planes) {
                    x[s] = *reinterpret_cast<const float2*>(src + (s0 + s) * stride + 2 * lane);
                    y[s] = *reinterpret_cast<const float2*>(src + (s0 + s) * stride + HD / 2 + 2 * lane);
                }
#pragma unroll
            for (int s = 0; s < 8; ++s)
                if (s0 + s < planes) {
                    if (s0 + s == 0) { v[0] = x[s].x; v[1] = x[s].y; v[2] = y[s].x; v[3] = y[s].y; }
                    else { v[0] += x[s].x; v[1] += x[s].y; v[2] += y[s].x; v[3] += y[s].y; }
                }
        }
        float ss = fmaf(v[0], v[0], fmaf(v[1], v[1], fmaf(v[2], v[2], v[3] * v[3])));
        const float normed = inverse_rms(wave_sum(ss), 1.0f / HD, a.eps), inv = gamma ? normed : 1.f;
        v[0] = v[0] * inv * g0.x; v[1] = v[1] * inv * g0.y; v[2] = v[2] * inv * g1.x; v[3] = v[3] * inv * g1.y;
        const float o0 = __fsub_rn(__fmul_rn(v[0], rot.x), __fmul_rn(v[2], rot.y)), o1 = __fsub_rn(__fmul_rn(v[1], rot.z), __fmul_rn(v[3], rot.w));
        const float o2 = __fadd_rn(__fmul_rn(v[0], rot.y), __fmul_rn(v[2], rot.x)), o3 = __fadd_rn(__fmul_rn(v[1], rot.w), __fmul_rn(v[3], rot.z));
        if (is_q) {
            *reinterpret_cast<float2*>(a.q_out + off + 2 * lane) = make_float2(o0, o1);
            *reinterpret_cast<float2*>(a.q_out + off + HD / 2 + 2 * lane) = make_float2(o2, o3);
        } else {
            auto narrow = [&](float x, float y) {   // round to nearest even, after rotation
                const _Float16 h0 = static_cast<_Float16>(x), h1 = static_cast<_Float16>(y);
                bad |= !(isfinite(static_cast<float>(h0)) && isfinite(static_cast<float>(h1)));
                return uint32_t(__builtin_bit_cast(uint16_t, h0)) | (uint32_t(__builtin_bit_cast(uint16_t, h1)) << 16);
            };
            *reinterpret_cast<uint32_t*>(a.k_out + off + 2 * lane) = narrow(o0, o1);
            *reinterpret_cast<uint32_t*>(a.k_out + off + HD / 2 + 2 * lane) = narrow(o2, o3);
        }
    } else {
        const uint32_t w = blockIdx.x - head_groups, kvh = w % kv_heads, v0 = (w / kv_heads) * 32;
        const size_t width = size_t(kv_heads) * HD, stride = size_t(rows) * width;
        static_assert(kQkvThreads == 32 * (HD / 8), "a thread: eight elements of a token");
        {
            const uint32_t token = threadIdx.x / (HD / 8), d8 = threadIdx.x % (HD / 8), kp = base32 + v0 + token;
            uint4 val = make_uint4(0, 0, 0, 0);   // outside the visible range
            if (kp >= position && kp < position + rows) {
                const size_t off = size_t(kp - position) * width + kvh * HD + 8 * d8;
                float f[8];
                sum_planes8<8>(v_planes + off, planes, stride, f);
                uint32_t o[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const _Float16 h0 = static_cast<_Float16>(f[2 * i]), h1 = static_cast<_Float16>(f[2 * i + 1]);
                    bad |= !(isfinite(static_cast<float>(h0)) && isfinite(static_cast<float>(h1)));
                    o[i] = uint32_t(__builtin_bit_cast(uint16_t, h0)) | (uint32_t(__builtin_bit_cast(uint16_t, h1)) << 16);
                }
                val = make_uint4(o[0], o[1], o[2], o[3]);
                *reinterpret_cast<uint4*>(a.v_out + off) = val;
            } else if (kp >= a.first_visible && kp < position) {
                const U4a4 t = *reinterpret_cast<const U4a4*>(ring_v + size_t(kp & a.ring_mask) * width + kvh * HD + 8 * d8);
                val = make_uint4(t.x, t.y, t.z, t.w);
            }
            *reinterpret_cast<uint4*>(&tile[token][8 * d8]) = val;
        }
        lds_barrier();
        const uint32_t dim = threadIdx.x >> 2, lg = threadIdx.x & 3;   // four threads: a dimension's 32 tokens
        uint32_t o[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) o[t] = uint32_t(tile[value_token(lg, 2 * t)][dim]) | (uint32_t(tile[value_token(lg, 2 * t + 1)][dim]) << 16);
        *reinterpret_cast<uint4*>(a.vt + size_t(kvh) * HD * a.T + size_t(v0) * HD + 32 * dim + 8 * lg) = make_uint4(o[0], o[1], o[2], o[3]);
    }
    if (bad && a.status) atomicOr(a.status, GUFFIN_STATUS_KV_NONFINITE);
}

uint32_t row_threads(uint32_t width) { return (width / 8 + 63) / 64 * 64; }

}  // namespace

int prefill_norm(hipStream_t s, const float* x, const float* gamma, uint8_t* image, uint32_t rows, uint32_t width, float eps, uint32_t* status) {
    launch(prefill_norm_kernel, dim3(rows), dim3(row_threads(width)), 0, s, x, gamma, image, rows, width, eps, status);
    return check_launch("prefill_norm");
}

int prefill_joint(hipStream_t s, const float* x, uint32_t planes, const float* gamma_post, const float* residual, float* out_residual,
                  const float* gamma_next, float* out_norm, uint8_t* image, uint32_t rows, uint32_t width, float eps, const RunRows& run,
                  uint32_t* status) {
    const uint32_t threads = row_threads(width);
    const uint64_t copies = run.run_k ? uint64_t(rows - run.first_row) * run.row_vec : 0;
    const dim3 grid(rows + static_cast<uint32_t>((copies + threads - 1) / threads));
#define GUFFIN_JOINT(...) launch((prefill_joint_kernel<__VA_ARGS__>), grid, dim3(threads), 0, s, x, residual, gamma_post, gamma_next, size_t(rows) * width, \
                                 planes, width, rows, eps, out_residual, out_norm, image, run, status)
    if (planes > 8 && threads <= 512) GUFFIN_JOINT(16, 512); else GUFFIN_JOINT(8, 1024);
#undef GUFFIN_JOINT
    return check_launch("prefill_joint");
}

int prefill_geglu(hipStream_t s, const float* gate, const float* up, uint32_t planes, uint8_t* image, uint32_t rows, uint32_t width) {
    launch(prefill_geglu_kernel, dim3((width + 255) / 256, (rows + 7) / 8), dim3(256), 0, s, gate, up, planes, size_t(rows) * width, image, rows, width);
    return check_launch("prefill_geglu");
}

int prefill_qkv(hipStream_t s, QkvRun a) {
    a.head_groups = (a.rows * (a.q_heads + a.kv_heads) + kQkvThreads / 64 - 1) / (kQkvThreads / 64);
    launch(prefill_qkv_kernel, dim3(a.head_groups + (a.T / 32) * a.kv_heads), dim3(kQkvThreads), 0, s, a.q_planes,
           a.k_planes, a.v_planes, a.ring_v, a.rows, a.head_groups, a.planes, a.kv_heads, a.position, a.base32, a);
    return check_launch("prefill_qkv");
}

}  // namespace guffin
