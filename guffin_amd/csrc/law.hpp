// The compact proposal law: what draft_law_kernel (sampling.hip) makes of a selection's record, and the selection that decides a law
// (head.hip) of its keys, in the workgroup that finishes it.  Reference: src/engine/gemma3_draft.mm:191-294, 995-1070.
#pragma once
#include "common.hpp"

namespace guffin {

constexpr uint64_t kMassTotal = uint64_t{1} << 32;
constexpr uint32_t kLawFull = 0xFFFFFFFFu;  // DraftLaw::count of a law held as a full-vocabulary table
constexpr uint32_t kMaxTopK = 256;

struct DraftLaw { uint32_t count; uint32_t pad; uint32_t ids[256]; uint64_t cdf[257]; };
struct SamplerOptions { float temperature; uint32_t top_k; float top_p; float min_p; float repetition_penalty; };
struct StepDraws { uint32_t word; uint32_t pad; double u_accept, u_residual, u_next; };
// where a law goes and what it is made with
struct LawCall {
    SamplerOptions opt;
    uint64_t seed, step;
    const StepDraws* injected;   // or null
    DraftLaw* law;
    uint32_t *proposal, *status;
    uint32_t* full_error;        // not null: the full-vocabulary kernels follow, guarded by law->count; a support of more than 256 ties then
                                 // hands over to them instead of failing
    uint32_t whole;              // the law is new memory, what it does not use becomes zero
};

// ---- Philox4x32-10 ----------------------------------------------------------------------
__device__ __forceinline__ void philox(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0, uint32_t k1,
                                       uint32_t (&out)[4]) {
#pragma unroll
    for (int round = 0; round < 10; ++round) {
        const uint64_t p0 = uint64_t{0xD2511F53u} * c0, p1 = uint64_t{0xCD9E8D57u} * c2;
        const uint32_t n0 = static_cast<uint32_t>(p1 >> 32) ^ c1 ^ k0, n1 = static_cast<uint32_t>(p1);
        const uint32_t n2 = static_cast<uint32_t>(p0 >> 32) ^ c3 ^ k1, n3 = static_cast<uint32_t>(p0);
        c0 = n0; c1 = n1; c2 = n2; c3 = n3;
        k0 += 0x9E3779B9u; k1 += 0xBB67AE85u;
    }
    out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}
__device__ __forceinline__ double unit_double(uint32_t hi, uint32_t lo) {
    return static_cast<double>(((uint64_t{hi} << 32) | lo) >> 11) * 0x1.0p-53;
}
// word, u_accept from counter (step, 0); u_residual, u_next from counter (step, 1)
__device__ __forceinline__ StepDraws step_draws(uint64_t seed, uint64_t step) {
    uint32_t a[4], b[4];
    const uint32_t k0 = static_cast<uint32_t>(seed), k1 = static_cast<uint32_t>(seed >> 32);
    const uint32_t s0 = static_cast<uint32_t>(step), s1 = static_cast<uint32_t>(step >> 32);
    philox(s0, s1, 0, 0, k0, k1, a);
    philox(s0, s1, 1, 0, k0, k1, b);
    StepDraws d;
    d.word = a[0]; d.pad = 0;
    d.u_accept = unit_double(a[1], a[2]);
    d.u_residual = unit_double(b[0], b[1]);
    d.u_next = unit_double(b[2], b[3]);
    return d;
}

// exp for the law's f32 weights from IEEE-exact operations only (fma, floor, exponent
// scaling), so the integer CDF is reproducible bit for bit on any conforming machine.
__device__ __forceinline__ float law_exp(float x) {
    if (!(x > -86.0f)) return x != x ? x : 0.0f;
    if (x > 88.0f) return INFINITY;
    const float kf = floorf(fmaf(x, 1.44269502162933349609375f, 0.5f));
    float r = fmaf(kf, -0.693145751953125f, x);
    r = fmaf(kf, -1.428606765330187045037746429443359375e-06f, r);
    float p = 1.0f / 5040.0f;
    p = fmaf(p, r, 1.0f / 720.0f);
    p = fmaf(p, r, 1.0f / 120.0f);
    p = fmaf(p, r, 1.0f / 24.0f);
    p = fmaf(p, r, 1.0f / 6.0f);
    p = fmaf(p, r, 0.5f);
    p = fmaf(p, r, 1.0f);
    p = fmaf(p, r, 1.0f);
    const int k = static_cast<int>(kf);
    return __fmul_rn(p, __uint_as_float(static_cast<uint32_t>(k + 127) << 23));
}

__device__ __forceinline__ bool options_valid(const SamplerOptions& o) {
    return isfinite(o.temperature) && o.temperature >= 0.f && o.top_k >= 1 && o.top_k <= kMaxTopK
        && isfinite(o.top_p) && o.top_p > 0.f && o.top_p <= 1.f && isfinite(o.min_p) && o.min_p >= 0.f
        && o.min_p <= 1.f && isfinite(o.repetition_penalty) && o.repetition_penalty > 0.f;
}

// Sums whose order matters, one lane's work over LDS: eight operands are read before the first of their adds, so the chain is
// one of additions, not of LDS reads.  v holds zeros from n up to the next multiple of eight: adding them changes nothing.
// running[i] = v[0] + ... + v[i]; returns the total
template <typename T>
__device__ __forceinline__ T ordered_sums(const T* __restrict__ v, uint32_t n, T* __restrict__ running) {
    T sum = T(0), x[8], next[8];
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) x[k] = v[k];
    for (uint32_t i0 = 0; i0 < n; i0 += 8) {
        const uint32_t ahead = i0 + 8 < n ? i0 + 8 : i0;
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) next[k] = v[ahead + k];
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) { sum += x[k]; x[k] = sum; }
        if (running)
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) running[i0 + k] = x[k];
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) x[k] = next[k];
    }
    return sum;
}

// The smallest index of `hit` threads into *to (LDS): a wave finds its own and one lane enters it.  (Every hit's atomicMin on the one word is
// served lane by lane: 2.0 us of a law's 6.7 for 200 of them, 1.8 of an acceptance's 11.8.)
__device__ __forceinline__ void note_first(bool hit, uint32_t index, uint32_t* to) {
    const uint64_t hits = __ballot(hit);
    if (hits && (threadIdx.x & 63u) == 0) atomicMin(to, index + static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(hits))) - 1u);
}

// The law from the best 257 scores (sorted, score = logit / T).  The 256 threads of a workgroup (those that are left of a
// larger one) call it: thread t with entry t, counted or not, all with the record's count and status and entry 256's score.
__device__ __forceinline__ void compact_law(const LawCall& call, uint32_t avail, uint32_t raised, uint32_t found_token, float found_logit, float more) {
    const SamplerOptions& opt = call.opt;
    const StepDraws* const injected = call.injected;
    DraftLaw* const law = call.law;
    uint32_t *const proposal = call.proposal, *const status = call.status, *const full_error = call.full_error;
    const uint64_t seed = call.seed, step = call.step;
    const bool whole = call.whole != 0;
    __shared__ uint64_t keys[256];
    __shared__ float score[256], weight[256], running[256];
    __shared__ uint64_t edge[257];
    __shared__ uint32_t ids[256];
    __shared__ uint32_t s_first, s_bad, s_chosen, s_word;
    const uint32_t t = threadIdx.x;
    const bool usable = options_valid(opt) && opt.temperature > 0.f && opt.top_k <= 64 && avail >= 1;
    const uint32_t k = usable ? (opt.top_k < avail ? opt.top_k : avail) : 1u;
    const float my_logit = t < avail ? found_logit : -INFINITY;
    const uint32_t my_token = t < avail ? found_token : 0u;
    if (t == 0) { s_first = 256u; s_bad = 0; s_chosen = 0xFFFFFFFFu; }
    score[t] = my_logit;
    __syncthreads();
    const float cutoff = usable ? score[k - 1] : 0.f, first_logit = usable ? score[0] : 0.f;
    // entries are sorted by (score desc, token asc): the support is a prefix, its length the first
    // entry that is below the cutoff or -inf
    note_first(!(t < avail && !(my_logit < cutoff) && my_logit != -INFINITY), t, &s_first);
    __syncthreads();
    uint32_t st = 0, n = 0;   // every thread's own, all alike
    if (!usable) st = GUFFIN_STATUS_LAW_INVALID;
    if (raised & GUFFIN_STATUS_NONFINITE) st = GUFFIN_STATUS_LAW_INVALID | GUFFIN_STATUS_NONFINITE;
    if (!st) {
        n = s_first;
        if (n == 256u && avail > 256u) {   // all 256 are in: a 257th eligible entry overflows the compact law
            if (!(more < cutoff) && more != -INFINITY) n = 257u;
        }
        if (n == 0) st = GUFFIN_STATUS_LAW_INVALID;  // nothing eligible
        if (n > 256) st = GUFFIN_STATUS_LAW_INVALID | 32u;  // support overflow: needs the full-vocabulary law
    }
    if (t == 0) {
        if (full_error) *full_error = 0;
        if (st == (GUFFIN_STATUS_LAW_INVALID | 32u) && full_error) { law->count = kLawFull; *proposal = 0xFFFFFFFFu; }
        else if (st) { atomicOr(status, st); law->count = 0; *proposal = 0xFFFFFFFFu; }
    }
    if (st) {
        if (whole) { law->ids[t] = 0; law->cdf[t] = 0; if (t == 0) { law->pad = 0; law->cdf[256] = 0; } }
        return;
    }
    // An entry's weight against the best one, which the filters always leave: the weights of the law are these, those of what is
    // filtered zero.
    const float own_weight = t < n ? law_exp(my_logit - first_logit) : 0.f;
    weight[t] = own_weight;
    __syncthreads();
    if (t == 64) s_word = injected ? injected->word : step_draws(seed, step).word;   // another wave's, beside the sums
    if (t == 0) {  // descending-tail top-p / min-p in the reference's sequential order
        // the tail sums from the last entry down; the last of them, in slot 0 (always kept), is the total: the
        // same adds in the same order
        float tail = 0.f, x[8], next[8];
        const uint32_t top = (n + 7) & ~7u;   // past the end zeros
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) x[k] = weight[top - 1 - k];
        for (uint32_t j0 = top; j0 > 0; j0 -= 8) {   // eight reads ahead of their adds
            const uint32_t ahead = j0 > 8 ? j0 - 8 : 8;
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) next[k] = weight[ahead - 1 - k];
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) { tail = __fadd_rn(tail, x[k]); x[k] = tail; }
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) { running[j0 - 1 - k] = x[k]; x[k] = next[k]; }
        }
    }
    __syncthreads();
    const bool keep = t == 0 || ((opt.top_p >= 1.0f || __fdiv_rn(running[t], running[0]) > __fsub_rn(1.0f, opt.top_p))
                                 && (opt.min_p <= 0.0f || own_weight >= opt.min_p));
    // ascending token id; the weight rides in the low half of the key
    keys[t] = t < n ? (uint64_t(my_token) << 32) | __float_as_uint(keep ? own_weight : 0.f) : ~uint64_t{0};
    __syncthreads();
    {   // places: the keys that go before one's own, counted by one, two or four neighbouring lanes
        const uint32_t part_bits = n <= 64 ? 2 : n <= 128 ? 1 : 0, i = t >> part_bits, part = t & ((1u << part_bits) - 1);
        const uint64_t mine = keys[i];
        uint32_t rank = 0;
#pragma unroll 8
        for (uint32_t j = part; j < n; j += 1u << part_bits) rank += keys[j] < mine;
        if (part_bits >= 1) rank += lane_cross_u32<0xB1, 0xF>(rank);
        if (part_bits >= 2) rank += lane_cross_u32<0x4E, 0xF>(rank);
        if (i < n && part == 0) {   // (weight: zeros behind the last entry as before)
            ids[rank] = static_cast<uint32_t>(mine >> 32);
            weight[rank] = __uint_as_float(static_cast<uint32_t>(mine));
        }
    }
    __syncthreads();
    if (t == 0) {   // the f32 running sums in token order; the quotients and edges are per-lane work
        ordered_sums(weight, n, running);
        edge[0] = 0;
    }
    __syncthreads();
    const float total = running[n - 1];
    const bool total_ok = total > 0.f && isfinite(total);
    uint64_t next = 0;
    if (t < n) {
        float scaled = __fmul_rn(__fdiv_rn(running[t], total), 4294967296.0f);
        scaled = fminf(fmaxf(scaled, 0.0f), 4294967296.0f);
        next = static_cast<uint64_t>(scaled);
        edge[t + 1] = next;
    }
    __syncthreads();
    if (t < n) {
        const uint64_t last = edge[t];
        if (next < last || next > kMassTotal || (t == n - 1 && next != kMassTotal)) s_bad = 1;
        if (uint64_t(s_word) >= last && uint64_t(s_word) < next) s_chosen = ids[t];
        law->ids[t] = ids[t];
        law->cdf[t + 1] = next;
    } else if (whole) {
        law->ids[t] = 0;
        law->cdf[t + 1] = 0;
    }
    __syncthreads();
    if (t == 0) {
        law->count = n; law->pad = 0; law->cdf[0] = 0;
        const bool bad = !total_ok || s_bad;
        if (bad) atomicOr(status, GUFFIN_STATUS_LAW_INVALID);
        *proposal = bad ? 0xFFFFFFFFu : s_chosen;
    }
}

// The selection of `retain` logits of one row that ends in a law (head.hip), for the vocabularies it covers.  workspace: as for
// guffin_hip_select_candidates of one row.
bool selection_makes_laws(uint32_t vocab, uint32_t retain);
int select_law(hipStream_t s, const float* logits, uint32_t vocab, uint32_t retain, uint32_t sure, void* workspace, const LawCall& law,
               bool suppressed_ok);

}  // namespace guffin
