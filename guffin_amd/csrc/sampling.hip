// Proposal law of the drafter and lossless accept / residual sampling (gfx950).
//
// Reference behaviour:
//   compact proposal law (integer 2^32-mass CDF)   src/engine/gemma3_draft.mm:191-294, 995-1070
//   gather of q on p's support                     src/engine/gemma3_draft.mm:1528-1581
//   target law p (all double)                      src/engine/sampling.cpp:394-499
//   validation / Neumaier total                    src/engine/sampling.cpp:117-158
//   accept min(1,p/q), residual max(p-q,0)         src/engine/sampling.cpp:561-656
//   inverse-CDF selections                         src/engine/sampling.cpp:247-257, 501-514
//   draw consumption order                         src/engine/sampling.cpp:896-934
// The reference evaluates the target law and the accept test on the host from a compact
// read-back; here both run on the device in the same fp64 operation order (sequential sums
// are taken by one lane in the reference's order), so decisions depend only on the inputs and
// the draws.  Draws come from Philox4x32-10 keyed (seed, step) unless injected.
#include "common.hpp"
#include "law.hpp"

namespace guffin {
namespace {

constexpr uint32_t kMaxCandidates = 384, kHistoryCap = 64;

struct Candidates { uint32_t count; uint32_t status; struct { uint32_t token; float logit; } values[384]; };
struct SpecResult {
    uint32_t accepted, token, next_root, status;
    double acceptance_probability, residual_total;
    uint32_t residual_count, proposal;
};

// bitonic sort of n (power of two) 64-bit keys in LDS, ascending or descending
__device__ __forceinline__ void bitonic(uint64_t* keys, uint32_t n, bool desc) {
    for (uint32_t width = 2; width <= n; width <<= 1)
        for (uint32_t stride = width >> 1; stride > 0; stride >>= 1) {
            __syncthreads();
            for (uint32_t i = threadIdx.x; i < n / 2; i += blockDim.x) {
                const uint32_t lo = 2 * i - (i & (stride - 1)), hi = lo + stride;
                const bool first_dir = (lo & width) == 0;
                const uint64_t a = keys[lo], b = keys[hi];
                if (((a < b) == desc) == first_dir) { keys[lo] = b; keys[hi] = a; }
            }
        }
    __syncthreads();
}

__device__ __forceinline__ uint64_t score_key(float score, uint32_t token) {
    const uint32_t b = __float_as_uint(score + 0.0f);
    const uint32_t ordered = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    return (uint64_t(ordered) << 32) | (0xFFFFFFFFu - token);
}

// =========================================================================================
// Compact proposal law from the best 257 scores (sorted, score = logit / T)
// =========================================================================================
__global__ void __launch_bounds__(256)
draft_law_kernel(const Candidates* __restrict__ top, LawCall call) {
    // the record (always whole in memory) comes in one trip: every thread fetches its own entry, counted or not
    const uint32_t t = threadIdx.x;
    compact_law(call, top->count, top->status, top->values[t].token, top->values[t].logit, top->values[256].logit);
}

// =========================================================================================
// Full-vocabulary proposal law: the drafter's law when the compact support does not apply
// (top_k > 64, greedy drafting, or more than 256 tokens tied into the support).
// src/engine/gemma3_draft.mm:295-395 (kernels), :1040-1166 (dispatch order).  Every f32 sum is
// taken in the reference's order: sequentially inside a 256-token tile, then sequentially over
// the tile totals.  A guard pointer makes every kernel a no-op unless the compact kernel handed
// over (law->count == kLawFull), like the reference's compact-count guards.
// =========================================================================================
constexpr uint32_t kSortTile = 2048, kLawTile = 256;

struct FullLawWs {
    uint64_t* keys_a; uint64_t* keys_b;  // sort ping-pong, padded to a power of two
    float* scores;                       // processed score by token id; -inf once filtered out
    float* prefix;                       // running f32 sums inside each 256-tile
    float* offsets;                      // [tiles + 1] running sums of the tile totals
    float* best;                         // [0] maximum of the surviving scores, [1] argmax as bits
    uint32_t* error;                     // law-local error word (also mirrored into status)
};

__device__ __forceinline__ bool guarded_off(const uint32_t* guard) { return guard && *guard != kLawFull; }
__device__ __forceinline__ float key_score(uint64_t key) {
    const uint32_t o = static_cast<uint32_t>(key >> 32);
    return __uint_as_float((o & 0x80000000u) ? (o & 0x7FFFFFFFu) : ~o);
}
__device__ __forceinline__ uint32_t key_token(uint64_t key) { return 0xFFFFFFFFu - static_cast<uint32_t>(key); }
__device__ __forceinline__ void law_fail(uint32_t* status, uint32_t* error, uint32_t bits) {
    atomicOr(status, bits);
    atomicOr(error, bits);
}

// unguarded entry: claims the law slot for the full table
__global__ void law_begin_kernel(DraftLaw* law, uint32_t* proposal, uint32_t* error) {
    law->count = kLawFull; law->pad = 0; *proposal = 0xFFFFFFFFu; *error = 0;
}

// score = logit / T (gd_process), then 2048-token tiles sorted by (score desc, token asc)
__global__ void __launch_bounds__(1024)
law_sort_tile_kernel(const float* __restrict__ logits, uint32_t vocab, float temperature, bool sort, bool suppressed_ok,
                     const uint32_t* __restrict__ guard, FullLawWs ws, uint32_t* __restrict__ status) {
    if (guarded_off(guard)) return;
    __shared__ uint64_t keys[kSortTile];
    for (uint32_t e = threadIdx.x; e < kSortTile; e += blockDim.x) {
        const uint32_t token = blockIdx.x * kSortTile + e;
        uint64_t key = 0;  // padding sorts behind every real entry
        if (token < vocab) {
            float score = logits[token];
            // a score of -inf marks a draft token the vocabulary map gives no target token (its raw logit was
            // validated where the scores were made): it stays out of every sum and sorts last
            const bool suppressed = suppressed_ok && score == -INFINITY;
            if (!suppressed) {
                if (!isfinite(score)) { law_fail(status, ws.error, GUFFIN_STATUS_LAW_INVALID | GUFFIN_STATUS_NONFINITE); score = 0.f; }
                if (temperature > 0.f) score = __fdiv_rn(score, temperature);
                if (!isfinite(score)) { law_fail(status, ws.error, GUFFIN_STATUS_LAW_INVALID | GUFFIN_STATUS_NONFINITE); score = 0.f; }
            }
            ws.scores[token] = score;
            key = score_key(score, token);
        }
        keys[e] = key;
    }
    if (!sort) return;
    bitonic(keys, kSortTile, true);
    for (uint32_t e = threadIdx.x; e < kSortTile; e += blockDim.x) ws.keys_a[size_t(blockIdx.x) * kSortTile + e] = keys[e];
}

// one merge level of sorted runs of `width` keys (descending; keys are distinct except padding)
__global__ void __launch_bounds__(256)
law_merge_kernel(const uint64_t* __restrict__ in, uint64_t* __restrict__ out, uint32_t width, uint32_t padded,
                 const uint32_t* __restrict__ guard) {
    if (guarded_off(guard)) return;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= padded) return;
    const uint32_t rank = i % (2 * width);
    const uint64_t* a = in + (i - rank);
    const uint64_t* b = a + width;
    uint32_t lo = rank > width ? rank - width : 0, hi = rank < width ? rank : width;
    while (lo < hi) {  // how many of the first `rank` outputs come from run a
        const uint32_t mid = (lo + hi) >> 1;
        if (a[mid] >= b[rank - mid - 1]) lo = mid + 1; else hi = mid;
    }
    const uint32_t ai = lo, bi = rank - lo;
    out[i] = (ai < width && (bi >= width || a[ai] >= b[bi])) ? a[ai] : b[bi];
}

// sequential offsets over the tile totals left in offsets[1..tiles] (gd_offsets); one thread
__device__ void finish_offsets(float* offsets, uint32_t tiles) {
    float s = 0.f;
    offsets[0] = 0.f;
    for (uint32_t g = 0; g < tiles; ++g) { s = __fadd_rn(s, offsets[g + 1]); offsets[g + 1] = s; }
}

// gd_filter_prefix + gd_offsets: weights of the sorted entries walked from the tail
__global__ void __launch_bounds__(1024)
law_filter_prefix_kernel(const uint64_t* __restrict__ sorted, uint32_t vocab, uint32_t top_k,
                         const uint32_t* __restrict__ guard, FullLawWs ws) {
    if (guarded_off(guard)) return;
    const uint32_t tiles = vocab / kLawTile;
    const float best = key_score(sorted[0]);
    const float cutoff = key_score(sorted[(top_k < vocab ? top_k : vocab) - 1]);
    for (uint32_t g = threadIdx.x; g < tiles; g += blockDim.x) {
        float run = 0.f;
        for (uint32_t j = 0; j < kLawTile; ++j) {
            const float score = key_score(sorted[vocab - 1 - (g * kLawTile + j)]);
            run = __fadd_rn(run, score >= cutoff ? law_exp(__fsub_rn(score, best)) : 0.f);
            ws.prefix[g * kLawTile + j] = run;
        }
        ws.offsets[g + 1] = run;
    }
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) finish_offsets(ws.offsets, tiles);
}

// gd_filter_apply: top-k cutoff (ties kept), ascending-tail top-p, min-p; the best entry always stays
__global__ void __launch_bounds__(256)
law_filter_apply_kernel(const uint64_t* __restrict__ sorted, uint32_t vocab, SamplerOptions opt,
                        const uint32_t* __restrict__ guard, FullLawWs ws) {
    if (guarded_off(guard)) return;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= vocab) return;
    const uint32_t tiles = vocab / kLawTile;
    const uint64_t item = sorted[vocab - 1 - i];
    const float score = key_score(item), best = key_score(sorted[0]);
    const float cutoff = key_score(sorted[(opt.top_k < vocab ? opt.top_k : vocab) - 1]);
    bool keep = score >= cutoff;
    const float tail = __fdiv_rn(__fadd_rn(ws.offsets[i / kLawTile], ws.prefix[i]), ws.offsets[tiles]);
    if (opt.top_p < 1.0f && tail <= __fsub_rn(1.0f, opt.top_p) && i != vocab - 1) keep = false;
    if (opt.min_p > 0.0f && law_exp(__fsub_rn(score, best)) < opt.min_p && i != vocab - 1) keep = false;
    if (!keep) ws.scores[key_token(item)] = -INFINITY;
}

// gd_max + gd_max_finish + gd_prefix + gd_offsets: maximum (lowest id on ties) of the surviving
// scores, then the weights exp(score - max) summed in token order
__global__ void __launch_bounds__(1024)
law_weights_kernel(uint32_t vocab, bool greedy, const uint32_t* __restrict__ guard, FullLawWs ws,
                   uint32_t* __restrict__ status) {
    if (guarded_off(guard)) return;
    __shared__ float s_max[1024];
    __shared__ uint32_t s_arg[1024];
    const uint32_t t = threadIdx.x, tiles = vocab / kLawTile;
    float m = -INFINITY;
    uint32_t arg = 0xFFFFFFFFu;
    for (uint32_t i = t; i < vocab; i += blockDim.x) {
        const float v = ws.scores[i];
        if (v > m) { m = v; arg = i; }  // ids ascend within a thread: the first maximum is the lowest id
    }
    s_max[t] = m; s_arg[t] = arg;
    __syncthreads();
    for (uint32_t half = blockDim.x >> 1; half > 0; half >>= 1) {
        if (t < half && (s_max[t + half] > s_max[t] || (s_max[t + half] == s_max[t] && s_arg[t + half] < s_arg[t]))) {
            s_max[t] = s_max[t + half]; s_arg[t] = s_arg[t + half];
        }
        __syncthreads();
    }
    const float maximum = s_max[0];
    if (t == 0) {
        ws.best[0] = maximum;
        ws.best[1] = __uint_as_float(s_arg[0]);
        if (!isfinite(maximum)) law_fail(status, ws.error, GUFFIN_STATUS_LAW_INVALID);
    }
    if (greedy) return;
    for (uint32_t g = t; g < tiles; g += blockDim.x) {
        float run = 0.f;
        for (uint32_t j = 0; j < kLawTile; ++j) {
            const float score = ws.scores[g * kLawTile + j];
            // the reference divides by a temperature of exactly 1 here: scores were tempered up front
            run = __fadd_rn(run, score > -INFINITY ? law_exp(__fdiv_rn(__fsub_rn(score, maximum), 1.0f)) : 0.f);
            ws.prefix[g * kLawTile + j] = run;
        }
        ws.offsets[g + 1] = run;
    }
    __threadfence();
    __syncthreads();
    if (t == 0) {
        finish_offsets(ws.offsets, tiles);
        const float total = ws.offsets[tiles];
        if (!(total > 0.f) || !isfinite(total)) law_fail(status, ws.error, GUFFIN_STATUS_LAW_INVALID);
    }
}

__device__ __forceinline__ uint64_t full_cdf_at(uint32_t i, uint32_t vocab, bool greedy, const FullLawWs& ws) {
    if (greedy) return i <= __float_as_uint(ws.best[1]) ? 0 : kMassTotal;
    if (i == 0) return 0;
    if (i == vocab) return kMassTotal;
    const uint32_t b = i / kLawTile;
    const float sum = (i % kLawTile == 0) ? ws.offsets[b] : __fadd_rn(ws.offsets[b], ws.prefix[i - 1]);
    float scaled = __fmul_rn(__fdiv_rn(sum, ws.offsets[vocab / kLawTile]), 4294967296.0f);
    scaled = fminf(fmaxf(scaled, 0.0f), 4294967296.0f);
    return static_cast<uint64_t>(scaled);
}

// gd_cdf + gd_select: the u64 table, its validation, and the token whose bin holds the step's word
__global__ void __launch_bounds__(256)
law_cdf_select_kernel(uint32_t vocab, bool greedy, uint64_t seed, uint64_t step, const StepDraws* __restrict__ injected,
                      const uint32_t* __restrict__ guard, FullLawWs ws, uint64_t* __restrict__ cdf,
                      uint32_t* __restrict__ proposal, uint32_t* __restrict__ status) {
    if (guarded_off(guard)) return;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > vocab) return;
    if (*ws.error != 0) { cdf[i] = 0; return; }  // raised by an earlier kernel: no law, no proposal
    const uint64_t begin = full_cdf_at(i, vocab, greedy, ws);
    cdf[i] = begin;
    if (i == vocab) return;
    const uint64_t end = full_cdf_at(i + 1, vocab, greedy, ws);
    if (begin > end || end > kMassTotal) { atomicOr(status, GUFFIN_STATUS_LAW_INVALID); return; }
    if (begin < end && !(ws.scores[i] > -INFINITY)) { atomicOr(status, GUFFIN_STATUS_LAW_INVALID); return; }
    const uint64_t word = injected ? injected->word : step_draws(seed, step).word;
    if (word >= begin && word < end) *proposal = i;
}

// =========================================================================================
// Target law (prepare_token_distribution) of the two candidate rows, and the accept / residual decision
// =========================================================================================
// One workgroup of two teams, a candidate row each: whether row 1 is wanted is known only at the end, and by then its law is
// ready.  The kernel is a chain of short dependent steps, so what it costs is their number: everything is requested at once;
// duplicates and places come out of one walk over the record; a sum whose order matters is one lane's, the masses of q another
// wave's beside it; running sums are kept, so that a draw is found by all
// lanes at once; at temperatures of 1 and 0 the tempered weights are the raw ones and their sums are not taken twice.
// An accepted proposal over 64 candidates takes 10.0 us (twice that with a row after the other, and a step after the other inside).
constexpr uint32_t kTeam = kMaxCandidates;   // threads of a row, a candidate each

struct Prepared {
    uint32_t count;
    double total;
    uint32_t token[kMaxTopK];
    double weight[kMaxTopK];         // zeros behind the last entry
    double run[kMaxTopK];            // running sums of the weights, in index order
};

struct RowScratch {
    uint64_t keys[kMaxCandidates], sorted[kMaxCandidates];
    float raw[kMaxCandidates];
    double w[kMaxTopK];              // raw weights, zeros behind the last entry
    double lost[kMaxTopK];           // what the running sums of the weights lost, entry by entry
    double lost_all;
    uint32_t hist[kHistoryCap];
    uint32_t kept, cut;              // ends of the top-p and min-p prefixes
    uint32_t dup, unique, flag, pick;
    int err;
};

// Neumaier's compensated sum over v[0] ... v[i] is run[i] plus the sum of what its additions lost: the terms of that sum are every
// lane's own where the running sums are known, and what is left of the order are additions.  (All of it by one lane, an entry after
// the other, beside the plain sums: an accepted proposal 10.4 us, so 10.0.)
__device__ __forceinline__ double lost_by(const double* __restrict__ v, const double* __restrict__ run, uint32_t i) {
    const double w = v[i], total = i ? run[i - 1] : 0.0, sum = run[i];
    return total >= w ? (total - sum) + w : (w - sum) + total;
}
// the reference's consistency check of a law's stored total against its compensated sum
__device__ __forceinline__ bool total_holds(double total, double stored, uint32_t count) {
    const double tol = static_cast<double>(count) * 2.220446049250313e-16 * total;
    return isfinite(total) && total > 0.0 && !(fabs(total - stored) > tol);
}
__device__ __forceinline__ bool total_usable(uint32_t count, double stored) {
    return !(count == 0 || count > kMaxTopK || !isfinite(stored) || stored <= 0.0);
}
__device__ __forceinline__ bool weight_usable(double w, double stored) {
    const double prob = w / stored;  // the stored probability is exactly this quotient
    return isfinite(prob) && !(prob < 0.0) && !(prob > 1.0) && isfinite(w) && !(w < 0.0);
}

// target_to_draft: null when both sides share one vocabulary; else the law lives in draft ids and a
// target token's mass is that of the draft token mapped to it, if any (Gemma3DraftPlan::gather,
// src/engine/gemma3_draft.mm:1570-1578)
// The compact law as the acceptance kernel keeps it in LDS (ids ascending, cdf[i] .. cdf[i + 1] the mass of ids[i]).
struct LawCopy { uint32_t count; uint32_t ids[256]; uint64_t cdf[257]; };

__device__ uint64_t law_mass(const LawCopy& law, const uint64_t* full_cdf, uint32_t vocab, uint32_t token,
                             uint64_t* begin, const int32_t* target_to_draft = nullptr) {
    if (target_to_draft) {
        const int32_t draft = target_to_draft[token];
        if (draft < 0) { if (begin) *begin = 0; return 0; }
        token = static_cast<uint32_t>(draft);
    }
    if (law.count == kLawFull) {  // gather from the full table (src/engine/gemma3_draft.mm:1544-1545)
        if (!full_cdf || token >= vocab) { if (begin) *begin = 0; return 0; }
        if (begin) *begin = full_cdf[token];
        return full_cdf[token + 1] - full_cdf[token];
    }
    const uint32_t count = law.count < 256u ? law.count : 256u;
    uint32_t lo = 0, hi = count;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (law.ids[mid] < token) lo = mid + 1; else hi = mid;
    }
    if (lo == count || law.ids[lo] != token) { if (begin) *begin = 0; return 0; }
    if (begin) *begin = law.cdf[lo];
    return law.cdf[lo + 1] - law.cdf[lo];
}

__global__ void __launch_bounds__(2 * kTeam)
spec_accept_kernel(const Candidates* __restrict__ rows, const DraftLaw* __restrict__ law,
                   const uint64_t* __restrict__ full_cdf, uint32_t vocab, const uint32_t* __restrict__ history,
                   const uint32_t* __restrict__ history_count, const uint32_t* __restrict__ proposal_ptr, SamplerOptions opt, uint64_t seed, uint64_t step,
                   const StepDraws* __restrict__ injected, SpecResult* __restrict__ result,
                   uint32_t* __restrict__ status, const int32_t* __restrict__ target_to_draft) {
    __shared__ RowScratch scratch[2];
    __shared__ Prepared prepared[2], residual;
    __shared__ uint64_t q[kMaxTopK];
    __shared__ double diff[kMaxTopK];
    __shared__ double s_acceptance;
    __shared__ uint64_t s_begin, s_mass;
    __shared__ LawCopy q_law;
    __shared__ uint64_t wave_mass[2 * kTeam / 64];
    __shared__ uint32_t wave_count[2 * kTeam / 64];
    const uint32_t team = __builtin_amdgcn_readfirstlane(threadIdx.x / kTeam), t = threadIdx.x - team * kTeam, lane = t & 63;
    RowScratch& sc = scratch[team];
    Prepared& out = prepared[team];
    // ---- everything in one trip: a row's record, its history and the compact law are always whole in memory ----
    const Candidates* cand = &rows[team];
    const uint32_t n = cand->count;
    const uint32_t token = cand->values[t].token;
    const float raw = cand->values[t].logit;
    const uint32_t history_n = history ? history_count[team] : 0u;
    const uint32_t past = history && t < kHistoryCap ? history[team * kHistoryCap + t] : 0u;
    const uint32_t law_id = team == 0 && t < 256 ? law->ids[t] : 0u;
    const uint64_t law_edge = team == 0 && t < 257 ? law->cdf[t] : 0u;
    const uint32_t law_count = law->count, proposal = *proposal_ptr;
    const StepDraws d = injected ? *injected : step_draws(seed, step);
    if (team == 0 && t < 256) q_law.ids[t] = law_id;
    if (team == 0 && t < 257) q_law.cdf[t] = law_edge;
    if (t == 0) {
        sc.err = !options_valid(opt) ? -1 : (n == 0 || n > kMaxCandidates) ? -2 : history_n > kHistoryCap ? -3 : 0;
        sc.dup = 0; sc.unique = 0; sc.flag = 0; sc.pick = 0xFFFFFFFFu;
        if (team == 0) { q_law.count = law_count; s_acceptance = 0.0; }
    }
    if (t < kHistoryCap) sc.hist[t] = past;
    __syncthreads();
    // ---- repetition penalty and sort key ------------------------------------------------------------------
    int rc = sc.err;
    const uint32_t entries = rc ? 0u : n;
    uint64_t key = 0;
    if (t < entries) {
        float logit = raw;
        for (uint32_t h = 0; h < history_n; ++h)
            if (sc.hist[h] == token) {
                logit = logit < 0.f ? __fmul_rn(logit, opt.repetition_penalty) : __fdiv_rn(logit, opt.repetition_penalty);
                break;
            }
        key = score_key(logit, token);
        sc.keys[t] = key;
        sc.raw[t] = raw;
    }
    __syncthreads();
    if (t < entries && !isfinite(raw)) atomicMin(&sc.err, -4);
    // ---- places: the keys ahead of one's own, counted by four neighbouring lanes where the team has them to spare ----
    {
        const bool fours = entries <= kTeam / 4;
        const uint32_t i = fours ? t >> 2 : t, from = fours ? t & 3u : 0u, by = fours ? 4u : 1u;
        const uint64_t own = i < entries ? sc.keys[i] : 0;
        uint32_t rank = 0, same = 0;
#pragma unroll 8
        for (uint32_t j = from; j < entries; j += by) {
            const uint64_t other = sc.keys[j];
            rank += other > own;
            same += static_cast<uint32_t>(other) == static_cast<uint32_t>(own);   // one's own token, once
        }
        if (fours) {
            rank += lane_cross_u32<0xB1, 0xF>(rank); rank += lane_cross_u32<0x4E, 0xF>(rank);
            same += lane_cross_u32<0xB1, 0xF>(same); same += lane_cross_u32<0x4E, 0xF>(same);
        }
        if (i < entries && from == 0) {
            if (same > 1) sc.dup = 1;
            sc.sorted[rank] = own;
        }
        if (t == 0) sc.unique = entries;
    }
    __syncthreads();
    if (scratch[0].dup | scratch[1].dup) {
        // a token more than once: the first entry stays, a later one must carry the same logit
        bool drop = false, differs = false;
        if (t < entries)
            for (uint32_t j = 0; j < t; ++j) {
                const bool same = static_cast<uint32_t>(sc.keys[j]) == static_cast<uint32_t>(key);
                drop |= same;
                differs |= same & (sc.raw[j] != raw);
            }
        if (differs) atomicMin(&sc.err, -5);
        __syncthreads();
        if (drop) key = 0;   // a real key of a finite logit is never 0
        if (t < entries) sc.keys[t] = key;
        sc.sorted[t] = 0;
        if (t == 0) sc.unique = 0;
        __syncthreads();
        if (key != 0) {
            uint32_t rank = 0;
            for (uint32_t j = 0; j < entries; ++j) rank += sc.keys[j] > key;
            sc.sorted[rank] = key;
            atomicAdd(&sc.unique, 1u);
        }
        __syncthreads();
    }
    // ---- raw weights of the best top_k -----------------------------------------------------------------------
    rc = sc.err;
    const uint32_t request_top_k = opt.temperature == 0.f ? 1u : opt.top_k;
    if (!rc && sc.unique < request_top_k) rc = -6;
    uint32_t count = rc ? 0u : request_top_k;
    const bool plain = opt.temperature == 1.f || opt.temperature == 0.f;
    float below = 0.f;   // how far the entry's logit lies under the best
    if (t < kMaxTopK) {
        double w = 0.0;
        if (t < count) {
            const uint64_t mine = sc.sorted[t];
            below = __fsub_rn(key_score(mine), key_score(sc.sorted[0]));
            out.token[t] = key_token(mine);
            w = opt.temperature == 0.f ? 1.0 : exp(static_cast<double>(below));   // greedy: one, also where the penalty made the best infinite
        }
        sc.w[t] = w;
    }
    if (t == 0) { sc.kept = count; sc.cut = count; }
    __syncthreads();
    if (t == 0) ordered_sums(sc.w, count, out.run);
    if (team == 0) {
        if (!target_to_draft && t >= 128 && t - 128 < count) q[t - 128] = law_mass(q_law, full_cdf, vocab, out.token[t - 128], nullptr);
    } else if (t == 128) {
        uint64_t begin = 0;   // a law that failed leaves no proposal
        s_mass = scratch[0].err || proposal == 0xFFFFFFFFu ? 0 : law_mass(q_law, full_cdf, vocab, proposal, &begin, target_to_draft);
        s_begin = begin;
    }
    __syncthreads();
    // ---- top-p keeps entries up to and including the first whose running share reaches top_p; min-p then keeps the leading
    // entries (the first always) whose weight is at least min_p
    if (count) {
        const double total = out.run[count - 1];
        note_first(t + 1 < count && !(out.run[t] / total < static_cast<double>(opt.top_p)), t + 1, &sc.kept);
        if (opt.min_p > 0.f) note_first(t >= 1 && t < count && !(sc.w[t] >= static_cast<double>(opt.min_p)), t, &sc.cut);
    }
    __syncthreads();
    count = sc.kept < sc.cut ? sc.kept : sc.cut;
    if (plain) {
        if (t < kMaxTopK) out.weight[t] = t < count ? sc.w[t] : 0.0;
    } else {
        if (t < kMaxTopK) out.weight[t] = t < count ? exp(static_cast<double>(below) / static_cast<double>(opt.temperature)) : 0.0;
        __syncthreads();
        if (t == 0) ordered_sums(out.weight, count, out.run);
        __syncthreads();
    }
    if (team == 0 && t < kMaxTopK) sc.lost[t] = t < count ? lost_by(out.weight, out.run, t) : 0.0;
    __syncthreads();
    if (team == 0 && t == 64) sc.lost_all = ordered_sums<double>(sc.lost, count, nullptr);
    const double norm = count ? out.run[count - 1] : 0.0;
    if (!rc && (!isfinite(norm) || norm <= 0.0)) rc = -7;
    if (t == 0) { out.count = rc ? 0u : count; out.total = norm; if (team == 1) sc.err = rc; }
    // ---- the checks of both laws, and what the proposal weighs in each ------------------------------------------
    // (from here on team 0's threads work on row 0's law; team 1 follows through the barriers)
    const bool head = team == 0;
    bool holds_proposal = false;
    uint64_t mass = 0;
    if (head && !rc && t < count) {
        // through a vocabulary map only the tokens that stay are looked up
        if (target_to_draft) q[t] = law_mass(q_law, full_cdf, vocab, out.token[t], nullptr, target_to_draft);
        // A mass is a difference of two edges: over edges out of order it wraps, and the sum of the masses may still be 2^32.
        // Counted as at most 2^32 + 1 each, 256 of them cannot wrap, and their sum, which as one of whole numbers does not
        // depend on the order, passes 2^32 exactly where some prefix does or some mass by itself.
        mass = q[t] <= kMassTotal ? q[t] : kMassTotal + 1;
        holds_proposal = out.token[t] == proposal;
        if (!weight_usable(out.weight[t], norm)) sc.flag = 1;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mass += __shfl_xor(mass, o, kWave);
    if (lane == 0) wave_mass[threadIdx.x >> 6] = mass;
    const bool in_target = __syncthreads_or(holds_proposal) != 0;
    // ---- from here every thread follows row 0's decision ---------------------------------------------------------
    const Prepared& target = prepared[0];
    int code = head ? rc : 0;
    double proposed = 0.0, normalization = -1.0;
    if (head && !code) {
        auto unit = [](double u) { return isfinite(u) && u >= 0.0 && u < 1.0; };
        normalization = norm + scratch[0].lost_all;
        const bool valid = total_usable(count, norm) && !sc.flag && total_holds(normalization, norm, count);
        uint64_t gathered = 0;
        for (uint32_t w = 0; w < kTeam / 64; ++w) gathered += wave_mass[w];
        if (!unit(d.u_accept) || !unit(d.u_residual) || !unit(d.u_next)) code = -20;
        else if (!valid) code = -21;
        else if (s_mass == 0 || s_mass > kMassTotal || s_begin > kMassTotal - s_mass) code = -22;
        else if (gathered > kMassTotal) code = -23;
        else if (!in_target && s_mass > kMassTotal - gathered) code = -24;
        proposed = static_cast<double>(s_mass) / static_cast<double>(kMassTotal);
    }
    // p, p / q of the proposal and p - q per lane; then the entries with an excess, in order, without gaps
    bool more = false;
    if (head && !code && t < count) {
        const double p = target.weight[t] / normalization;
        if (target.token[t] == proposal) s_acceptance = fmin(1.0, p / proposed);   // tokens are distinct
        diff[t] = p - static_cast<double>(q[t]) / static_cast<double>(kMassTotal);
        more = !(diff[t] <= 0.0);
    }
    const uint64_t ahead = __ballot(more);
    if (lane == 0) wave_count[threadIdx.x >> 6] = static_cast<uint32_t>(__popcll(ahead));
    __syncthreads();
    uint32_t at = static_cast<uint32_t>(__popcll(ahead & ((uint64_t{1} << lane) - 1))), excess = 0;
    for (uint32_t w = 0; w < kTeam / 64; ++w) {
        if (w < (t >> 6)) at += wave_count[w];
        excess += wave_count[w];
    }
    if (head) {
        if (t >= excess && t < kMaxTopK) residual.weight[t] = 0.0;
        if (more) { residual.token[at] = target.token[t]; residual.weight[at] = diff[t]; }
        if (t == 0) sc.flag = 0;
    }
    __syncthreads();
    if (head && t == 0) ordered_sums(residual.weight, excess, residual.run);
    __syncthreads();
    if (head && t < kMaxTopK) sc.lost[t] = t < excess ? lost_by(residual.weight, residual.run, t) : 0.0;
    __syncthreads();
    if (head && t == 0) sc.lost_all = ordered_sums<double>(sc.lost, excess, nullptr);
    __syncthreads();
    const double acceptance = s_acceptance, residual_total = excess ? residual.run[excess - 1] : 0.0;
    const bool decided = code == 0;
    bool accepted = false;
    if (head && decided) {
        if (excess == 0 && acceptance < 1.0) code = -25;
        else accepted = d.u_accept < acceptance;
    }
    // ---- the draw: row 1's law behind an accepted proposal, the residual otherwise ---------------------------------
    if (head && code == 0) {
        if (accepted) {
            const Prepared& after = prepared[1];
            if (scratch[1].err) code = scratch[1].err - 100;
            else note_first(t < after.count && d.u_next * after.total < after.run[t], t, &sc.pick);
        } else {
            if (!total_usable(excess, residual_total) || !total_holds(residual_total + sc.lost_all, residual_total, excess)) code = -26;
            else {
                if (t < excess && !weight_usable(residual.weight[t], residual_total)) sc.flag = 1;
                note_first(t < excess && d.u_residual * residual_total < residual.run[t], t, &sc.pick);
            }
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        if (!code && !accepted && sc.flag) code = -26;
        const Prepared& from = accepted ? prepared[1] : residual;
        const uint32_t length = accepted ? prepared[1].count : excess;
        const uint32_t drawn = code ? 0xFFFFFFFFu : from.token[opt.temperature == 0.f && accepted ? 0u : min(sc.pick, length - 1)];
        result->accepted = !code && accepted;
        result->token = code ? 0xFFFFFFFFu : accepted ? proposal : drawn;
        result->next_root = drawn;
        result->status = static_cast<uint32_t>(-code);
        result->acceptance_probability = decided ? acceptance : 0.0;
        result->residual_total = decided ? residual_total : 0.0;
        result->residual_count = decided ? excess : 0u;
        result->proposal = proposal;
        if (code && status) atomicOr(status, GUFFIN_STATUS_LAW_INVALID);
    }
}

}  // namespace

int select_candidates_scaled(hipStream_t s, const float* logits, uint32_t rows, uint32_t vocab, uint32_t retain,
                             float divisor, const uint32_t* history, const uint32_t* history_count,
                             void* workspace, void* result, uint32_t* status, bool suppressed_ok = false,
                             const uint32_t* row_retain = nullptr, uint32_t row_stride = 1, uint32_t sure = 0, bool fresh = false);

}  // namespace guffin

using namespace guffin;

extern "C" uint64_t guffin_hip_draft_law_workspace_bytes(uint32_t vocab) {
    // workspace of the 257-best selection plus the sorted candidate row
    return ((guffin_hip_select_workspace_bytes(1, vocab, 257) + 15) & ~uint64_t{15}) + sizeof(Candidates) + 16;
}

namespace {

uint32_t padded_vocab(uint32_t vocab) {
    uint32_t p = kSortTile;
    while (p < vocab) p <<= 1;
    return p;
}
uint64_t align16(uint64_t v) { return (v + 15) & ~uint64_t{15}; }
uint64_t compact_ws_bytes(uint32_t vocab) { return align16(guffin_hip_draft_law_workspace_bytes(vocab)); }

FullLawWs carve_full_ws(uint8_t* base, uint32_t vocab) {
    const uint64_t padded = padded_vocab(vocab), tiles = vocab / kLawTile;
    FullLawWs ws;
    uint64_t at = 0;
    auto take = [&](uint64_t bytes) { uint8_t* p = base ? base + at : nullptr; at += align16(bytes); return p; };
    ws.keys_a = reinterpret_cast<uint64_t*>(take(padded * 8));
    ws.keys_b = reinterpret_cast<uint64_t*>(take(padded * 8));
    ws.scores = reinterpret_cast<float*>(take(uint64_t(vocab) * 4));
    ws.prefix = reinterpret_cast<float*>(take(uint64_t(vocab) * 4));
    ws.offsets = reinterpret_cast<float*>(take((tiles + 1) * 4));
    ws.best = reinterpret_cast<float*>(take(8));
    ws.error = reinterpret_cast<uint32_t*>(take(4));
    return ws;
}
uint64_t full_ws_bytes(uint32_t vocab) {
    const uint64_t padded = padded_vocab(vocab), tiles = vocab / kLawTile;
    return align16(padded * 8) * 2 + align16(uint64_t(vocab) * 4) * 2 + align16((tiles + 1) * 4) + 16 + 16;
}
bool compact_options(const SamplerOptions& o) { return o.temperature > 0.f && o.top_k >= 1 && o.top_k <= 64; }

int launch_compact_law(hipStream_t s, const float* logits, uint32_t vocab, const SamplerOptions& opt, uint64_t seed,
                       uint64_t step, const void* injected_draws, void* workspace, void* law, uint32_t* proposal,
                       uint32_t* status, uint32_t* full_error, bool suppressed_ok = false, bool fresh = false) {
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    const LawCall call {opt, seed, step, static_cast<const StepDraws*>(injected_draws), static_cast<DraftLaw*>(law), proposal, status, full_error, fresh};
    if (selection_makes_laws(vocab, 257)) return select_law(s, logits, vocab, 257, opt.top_k, ws, call, suppressed_ok);
    Candidates* top = reinterpret_cast<Candidates*>(ws + ((guffin_hip_select_workspace_bytes(1, vocab, 257) + 15) & ~uint64_t{15}));
    // the k-th best score and every tie with it, up to one more than a compact law holds, decide it
    if (int rc = select_candidates_scaled(s, logits, 1, vocab, vocab < 257 ? vocab : 257, opt.temperature, nullptr,
                                          nullptr, ws, top, status, suppressed_ok, nullptr, 1, opt.top_k, fresh))
        return rc;
    launch(draft_law_kernel, dim3(1), dim3(256), 0, s, top, call);
    return check_launch("draft_law");
}

// the full-vocabulary kernels in the reference's dispatch order (src/engine/gemma3_draft.mm:1040-1166)
int launch_full_law(hipStream_t s, const float* logits, uint32_t vocab, const SamplerOptions& opt, uint64_t seed,
                    uint64_t step, const void* injected_draws, const uint32_t* guard, const FullLawWs& ws,
                    uint64_t* cdf, uint32_t* proposal, uint32_t* status, bool suppressed_ok = false) {
    const bool greedy = opt.temperature == 0.f;
    const uint32_t padded = padded_vocab(vocab);
    launch(law_sort_tile_kernel, dim3(padded / kSortTile), dim3(1024), 0, s, logits, vocab, opt.temperature,
                       !greedy, suppressed_ok, guard, ws, status);
    if (!greedy) {
        const uint64_t* sorted = ws.keys_a;
        uint64_t* other = ws.keys_b;
        for (uint32_t width = kSortTile; width < padded; width <<= 1) {
            launch(law_merge_kernel, dim3(padded / 256), dim3(256), 0, s, sorted, other, width, padded, guard);
            const uint64_t* done = other;
            other = const_cast<uint64_t*>(sorted);
            sorted = done;
        }
        launch(law_filter_prefix_kernel, dim3(1), dim3(1024), 0, s, sorted, vocab, opt.top_k, guard, ws);
        launch(law_filter_apply_kernel, dim3((vocab + 255) / 256), dim3(256), 0, s, sorted, vocab, opt, guard, ws);
    }
    launch(law_weights_kernel, dim3(1), dim3(1024), 0, s, vocab, greedy, guard, ws, status);
    launch(law_cdf_select_kernel, dim3(vocab / 256 + 1), dim3(256), 0, s, vocab, greedy, seed, step,
                       static_cast<const StepDraws*>(injected_draws), guard, ws, cdf, proposal, status);
    return check_launch("draft_law_full");
}

}  // namespace

namespace {
int draft_law_compact(void* stream, const float* logits, uint32_t vocab, const void* options, uint64_t seed, uint64_t step,
                      const void* injected_draws, void* workspace, void* law, uint32_t* proposal, uint32_t* status, bool fresh) {
    if (!logits || !options || !workspace || !law || !proposal || !status) return fail(GUFFIN_E_ARG, "draft_law: null pointer");
    if (vocab < 1) return fail(GUFFIN_E_SHAPE, "draft_law: empty vocabulary");
    if (reinterpret_cast<uintptr_t>(workspace) & 7u) return fail(GUFFIN_E_ALIGN, "draft_law: workspace must be 8-byte aligned");
    const SamplerOptions opt = *static_cast<const SamplerOptions*>(options);
    if (!compact_options(opt))
        return fail(GUFFIN_E_ARG, "draft_law: the compact law needs temperature > 0 and top_k in [1, 64]");
    return launch_compact_law(as_stream(stream), logits, vocab, opt, seed, step, injected_draws, workspace, law,
                              proposal, status, nullptr, false, fresh);
}
}  // namespace

extern "C" int guffin_hip_draft_law(void* stream, const float* logits, uint32_t vocab, const void* options,
                                    uint64_t seed, uint64_t step, const void* injected_draws, void* workspace,
                                    void* law, uint32_t* proposal, uint32_t* status) {
    return draft_law_compact(stream, logits, vocab, options, seed, step, injected_draws, workspace, law, proposal, status, false);
}

extern "C" int guffin_hip_draft_law_fresh(void* stream, const float* logits, uint32_t vocab, const void* options,
                                          uint64_t seed, uint64_t step, const void* injected_draws, void* workspace,
                                          void* law, uint32_t* proposal, uint32_t* status) {
    return draft_law_compact(stream, logits, vocab, options, seed, step, injected_draws, workspace, law, proposal, status, true);
}

namespace guffin {
namespace {
// scores[i] = logits[i], divided by the penalty (multiplied when negative) for the tokens of the
// sampler history, and -inf for a draft token that the vocabulary map gives no target token: the
// drafter's gd_process without its division by the temperature, which follows in the selection
// (src/engine/gemma3_draft.mm:191-204).  With a map the raw logits are validated here, the
// suppressed ones included.
__global__ void __launch_bounds__(256)
draft_process_kernel(const float* __restrict__ logits, uint32_t vocab, const uint32_t* __restrict__ history,
                     uint32_t count, float penalty, const int32_t* __restrict__ draft_to_target,
                     float* __restrict__ scores, uint32_t* __restrict__ status) {
    __shared__ uint32_t seen[kHistoryCap];
    if (threadIdx.x < count) seen[threadIdx.x] = history[threadIdx.x];
    __syncthreads();
    bool bad = false;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < vocab; i += gridDim.x * blockDim.x) {
        float v = logits[i];
        bad |= !isfinite(v);
        bool hit = false;
        for (uint32_t j = 0; j < count; ++j) hit |= seen[j] == i;
        if (hit && penalty != 1.0f) v = v < 0.f ? v * penalty : v / penalty;
        if (draft_to_target && draft_to_target[i] < 0) v = -INFINITY;
        scores[i] = v;
    }
    if (bad && draft_to_target && status) atomicOr(status, GUFFIN_STATUS_NONFINITE);
}

// proposal in draft ids -> the target's id for it
__global__ void map_proposal_kernel(const int32_t* __restrict__ draft_to_target, uint32_t vocab,
                                    const uint32_t* __restrict__ draft_proposal, uint32_t* __restrict__ target_proposal) {
    const uint32_t d = *draft_proposal;
    *target_proposal = d < vocab && draft_to_target[d] >= 0 ? static_cast<uint32_t>(draft_to_target[d]) : 0xFFFFFFFFu;
}
}  // namespace
}  // namespace guffin

extern "C" int guffin_hip_draft_process(void* stream, const float* logits, uint32_t vocab, const uint32_t* history,
                                        uint32_t history_count, float repetition_penalty, float* scores) {
    if (!logits || !scores || (history_count && !history)) return fail(GUFFIN_E_ARG, "draft_process: null pointer");
    if (vocab == 0) return fail(GUFFIN_E_SHAPE, "draft_process: empty vocabulary");
    if (history_count > kHistoryCap) return fail(GUFFIN_E_CAPACITY, "draft_process: at most 64 history tokens");
    if (!std::isfinite(repetition_penalty) || !(repetition_penalty > 0.f)) return fail(GUFFIN_E_ARG, "draft_process: the penalty must be positive");
    const uint32_t blocks = std::min<uint32_t>((vocab + 255) / 256, 1024);
    launch(draft_process_kernel, dim3(blocks), dim3(256), 0, as_stream(stream), logits, vocab, history,
                       history_count, repetition_penalty, static_cast<const int32_t*>(nullptr), scores,
                       static_cast<uint32_t*>(nullptr));
    return check_launch("draft_process");
}

extern "C" int guffin_hip_draft_law_mapped(void* stream, const float* logits, uint32_t vocab, const int32_t* draft_to_target,
                                           const uint32_t* history, uint32_t history_count, const void* options,
                                           uint64_t seed, uint64_t step, const void* injected_draws, void* workspace,
                                           float* scores, void* law, uint32_t* draft_proposal, uint32_t* target_proposal,
                                           uint32_t* status) {
    if (!logits || !draft_to_target || !options || !workspace || !scores || !law || !draft_proposal || !target_proposal || !status
        || (history_count && !history))
        return fail(GUFFIN_E_ARG, "draft_law_mapped: null pointer");
    if (vocab == 0) return fail(GUFFIN_E_SHAPE, "draft_law_mapped: empty vocabulary");
    if (history_count > kHistoryCap) return fail(GUFFIN_E_CAPACITY, "draft_law_mapped: at most 64 history tokens");
    if (reinterpret_cast<uintptr_t>(workspace) & 15u) return fail(GUFFIN_E_ALIGN, "draft_law_mapped: workspace must be 16-byte aligned");
    const SamplerOptions opt = *static_cast<const SamplerOptions*>(options);
    if (!compact_options(opt))
        return fail(GUFFIN_E_ARG, "draft_law_mapped: the compact law needs temperature > 0 and top_k in [1, 64]");
    if (!std::isfinite(opt.repetition_penalty) || !(opt.repetition_penalty > 0.f)) return fail(GUFFIN_E_ARG, "draft_law_mapped: the penalty must be positive");
    hipStream_t s = as_stream(stream);
    const uint32_t blocks = std::min<uint32_t>((vocab + 255) / 256, 1024);
    launch(draft_process_kernel, dim3(blocks), dim3(256), 0, s, logits, vocab, history, history_count,
                       opt.repetition_penalty, draft_to_target, scores, status);
    if (int rc = check_launch("draft_process")) return rc;
    if (int rc = launch_compact_law(s, scores, vocab, opt, seed, step, injected_draws, workspace, law, draft_proposal, status,
                                    nullptr, true))
        return rc;
    launch(map_proposal_kernel, dim3(1), dim3(1), 0, s, draft_to_target, vocab, draft_proposal, target_proposal);
    return check_launch("map_proposal");
}

extern "C" uint64_t guffin_hip_draft_law_any_workspace_bytes(uint32_t vocab) {
    return compact_ws_bytes(vocab) + full_ws_bytes(vocab);
}

namespace {
int draft_law_any(void* stream, const float* logits, uint32_t vocab, const void* options, uint64_t seed, uint64_t step,
                  const void* injected_draws, void* workspace, void* law, uint64_t* full_cdf, uint32_t* proposal,
                  uint32_t* status, bool suppressed_ok) {
    if (!logits || !options || !workspace || !law || !full_cdf || !proposal || !status)
        return fail(GUFFIN_E_ARG, "draft_law_any: null pointer");
    if (vocab < kLawTile || vocab % kLawTile != 0)
        return fail(GUFFIN_E_SHAPE, "draft_law_any: the vocabulary must be a positive multiple of 256");
    if (reinterpret_cast<uintptr_t>(workspace) & 15u) return fail(GUFFIN_E_ALIGN, "draft_law_any: workspace must be 16-byte aligned");
    if (reinterpret_cast<uintptr_t>(full_cdf) & 7u) return fail(GUFFIN_E_ALIGN, "draft_law_any: the table must be 8-byte aligned");
    const SamplerOptions opt = *static_cast<const SamplerOptions*>(options);
    if (!std::isfinite(opt.temperature) || opt.temperature < 0.f || opt.top_k < 1 || opt.top_k > kMaxTopK
        || !(opt.top_p > 0.f) || opt.top_p > 1.f || !(opt.min_p >= 0.f) || opt.min_p > 1.f)
        return fail(GUFFIN_E_ARG, "draft_law_any: sampler options out of range");
    hipStream_t s = as_stream(stream);
    uint8_t* base = static_cast<uint8_t*>(workspace);
    const FullLawWs ws = carve_full_ws(base + compact_ws_bytes(vocab), vocab);
    DraftLaw* slot = static_cast<DraftLaw*>(law);
    if (compact_options(opt)) {
        // the compact law; its kernel hands over to the guarded full-vocabulary kernels when more
        // than 256 tokens tie into the support
        if (int rc = launch_compact_law(s, logits, vocab, opt, seed, step, injected_draws, base, law, proposal, status, ws.error, suppressed_ok))
            return rc;
        return launch_full_law(s, logits, vocab, opt, seed, step, injected_draws, &slot->count, ws, full_cdf, proposal, status, suppressed_ok);
    }
    launch(law_begin_kernel, dim3(1), dim3(1), 0, s, slot, proposal, ws.error);
    return launch_full_law(s, logits, vocab, opt, seed, step, injected_draws, nullptr, ws, full_cdf, proposal, status, suppressed_ok);
}
}  // namespace


extern "C" int guffin_hip_draft_law_any(void* stream, const float* logits, uint32_t vocab, const void* options,
                                        uint64_t seed, uint64_t step, const void* injected_draws, void* workspace,
                                        void* law, uint64_t* full_cdf, uint32_t* proposal, uint32_t* status) {
    return draft_law_any(stream, logits, vocab, options, seed, step, injected_draws, workspace, law, full_cdf, proposal, status, false);
}

extern "C" int guffin_hip_draft_law_any_mapped(void* stream, const float* logits, uint32_t vocab, const int32_t* draft_to_target,
                                               const uint32_t* history, uint32_t history_count, const void* options,
                                               uint64_t seed, uint64_t step, const void* injected_draws, void* workspace,
                                               float* scores, void* law, uint64_t* full_cdf, uint32_t* draft_proposal,
                                               uint32_t* target_proposal, uint32_t* status) {
    if (!logits || !draft_to_target || !options || !scores || !draft_proposal || !target_proposal || !status || (history_count && !history))
        return fail(GUFFIN_E_ARG, "draft_law_any_mapped: null pointer");
    if (vocab == 0) return fail(GUFFIN_E_SHAPE, "draft_law_any_mapped: empty vocabulary");
    if (history_count > kHistoryCap) return fail(GUFFIN_E_CAPACITY, "draft_law_any_mapped: at most 64 history tokens");
    const SamplerOptions opt = *static_cast<const SamplerOptions*>(options);
    if (!std::isfinite(opt.repetition_penalty) || !(opt.repetition_penalty > 0.f)) return fail(GUFFIN_E_ARG, "draft_law_any_mapped: the penalty must be positive");
    hipStream_t s = as_stream(stream);
    const uint32_t blocks = std::min<uint32_t>((vocab + 255) / 256, 1024);
    launch(draft_process_kernel, dim3(blocks), dim3(256), 0, s, logits, vocab, history, history_count,
                       opt.repetition_penalty, draft_to_target, scores, status);
    if (int rc = check_launch("draft_process")) return rc;
    if (int rc = draft_law_any(stream, scores, vocab, options, seed, step, injected_draws, workspace, law, full_cdf, draft_proposal,
                               status, true))
        return rc;
    launch(map_proposal_kernel, dim3(1), dim3(1), 0, s, draft_to_target, vocab, draft_proposal, target_proposal);
    return check_launch("map_proposal");
}

extern "C" int guffin_hip_spec_accept_mapped(void* stream, const void* target_candidates, const void* law,
                                             const uint64_t* full_cdf, uint32_t vocab, const int32_t* target_to_draft,
                                             const uint32_t* history, const uint32_t* history_count,
                                             const uint32_t* proposal, const void* options, uint64_t seed, uint64_t step,
                                             const void* injected_draws, void* result, uint32_t* status) {
    if (!target_candidates || !law || !proposal || !options || !result) return fail(GUFFIN_E_ARG, "spec_accept: null pointer");
    if ((history == nullptr) != (history_count == nullptr)) return fail(GUFFIN_E_ARG, "spec_accept: history needs its counts");
    const SamplerOptions opt = *static_cast<const SamplerOptions*>(options);
    launch(spec_accept_kernel, dim3(1), dim3(2 * kTeam), 0, as_stream(stream),
                       static_cast<const Candidates*>(target_candidates), static_cast<const DraftLaw*>(law), full_cdf,
                       vocab, history, history_count, proposal, opt, seed, step,
                       static_cast<const StepDraws*>(injected_draws), static_cast<SpecResult*>(result), status,
                       target_to_draft);
    return check_launch("spec_accept");
}

extern "C" int guffin_hip_spec_accept_history(void* stream, const void* target_candidates, const void* law,
                                              const uint64_t* full_cdf, uint32_t vocab, const uint32_t* history,
                                              const uint32_t* history_count, const uint32_t* proposal,
                                              const void* options, uint64_t seed, uint64_t step,
                                              const void* injected_draws, void* result, uint32_t* status) {
    return guffin_hip_spec_accept_mapped(stream, target_candidates, law, full_cdf, vocab, nullptr, history, history_count,
                                         proposal, options, seed, step, injected_draws, result, status);
}

extern "C" int guffin_hip_spec_accept_law(void* stream, const void* target_candidates, const void* law,
                                          const uint64_t* full_cdf, uint32_t vocab, const uint32_t* proposal,
                                          const void* options, uint64_t seed, uint64_t step,
                                          const void* injected_draws, void* result, uint32_t* status) {
    return guffin_hip_spec_accept_history(stream, target_candidates, law, full_cdf, vocab, nullptr, nullptr, proposal,
                                          options, seed, step, injected_draws, result, status);
}

extern "C" int guffin_hip_spec_accept(void* stream, const void* target_candidates, const void* law,
                                      const uint32_t* proposal, const void* options, uint64_t seed, uint64_t step,
                                      const void* injected_draws, void* result, uint32_t* status) {
    return guffin_hip_spec_accept_law(stream, target_candidates, law, nullptr, 0, proposal, options, seed, step,
                                      injected_draws, result, status);
}

extern "C" int guffin_hip_step_draws(uint64_t seed, uint64_t step, void* out_draws_host) {
    // host restatement of the device draw schedule, for callers that log or inject draws
    if (!out_draws_host) return fail(GUFFIN_E_ARG, "step_draws: null pointer");
    auto round = [](uint32_t (&c)[4], uint32_t (&k)[2]) {
        const uint64_t p0 = uint64_t{0xD2511F53u} * c[0], p1 = uint64_t{0xCD9E8D57u} * c[2];
        const uint32_t n0 = static_cast<uint32_t>(p1 >> 32) ^ c[1] ^ k[0], n1 = static_cast<uint32_t>(p1);
        const uint32_t n2 = static_cast<uint32_t>(p0 >> 32) ^ c[3] ^ k[1], n3 = static_cast<uint32_t>(p0);
        c[0] = n0; c[1] = n1; c[2] = n2; c[3] = n3;
        k[0] += 0x9E3779B9u; k[1] += 0xBB67AE85u;
    };
    StepDraws d {};
    uint32_t out[2][4];
    for (uint32_t block = 0; block < 2; ++block) {
        uint32_t c[4] = {static_cast<uint32_t>(step), static_cast<uint32_t>(step >> 32), block, 0};
        uint32_t k[2] = {static_cast<uint32_t>(seed), static_cast<uint32_t>(seed >> 32)};
        for (int r = 0; r < 10; ++r) round(c, k);
        for (int i = 0; i < 4; ++i) out[block][i] = c[i];
    }
    auto unit = [](uint32_t hi, uint32_t lo) { return static_cast<double>(((uint64_t{hi} << 32) | lo) >> 11) * 0x1.0p-53; };
    d.word = out[0][0];
    d.u_accept = unit(out[0][1], out[0][2]);
    d.u_residual = unit(out[1][0], out[1][1]);
    d.u_next = unit(out[1][2], out[1][3]);
    *static_cast<StepDraws*>(out_draws_host) = d;
    return GUFFIN_OK;
}
