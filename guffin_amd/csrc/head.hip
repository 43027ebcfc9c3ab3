// Output-head selection over the 262144-entry logits rows (gfx950).
//
// Replaces encode_token_candidates / encode_target_token_candidates and their tile-sort,
// merge-tree and finalize kernels (src/tensor/backends/metal/metal_command_context.hpp:326-345,
// src/tensor/backends/metal/metal_kernels.mm:3444-3884), and the CPU argmax
// (src/tensor/ops/reduction.cpp:93-117).  Order everywhere: higher logit first, then lower
// token id (src/engine/sampling.cpp:25-30, metal_kernels.mm:171-173).
//
// An entry is one 64-bit key {ordered(logit) : 32 | ~token : 32}; descending key order is the
// candidate order and keys are unique, so selection is a pure comparison network and the
// result is exact including ties.
//   stage 1  every workgroup sorts a 2048-logit tile in LDS (bitonic) and keeps its best R
//   stage 2  one workgroup per row picks the best `retain` of the G*R survivors (a threshold from
//            the sorted tile lists' heads plus a rank sort; a radix select where that does not
//            apply), then appends the logits of the history tokens
// A global top-R entry is necessarily a top-R entry of its own tile, so the two stages lose
// nothing.
#include "common.hpp"
#include "law.hpp"
#include "selection_request.hpp"

#include <cstddef>

namespace guffin {
namespace {

constexpr uint32_t kTile = 2048;          // logits per stage-1 workgroup

__device__ __forceinline__ uint64_t make_key(float logit, uint32_t token) {
    const uint32_t b = __float_as_uint(logit + 0.0f);  // -0 orders as +0, as a float comparison does
    const uint32_t ordered = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    return (uint64_t(ordered) << 32) | (0xFFFFFFFFu - token);
}
__device__ __forceinline__ float key_logit(uint64_t key) {
    const uint32_t o = static_cast<uint32_t>(key >> 32);
    return __uint_as_float((o & 0x80000000u) ? (o & 0x7FFFFFFFu) : ~o);
}
__device__ __forceinline__ uint32_t key_token(uint64_t key) { return 0xFFFFFFFFu - static_cast<uint32_t>(key); }

// descending bitonic sort of n (power of two) keys in LDS by all threads of the workgroup
__device__ __forceinline__ void bitonic_desc(uint64_t* keys, uint32_t n) {
    for (uint32_t width = 2; width <= n; width <<= 1) {
        for (uint32_t stride = width >> 1; stride > 0; stride >>= 1) {
            __syncthreads();
            for (uint32_t i = threadIdx.x; i < n / 2; i += blockDim.x) {
                const uint32_t lo = 2 * i - (i & (stride - 1));   // index with the `stride` bit clear
                const uint32_t hi = lo + stride;
                const bool descending = (lo & width) == 0;
                const uint64_t a = keys[lo], b = keys[hi];
                if ((a < b) == descending) { keys[lo] = b; keys[hi] = a; }
            }
        }
    }
    __syncthreads();
}

__global__ void __launch_bounds__(1024)
topk_tile_kernel(const float* __restrict__ logits, uint64_t* __restrict__ survivors, uint32_t vocab,
                 uint32_t keep, float divisor, uint32_t* __restrict__ status, bool suppressed_ok) {
    __shared__ uint64_t keys[kTile];
    const uint32_t tile = blockIdx.x, row = blockIdx.y;
    const float* lr = logits + size_t(row) * vocab;
    bool bad = false;
    for (uint32_t i = threadIdx.x; i < kTile; i += blockDim.x) {
        const uint32_t t = tile * kTile + i;
        uint64_t k = 0;  // below every real key
        if (t < vocab) {
            const float v = lr[t] / divisor;  // IEEE division: the drafter's score = logit / T
            // -inf marks a score that its producer suppressed (a draft token without a target token)
            bad |= (!isfinite(v) || !isfinite(lr[t])) && !(suppressed_ok && lr[t] == -INFINITY);
            k = make_key(v, t);
        }
        keys[i] = k;
    }
    if (bad && status) atomicOr(status + row, GUFFIN_STATUS_NONFINITE);
    bitonic_desc(keys, kTile);
    uint64_t* out = survivors + (size_t(row) * gridDim.x + tile) * keep;
    for (uint32_t i = threadIdx.x; i < keep; i += blockDim.x) out[i] = keys[i];
}

struct Candidates {  // layout of one row of the result (sampling.hpp:57-61 plus a status word)
    uint32_t count;
    uint32_t status;
    struct { uint32_t token; float logit; } values[384];
};

// Adds one to hist[bin] for every lane with `valid`; lanes of a wave that hit the same bin are
// counted with one atomic (keys cluster in a few bins, and same-address LDS atomics serialise).  (The leader's bin read into a
// scalar register instead: 9.5 us for the 8.8 of threshold_select_kernel, 1018 for the 920 of its walk over a whole row.)
__device__ __forceinline__ void hist_add(uint32_t* hist, bool valid, uint32_t bin, uint32_t lane) {
    uint64_t todo = __ballot(valid);
    for (int it = 0; it < 8 && todo; ++it) {
        const int leader = __ffsll(static_cast<long long>(todo)) - 1;
        const uint32_t b0 = __shfl(bin, leader, kWave);
        const uint64_t same = __ballot(valid && bin == b0) & todo;
        if (lane == uint32_t(leader)) atomicAdd(&hist[b0], static_cast<uint32_t>(__popcll(same)));
        todo &= ~same;
    }
    if ((todo >> lane) & 1u) atomicAdd(&hist[bin], 1u);
}

// The same where the bins were made to spread the words: lanes of one wave rarely share one, and each counts for itself.
__device__ __forceinline__ void hist_add_spread(uint32_t* hist, bool valid, uint32_t bin, uint32_t lane) {
    const uint64_t live = __ballot(valid);
    if (!live) return;
    const uint32_t first = __builtin_amdgcn_readlane(bin, __ffsll(static_cast<long long>(live)) - 1);
    if (__popcll(__ballot(valid && bin == first)) > 8) hist_add(hist, valid, bin, lane);
    else if (valid) atomicAdd(&hist[bin], 1u);
}

// Writes one row of the result from its `retain` selected keys (candidate order) and appends the logits of
// the row's history tokens; all threads of the workgroup call it after the keys are complete.  raised: the row's status word;
// whole: the record is new memory, what it does not use becomes zero.
__device__ void emit_candidates(const uint64_t* keys, uint32_t retain, uint32_t row, const float* __restrict__ logits,
                                uint32_t vocab, float divisor, const uint32_t* __restrict__ history,
                                uint32_t hc, uint32_t history_stride, uint32_t raised, bool whole,
                                Candidates* __restrict__ result, uint32_t* __restrict__ status) {
    __syncthreads();
    Candidates& out = result[row];
    for (uint32_t i = threadIdx.x; i < retain; i += blockDim.x) {
        const uint32_t token = key_token(keys[i]);
        // the key holds the value's bits but for a zero's sign and what adding zero does to a NaN: those are read again
        float v = key_logit(keys[i]);
        if (!(v < 0.f || v > 0.f)) v = logits[size_t(row) * vocab + token] / divisor;
        out.values[i].token = token;
        out.values[i].logit = v;
    }
    if (whole)
        for (uint32_t i = retain + hc + threadIdx.x; i < 384; i += blockDim.x) { out.values[i].token = 0; out.values[i].logit = 0.f; }
    uint32_t st = 0;
    for (uint32_t i = threadIdx.x; i < hc; i += blockDim.x) {
        const uint32_t token = history[size_t(row) * history_stride + i];
        if (token >= vocab) {
            st |= GUFFIN_STATUS_BAD_TOKEN;
            out.values[retain + i].token = 0xFFFFFFFFu;
            out.values[retain + i].logit = -INFINITY;
        } else {
            const float v = logits[size_t(row) * vocab + token] / divisor;
            if (!isfinite(v)) st |= GUFFIN_STATUS_NONFINITE;
            out.values[retain + i].token = token;
            out.values[retain + i].logit = v;
        }
    }
    if (st && status) atomicOr(status + row, st);
    if (hc && status) {
        raised |= __syncthreads_or(st & GUFFIN_STATUS_BAD_TOKEN) ? GUFFIN_STATUS_BAD_TOKEN : 0u;
        raised |= __syncthreads_or(st & GUFFIN_STATUS_NONFINITE) ? GUFFIN_STATUS_NONFINITE : 0u;
    }
    if (threadIdx.x == 0) {
        out.count = retain + hc;
        out.status = raised;
    }
}

// Stage 2: exact selection of the best `retain` of n unique keys.  Sorted tile lists take the
// threshold shortcut below; otherwise an 8-pass radix select (one byte per pass, most significant
// first: a 256-bin histogram in LDS, then the bin that holds the retain-th largest key).  Either
// way a rank sort of the selected keys follows.
template <int kMine>
__global__ void __launch_bounds__(1024)
topk_merge_kernel(const float* __restrict__ logits, const uint64_t* __restrict__ survivors, uint32_t n_survivors,
                  uint32_t tile_keep, uint32_t vocab, uint32_t retain_cap, float divisor, const uint32_t* __restrict__ history,
                  const uint32_t* __restrict__ history_count, const uint32_t* __restrict__ row_retain, uint32_t row_stride,
                  uint32_t history_stride, bool whole, Candidates* __restrict__ result, uint32_t* __restrict__ status) {
    __shared__ uint32_t hist[256];
    __shared__ uint64_t sel[512];
    __shared__ uint64_t keys[512];  // selected keys in candidate order
    __shared__ uint32_t s_bin, s_above, s_count, s_in_bin;
    __shared__ uint64_t floor_key;
    const uint32_t row = blockIdx.x, lane = threadIdx.x & 63;
    // a row may ask for fewer than the launch's capacity (top_k plus ITS history count); history_count
    // and row_retain are read `row_stride` words apart (1, or the stride of a resolved-request record)
    uint32_t retain = retain_cap;
    if (row_retain) {
        const uint32_t want = row_retain[size_t(row) * row_stride];
        retain = want < 1 ? 1 : (want < retain_cap ? want : retain_cap);
    }
    const uint32_t hc = history_count ? history_count[size_t(row) * row_stride] : 0, raised = status ? status[row] : 0;
    const uint64_t* src = survivors + size_t(row) * n_survivors;
    // up to kMine keys per thread stay in registers (8 for the verify pass's lists, 34 for the 257 per
    // tile that the proposal law asks for); longer survivor lists are re-read from memory in every pass
    const bool cached = n_survivors <= kMine * blockDim.x;
    uint64_t mine[kMine];
#pragma unroll
    for (int u = 0; u < kMine; ++u) {
        const uint32_t i = threadIdx.x + u * blockDim.x;
        mine[u] = cached && i < n_survivors ? src[i] : 0;
    }
    // Shortcut for sorted tile lists (tile_keep > 0: the survivors are `tiles` descending lists of tile_keep
    // keys): the retain-th largest of the tiles' first r keys (tiles * r >= retain of them) is a lower bound
    // of the retain-th largest key overall, so only keys at or above it can be selected.  They are few (a
    // little over `retain` unless the logits tie massively); a rank sort of them is the exact answer.
    bool done = false;
    if (cached && tile_keep > 0) {
        const uint32_t tiles = n_survivors / tile_keep;
        const uint32_t r = (retain + tiles - 1) / tiles;
        const uint32_t heads = tiles * r;
        if (r <= tile_keep && heads <= 512) {
            for (uint32_t i = threadIdx.x; i < heads; i += blockDim.x) sel[i] = src[(i / r) * tile_keep + i % r];
            if (threadIdx.x == 0) { s_count = 0; floor_key = 0; }   // a floor of zero lets every key through
            __syncthreads();
            for (uint32_t i = threadIdx.x; i < heads; i += blockDim.x) {
                const uint64_t k = sel[i];
                uint32_t rank = 0;
                for (uint32_t j = 0; j < heads; ++j) rank += sel[j] > k;
                if (rank == retain - 1) floor_key = k;   // real keys are unique; only the zero padding repeats
            }
            __syncthreads();
            const uint64_t bound = floor_key;
            __syncthreads();
#pragma unroll
            for (int u = 0; u < kMine; ++u) {
                if (threadIdx.x + u * blockDim.x < n_survivors && mine[u] >= bound) {
                    const uint32_t at = atomicAdd(&s_count, 1u);
                    if (at < 512) sel[at] = mine[u];
                }
            }
            __syncthreads();
            const uint32_t n = s_count;
            if (n <= 512) {   // else: too many ties at the bound, the general path below decides
                for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
                    const uint64_t k = sel[i];
                    uint32_t rank = 0;
                    for (uint32_t j = 0; j < n; ++j) rank += sel[j] > k;
                    if (rank < retain) keys[rank] = k;
                }
                done = true;
            }
            __syncthreads();
        }
    }
    if (!done) {
        uint64_t prefix = 0;
        uint32_t remaining = retain;  // rank of the wanted key among the keys that match `prefix`
        for (int pass = 0; pass < 8; ++pass) {
            const int shift = 56 - 8 * pass;
            for (uint32_t i = threadIdx.x; i < 256; i += blockDim.x) hist[i] = 0;
            __syncthreads();
            if (cached) {
    #pragma unroll
                for (int u = 0; u < kMine; ++u) {
                    const uint64_t k = mine[u];
                    hist_add(hist, threadIdx.x + u * blockDim.x < n_survivors && (pass == 0 || (k >> (shift + 8)) == prefix),
                             static_cast<uint32_t>(k >> shift) & 255u, lane);
                }
            } else {
                for (uint32_t i0 = 0; i0 < n_survivors; i0 += blockDim.x) {  // whole waves stay converged
                    const uint32_t i = i0 + threadIdx.x;
                    const uint64_t k = i < n_survivors ? src[i] : 0;
                    hist_add(hist, i < n_survivors && (pass == 0 || (k >> (shift + 8)) == prefix),
                             static_cast<uint32_t>(k >> shift) & 255u, lane);
                }
            }
            __syncthreads();
            if (threadIdx.x < 64) {  // lane l owns bins 255-4l .. 252-4l, highest first
                uint32_t c[4];
    #pragma unroll
                for (int j = 0; j < 4; ++j) c[j] = hist[255 - 4 * lane - j];
                const uint32_t own = c[0] + c[1] + c[2] + c[3];
                const uint32_t incl = wave_inclusive_scan(own);
                uint32_t above = incl - own;
                if (above < remaining && remaining <= incl) {
    #pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        if (remaining <= above + c[j]) { s_bin = 255 - 4 * lane - j; s_above = above; s_in_bin = c[j]; break; }
                        above += c[j];
                    }
                }
            }
            __syncthreads();
            prefix = (prefix << 8) | s_bin;
            remaining -= s_above;
            // the upper 32 bits are the logit: if every key that shares the threshold logit is wanted
            // (no tie across the cut), the token bits need no passes
            if (pass == 3 && s_in_bin == remaining) { prefix <<= 32; remaining = 0; break; }
        }
        // `prefix` is the retain-th largest key; keys above it are taken, then `remaining` copies of it
        // (more than one only for the zero padding of a short last tile)
        if (threadIdx.x == 0) s_count = 0;
        __syncthreads();
        if (cached) {
    #pragma unroll
            for (int u = 0; u < kMine; ++u)
                if (threadIdx.x + u * blockDim.x < n_survivors && mine[u] > prefix) sel[atomicAdd(&s_count, 1u)] = mine[u];
        } else {
            for (uint32_t i = threadIdx.x; i < n_survivors; i += blockDim.x) {
                const uint64_t k = src[i];
                if (k > prefix) sel[atomicAdd(&s_count, 1u)] = k;
            }
        }
        __syncthreads();
        const uint32_t above_total = s_count;
        for (uint32_t i = threadIdx.x; i < remaining; i += blockDim.x) sel[above_total + i] = prefix;
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < retain; i += blockDim.x) {
            const uint64_t k = sel[i];
            uint32_t rank = 0;
            for (uint32_t j = 0; j < retain; ++j) {
                const uint64_t o = sel[j];
                rank += (o > k) || (o == k && j < i);
            }
            keys[rank] = k;
        }
    }
    emit_candidates(keys, retain, row, logits, vocab, divisor, history, hc, history_stride, raised, whole, result, status);
}

// ---- selection by threshold ------------------------------------------------------------------
// For large vocabularies the sort of every tile is more work than the answer needs.  The maxima of the
// 256-logit segments give a bound first: with at least `retain` segments, the retain-th largest segment
// maximum is at or below the retain-th largest logit of the row, so only logits at or above it can be
// selected, and on anything but massively tied rows they are few more than `retain`.  Two launches:
//   segment_max_kernel       the ordered score bits of every segment's maximum; clears the row's counters
//   threshold_select_kernel  every workgroup finds the bound for itself (a radix select over at most 1024
//                            words that stops as soon as few maxima lie between it and the exact one),
//                            collects the keys of its 4096 logits that reach it, and the workgroup that
//                            finishes last sorts all of them and writes the row
// A caller that needs the best `sure` logits and every tie with the last of them, and as many of the following
// (up to `retain`) as come with these, passes `sure` != 0: the bound is then the one for `sure`.
// What bounds the second launch is the chain of trips to memory behind one another (the workgroups sit on different
// L2s, so what they exchange moves with device-scope accesses).  A workgroup therefore has places of its own
// for kSlots keys and its count, stored without asking anybody; only what does not fit goes through a
// reservation in the row's common list, and the last workgroup asks for counts and places at once.  Its
// logits lie 64 apart from its neighbours', so that a run of equal or large ones is dealt to all.  Every
// workgroup waits for its own stores before it counts itself done, and nobody waits for anybody: the last
// arrival is whoever draws the last ticket.  Up to kCollectCap keys of a row are sorted in LDS, however they
// lie: the common list holds what the places of a single collector leave of that many.  A row with more is
// selected exactly, and slowly, by a radix select over the whole row in that workgroup.
// 262144 logits: 64 of two rows 6.8 us (an exact bound and every key through one reservation cost 1.8 more), a compact law of 64
// and its proposal 10.5.  Ties, both launches and the call: 300 to 2000 keys 18 to 29 us,
// beyond 2048 keys 920.
constexpr uint32_t kSeg = 256, kMaxSegs = 1024, kCollectTile = 4096, kCollectCap = 2048;
struct Nothing {};
// large vocabularies, where the segment maxima give a bound for the best `keep` logits
bool by_threshold(uint32_t vocab, uint32_t keep) {
    const uint32_t segs = (vocab + kSeg - 1) / kSeg;
    return segs <= kMaxSegs && segs >= 2 * keep;
}
constexpr uint32_t kMaxCollectors = kMaxSegs * kSeg / kCollectTile, kSlots = 16, kCommonCap = kCollectCap - kSlots;
// segment maxima; common list's length, workgroups done, pad; the workgroups' counts, their places, the common list
constexpr uint32_t kThresholdRowWords = kMaxSegs + 4 + kMaxCollectors + 2 * (kMaxCollectors * kSlots + kCommonCap);
static_assert((kMaxSegs + 4 + kMaxCollectors) % 2 == 0 && kThresholdRowWords % 2 == 0, "keys on 8 bytes");
static_assert(kMaxCollectors == 64, "a wave scans the workgroups' counts");

__device__ __forceinline__ uint32_t ordered_bits(float v) {
    const uint32_t b = __float_as_uint(v + 0.0f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

__global__ void __launch_bounds__(256)
segment_max_kernel(const float* __restrict__ logits, uint32_t vocab, uint32_t segs, float divisor, uint32_t* __restrict__ ws,
                   uint32_t* __restrict__ new_status) {
    const uint32_t row = blockIdx.y, lane = threadIdx.x & 63;
    const uint32_t seg = blockIdx.x * 4 + (threadIdx.x >> 6);
    uint32_t* row_ws = ws + size_t(row) * kThresholdRowWords;
    if (blockIdx.x == 0 && threadIdx.x < 4) row_ws[kMaxSegs + threadIdx.x] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 4 && new_status) new_status[row] = 0;
    if (seg >= segs) return;
    const float* lr = logits + size_t(row) * vocab;
    uint32_t best = 0;
#pragma unroll
    for (uint32_t u = 0; u < kSeg / 64; ++u) {
        const uint32_t t = seg * kSeg + u * 64 + lane;
        if (t < vocab) {
            const uint32_t o = ordered_bits(divisor == 1.f ? lr[t] : lr[t] / divisor);
            best = o > best ? o : best;
        }
    }
    best = wave_max_u32(best);
    if (lane == 0) row_ws[seg] = best;
}

// the bin (highest first) that holds the `remaining`-th largest entry of a 256-bin histogram; first wave only
__device__ __forceinline__ void find_bin(const uint32_t* hist, uint32_t remaining, uint32_t lane, uint32_t& s_bin,
                                         uint32_t& s_above, uint32_t& s_in) {
    uint32_t c[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) c[j] = hist[255 - 4 * lane - j];
    const uint32_t own = c[0] + c[1] + c[2] + c[3];
    const uint32_t incl = wave_inclusive_scan(own);
    uint32_t above = incl - own;
    if (above < remaining && remaining <= incl) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (remaining <= above + c[j]) { s_bin = 255 - 4 * lane - j; s_above = above; s_in = c[j]; break; }
            above += c[j];
        }
    }
}

template <typename T>
__device__ __forceinline__ T shared_load(const T* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename T>
__device__ __forceinline__ void shared_store(T* p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

template <bool LAW>
__global__ void __launch_bounds__(1024)
threshold_select_kernel(const float* __restrict__ logits, uint32_t* __restrict__ ws, uint32_t vocab, uint32_t segs, uint32_t retain_cap,
                        uint32_t sure, float divisor, uint32_t row_stride, const uint32_t* __restrict__ history_count,
                        const uint32_t* __restrict__ row_retain, const uint32_t* __restrict__ history, uint32_t history_stride,
                        Candidates* __restrict__ result, uint32_t* __restrict__ status, bool suppressed_ok, bool whole, std::conditional_t<LAW, LawCall, Nothing> law) {
    __shared__ uint32_t hist[256];
    __shared__ uint64_t sel[kCollectCap];
    __shared__ uint64_t keys[512];
    __shared__ uint32_t s_bin, s_above, s_in, s_last, s_count;
    __shared__ uint32_t s_low[16], s_top[16];   // the waves' least (inverted) and largest maxima
    const uint32_t row = blockIdx.y, tid = threadIdx.x, lane = tid & 63, collectors = (vocab + kCollectTile - 1) / kCollectTile;
    uint32_t* row_ws = ws + size_t(row) * kThresholdRowWords;
    uint32_t* counter = row_ws + kMaxSegs;
    uint32_t* done = counter + 1;
    uint32_t* counts = counter + 4;
    uint64_t* places = reinterpret_cast<uint64_t*>(counts + kMaxCollectors);
    uint64_t* common = places + kMaxCollectors * kSlots;
    const float* lr = logits + size_t(row) * vocab;
    // this workgroup's logits are requested before the bound is worked out
    auto token_of = [&](uint32_t u) { return ((u * (1024 / 64) + (tid >> 6)) * collectors + blockIdx.x) * 64 + lane; };
    float mine[kCollectTile / 1024];
#pragma unroll
    for (uint32_t u = 0; u < kCollectTile / 1024; ++u) mine[u] = token_of(u) < vocab ? lr[token_of(u)] : 0.f;
    const uint32_t word = tid < segs ? row_ws[tid] : 0u;
    uint32_t retain = retain_cap;
    if (row_retain) {
        const uint32_t want = row_retain[size_t(row) * row_stride];
        retain = want < 1 ? 1 : (want < retain_cap ? want : retain_cap);
    }
    const uint32_t hc = history_count ? history_count[size_t(row) * row_stride] : 0;
    // ---- the bound: at or below the largest segment maximum but `least` - 1 (there are as many by the launch's condition), with
    // no more than an eighth of `least` maxima too many above it; every further byte would cost a pass, most rows stop after two
    // The first pass has 256 bins between the least and the largest maximum: maxima are alike, and the top byte of their bits says
    // next to nothing.  (Passes from the top byte down, equal bins counted by one lane: 64 of two rows 8.8 us, so 6.8.)
    const uint32_t least = sure ? sure : retain;
    const uint32_t wave_top = wave_max_u32(tid < segs ? word : 0u), wave_low = wave_max_u32(tid < segs ? ~word : 0u);
    if (lane == 0) { s_top[tid >> 6] = wave_top; s_low[tid >> 6] = wave_low; }
    if (tid < 256) hist[tid] = 0;
    if (tid == 0) s_count = 0;
    __syncthreads();
    auto of_waves = [](uint32_t v) {   // the largest of sixteen, in every lane
        v = max(v, lane_cross_u32<0xB1, 0xF>(v));
        v = max(v, lane_cross_u32<0x4E, 0xF>(v));
        v = max(v, lane_cross_u32<0x141, 0xF>(v));
        v = max(v, lane_cross_u32<0x140, 0xF>(v));
        return __builtin_amdgcn_readfirstlane(v);
    };
    const uint32_t top = of_waves(s_top[lane & 15u]);
    uint32_t bound = ~of_waves(s_low[lane & 15u]);   // the lower edge of bin 0, then of the bin that was found
    uint32_t remaining = least, bins = 256u, shift = top > bound ? 24u - min(24u, static_cast<uint32_t>(__clz(static_cast<int>(top - bound)))) : 0u;
    for (;;) {
        const uint32_t bin = (word - bound) >> shift;
        hist_add_spread(hist, tid < segs && word >= bound && bin < bins, bin, lane);
        __syncthreads();
        if (tid < 64) find_bin(hist, remaining, lane, s_bin, s_above, s_in);
        __syncthreads();
        bound += s_bin << shift;
        remaining -= s_above;
        if (shift == 0 || s_in - remaining <= least / 8) break;
        const uint32_t finer = shift > 8 ? shift - 8 : 0u;
        bins = 1u << (shift - finer);
        shift = finer;
        if (tid < 256) hist[tid] = 0;
        __syncthreads();
    }
    // ---- collect: this workgroup's keys into LDS, then into its places and, past them, the row's common list ----
    bool bad = false;
    auto collect = [&](auto scaled) {   // (sixteen waves and exact division: dividing by one is not free)
#pragma unroll
        for (uint32_t u = 0; u < kCollectTile / 1024; ++u) {
            const uint32_t t = token_of(u);
            if (t < vocab) {
                const float v = scaled(mine[u]);
                bad |= (!isfinite(v) || !isfinite(mine[u])) && !(suppressed_ok && mine[u] == -INFINITY);
                if (ordered_bits(v) >= bound) {
                    const uint32_t at = atomicAdd(&s_count, 1u);
                    if (at < kCollectCap) sel[at] = make_key(v, t);
                }
            }
        }
    };
    if (divisor == 1.f) collect([](float x) { return x; });
    else collect([&](float x) { return x / divisor; });
    __syncthreads();
    const uint32_t found = s_count;
    if (tid < kSlots && tid < found) shared_store(places + blockIdx.x * kSlots + tid, sel[tid]);
    if (tid == kSlots) shared_store(counts + blockIdx.x, found);
    if (found > kSlots) {
        const uint32_t more = found - kSlots;   // beyond the list: the row's counter shows it too, and nobody reads the list
        if (tid == 0) s_bin = __hip_atomic_fetch_add(counter, more, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        for (uint32_t i = tid; i < min(more, kCommonCap); i += 1024)
            if (s_bin + i < kCommonCap) shared_store(common + s_bin + i, sel[kSlots + i]);
    }
    if (bad && status) atomicOr(status + row, GUFFIN_STATUS_NONFINITE);
    // ---- the last workgroup of the row to get here finishes it -----------------------------------------
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) {
        const uint32_t before = __hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = before + 1 == collectors;
        s_count = 0;
    }
    __syncthreads();
    if (!s_last) return;
    // every wave scans the counts for itself; a thread takes one place
    const uint32_t count = lane < collectors ? shared_load(counts + lane) : 0;
    const uint32_t owner = tid / kSlots, raised = status ? shared_load(status + row) : 0;
    const uint64_t place = owner < collectors ? shared_load(places + tid) : 0;   // its collector may have left it as it was
    const uint32_t kept = min(count, kSlots), upto = wave_inclusive_scan(kept), all = wave_inclusive_scan(count);
    const uint32_t n = __builtin_amdgcn_readlane(all, 63), placed = __builtin_amdgcn_readlane(upto, 63);
    const uint32_t own_kept = __shfl(kept, owner, kWave), own_upto = __shfl(upto, owner, kWave);
    static_assert(kMaxCollectors * kSlots == 1024, "a place per thread");
    if (n <= kCollectCap) {
        if (tid % kSlots < own_kept) sel[own_upto - own_kept + tid % kSlots] = place;
        for (uint32_t i = tid; i < n - placed; i += 1024) sel[placed + i] = shared_load(common + i);
        if (n <= 512) {
            __syncthreads();
            // the workgroup's 1024 threads over n keys: 2, 4, 8 or 16 neighbouring lanes count for one of them
            const uint32_t part_bits = n <= 64 ? 4 : n <= 128 ? 3 : n <= 256 ? 2 : 1, i = tid >> part_bits, part = tid & ((1u << part_bits) - 1);
            const uint64_t k = i < n ? sel[i] : 0;
            uint32_t rank = 0;
#pragma unroll 8
            for (uint32_t j = part; j < n; j += 1u << part_bits) rank += sel[j] > k;
            rank += lane_cross_u32<0xB1, 0xF>(rank);                        // the neighbour,
            if (part_bits >= 2) rank += lane_cross_u32<0x4E, 0xF>(rank);    // the pair, the four, the eight beside
            if (part_bits >= 3) rank += lane_cross_u32<0x141, 0xF>(rank);
            if (part_bits >= 4) rank += lane_cross_u32<0x140, 0xF>(rank);
            if (i < n && part == 0 && rank < retain) keys[rank] = k;
            retain = min(retain, n);   // fewer only where the call is sure of fewer
        } else {
            for (uint32_t i = n + tid; i < kCollectCap; i += 1024) sel[i] = 0;
            bitonic_desc(sel, kCollectCap);
            for (uint32_t i = tid; i < retain; i += 1024) keys[i] = sel[i];
        }
    } else {
        // more ties than the list holds: an 8-pass radix select over the whole row's keys, exact and slow
        uint64_t kprefix = 0;
        uint32_t left = retain;
        for (int pass = 0; pass < 8; ++pass) {
            const int down = 56 - 8 * pass;
            if (tid < 256) hist[tid] = 0;
            __syncthreads();
            for (uint32_t i0 = 0; i0 < vocab; i0 += 1024) {   // whole waves stay converged
                const uint32_t i = i0 + tid;
                const uint64_t k = i < vocab ? make_key(lr[i] / divisor, i) : 0;
                hist_add(hist, i < vocab && (pass == 0 || (k >> (down + 8)) == kprefix), static_cast<uint32_t>(k >> down) & 255u, lane);
            }
            __syncthreads();
            if (tid < 64) find_bin(hist, left, lane, s_bin, s_above, s_in);
            __syncthreads();
            kprefix = (kprefix << 8) | s_bin;
            left -= s_above;
        }
        // kprefix is the retain-th largest key (keys are unique): everything above it, then it
        for (uint32_t i = tid; i < vocab; i += 1024) {
            const uint64_t k = make_key(lr[i] / divisor, i);
            if (k >= kprefix) sel[atomicAdd(&s_count, 1u)] = k;
        }
        __syncthreads();
        for (uint32_t i = tid; i < retain; i += 1024) {
            const uint64_t k = sel[i];
            uint32_t rank = 0;
            for (uint32_t j = 0; j < retain; ++j) rank += sel[j] > k;
            keys[rank] = k;
        }
    }
    if constexpr (LAW) {
        __syncthreads();
        if (tid >= 256) return;   // a law is four waves' work: the meetings are theirs from here on
        auto logit_of = [&](uint32_t i) {   // as emit_candidates has it
            const float v = key_logit(keys[i]);
            return v < 0.f || v > 0.f ? v : lr[key_token(keys[i])] / divisor;
        };
        const bool mine_too = tid < retain;
        compact_law(law, retain, raised, mine_too ? key_token(keys[tid]) : 0u, mine_too ? logit_of(tid) : 0.f, retain > 256 ? logit_of(256) : 0.f);
    } else {
        emit_candidates(keys, retain, row, logits, vocab, divisor, history, hc, history_stride, raised, whole, result, status);
    }
}

__global__ void clear_words_kernel(uint32_t* words, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) words[i] = 0;
}

// ---- verify-row input validation --------------------------------------------------------------
__global__ void input_validation_kernel(const uint32_t* __restrict__ actual, const uint32_t* __restrict__ expected,
                                        uint32_t rows, uint32_t vocab, uint32_t* __restrict__ status) {
    const uint32_t row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row < rows && (actual[row] >= vocab || actual[row] != expected[row])) atomicOr(status, GUFFIN_STATUS_BAD_TOKEN);
}

// ---- selection requests --------------------------------------------------------------------
// One wave per row: the raw ring and suffix become the resolved record and the row's history list.
__global__ void __launch_bounds__(64)
selection_requests_kernel(const SelectionRow* __restrict__ raw, uint32_t vocab, uint32_t top_k, uint32_t repetition,
                          ResolvedRow* __restrict__ resolved, uint32_t* __restrict__ histories,
                          uint32_t* __restrict__ status) {
    const uint32_t row = blockIdx.x, lane = threadIdx.x;
    const SelectionRow& r = raw[row];
    uint32_t token = 0, st = 0;
    const uint32_t count = resolve_history(r.history_token_ids, r.history_head, r.history_length, r.history_window_limit,
                                           r.suffix_token_ids, r.suffix_count, vocab, repetition != 0, lane, token, st);
    ResolvedRow& out = resolved[row];
    out.history_token_ids[lane] = token;
    if (histories) histories[size_t(row) * kRequestHistory + lane] = token;
    if (lane == 0) {
        out.top_k = top_k;
        out.base_candidate_count = top_k + count;
        out.history_count = count;
        out.reserved = 0;
        if (st && status) atomicOr(status, st);
    }
}

// ---- greedy argmax ---------------------------------------------------------------------
__global__ void __launch_bounds__(256)
argmax_tile_kernel(const float* __restrict__ logits, uint64_t* __restrict__ partial, uint32_t vocab,
                   uint32_t* __restrict__ status) {
    __shared__ uint64_t best[4];
    const uint32_t row = blockIdx.y;
    const float* lr = logits + size_t(row) * vocab;
    uint64_t k = 0;
    bool bad = false;
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < vocab; t += gridDim.x * blockDim.x) {
        const float v = lr[t];
        bad |= !isfinite(v);
        const uint64_t c = make_key(v, t);
        k = c > k ? c : k;
    }
    if (bad && status) atomicOr(status + row, GUFFIN_STATUS_NONFINITE);
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        const uint64_t o = __shfl_xor(k, s, kWave);
        k = o > k ? o : k;
    }
    if ((threadIdx.x & 63) == 0) best[threadIdx.x >> 6] = k;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < 4; ++i) k = best[i] > k ? best[i] : k;
        partial[size_t(row) * gridDim.x + blockIdx.x] = k;
    }
}

__global__ void __launch_bounds__(256)
argmax_final_kernel(const uint64_t* __restrict__ partial, uint32_t n, uint32_t* __restrict__ token,
                    float* __restrict__ logit) {
    __shared__ uint64_t best[4];
    const uint32_t row = blockIdx.x;
    uint64_t k = 0;
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
        const uint64_t c = partial[size_t(row) * n + i];
        k = c > k ? c : k;
    }
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        const uint64_t o = __shfl_xor(k, s, kWave);
        k = o > k ? o : k;
    }
    if ((threadIdx.x & 63) == 0) best[threadIdx.x >> 6] = k;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < 4; ++i) k = best[i] > k ? best[i] : k;
        token[row] = key_token(k);
        if (logit) logit[row] = key_logit(k);
    }
}

}  // namespace

int head_init() { return 0; }

}  // namespace guffin

using namespace guffin;

extern "C" uint64_t guffin_hip_select_workspace_bytes(uint32_t rows, uint32_t vocab, uint32_t retain) {
    const uint64_t tiles = (uint64_t(vocab) + kTile - 1) / kTile;
    const uint64_t keep = retain < kTile ? retain : kTile;
    const uint64_t sorted_tiles = rows * tiles * keep * 8, by_threshold = uint64_t(rows) * kThresholdRowWords * 4;
    return sorted_tiles > by_threshold ? sorted_tiles : by_threshold;   // either path may serve the call
}

namespace guffin {
int select_candidates_scaled(hipStream_t s, const float* logits, uint32_t rows, uint32_t vocab, uint32_t retain,
                             float divisor, const uint32_t* history, const uint32_t* history_count,
                             void* workspace, void* result, uint32_t* status, bool suppressed_ok = false,
                             const uint32_t* row_retain = nullptr, uint32_t row_stride = 1, uint32_t sure = 0, bool fresh = false);
}

extern "C" int guffin_hip_select_candidates_fresh(void* stream, const float* logits, uint32_t rows, uint32_t vocab,
                                                  uint32_t retain, const uint32_t* history, const uint32_t* history_count,
                                                  void* workspace, void* result, uint32_t* status) {
    if (!status) return fail(GUFFIN_E_ARG, "select_candidates_fresh: null pointer");
    return select_candidates_scaled(as_stream(stream), logits, rows, vocab, retain, 1.0f, history, history_count,
                                    workspace, result, status, false, nullptr, 1, 0, true);
}

extern "C" int guffin_hip_select_candidates(void* stream, const float* logits, uint32_t rows, uint32_t vocab,
                                            uint32_t retain, const uint32_t* history, const uint32_t* history_count,
                                            void* workspace, void* result, uint32_t* status) {
    return select_candidates_scaled(as_stream(stream), logits, rows, vocab, retain, 1.0f, history, history_count,
                                    workspace, result, status);
}

int guffin::select_candidates_scaled(hipStream_t s, const float* logits, uint32_t rows, uint32_t vocab,
                                     uint32_t retain, float divisor, const uint32_t* history,
                                     const uint32_t* history_count, void* workspace, void* result, uint32_t* status,
                                     bool suppressed_ok, const uint32_t* row_retain, uint32_t row_stride, uint32_t sure, bool fresh) {
    if (!logits || !workspace || !result) return fail(GUFFIN_E_ARG, "select_candidates: null pointer");
    if (rows == 0 || vocab == 0) return fail(GUFFIN_E_SHAPE, "select_candidates: empty shape");
    if (retain == 0 || retain > 320) return fail(GUFFIN_E_CAPACITY, "select_candidates: retain must be in [1, 320] (top_k <= 256 plus 64 history tokens)");
    if ((history == nullptr) != (history_count == nullptr)) return fail(GUFFIN_E_ARG, "select_candidates: history and its counts come together");
    if (reinterpret_cast<uintptr_t>(workspace) & 7u) return fail(GUFFIN_E_ALIGN, "select_candidates: workspace must be 8-byte aligned");
    const uint32_t keep = retain < vocab ? retain : vocab;
    const uint32_t tiles = (vocab + kTile - 1) / kTile;
    const uint32_t segs = (vocab + kSeg - 1) / kSeg;
    if (by_threshold(vocab, keep)) {   // large vocabulary: a bound from the segment maxima, then one pass
        uint32_t* words = static_cast<uint32_t*>(workspace);
        launch(segment_max_kernel, dim3((segs + 3) / 4, rows), dim3(256), 0, s, logits, vocab, segs, divisor, words,
               fresh ? status : nullptr);
        if (int rc = check_launch("select_candidates(segment maxima)")) return rc;
        launch(threshold_select_kernel<false>, dim3((vocab + kCollectTile - 1) / kCollectTile, rows), dim3(1024), 0, s,
                           logits, words, vocab, segs, keep, sure, divisor, row_stride, history_count, row_retain, history,
                           row_stride == 1 ? 64u : row_stride, static_cast<Candidates*>(result), status, suppressed_ok, fresh, Nothing {});
        return check_launch("select_candidates(threshold)");
    }
    if (fresh) launch(clear_words_kernel, dim3((rows + 63) / 64), dim3(64), 0, s, status, rows);
    uint64_t* surv = static_cast<uint64_t*>(workspace);
    launch(topk_tile_kernel, dim3(tiles, rows), dim3(1024), 0, s, logits, surv, vocab, keep, divisor, status, suppressed_ok);
    if (int rc = check_launch("select_candidates(tile)")) return rc;
    if (tiles * keep <= 8 * 1024)
        launch(topk_merge_kernel<8>, dim3(rows), dim3(1024), 0, s, logits, surv, tiles * keep, keep, vocab,
                           keep, divisor, history, history_count, row_retain, row_stride, row_stride == 1 ? 64u : row_stride,
                           fresh, static_cast<Candidates*>(result), status);
    else
        launch(topk_merge_kernel<34>, dim3(rows), dim3(1024), 0, s, logits, surv, tiles * keep, keep, vocab,
                           keep, divisor, history, history_count, row_retain, row_stride, row_stride == 1 ? 64u : row_stride,
                           fresh, static_cast<Candidates*>(result), status);
    return check_launch("select_candidates(merge)");
}

// A law is decided where its selection ends: the workgroup that sorts a row's keys goes on with them, and the record, its trip and a
// launch fall away (one row of 262144, 64 kept: 9.0 + 7.1 us and the boundary between them are 15.7; with all sixteen waves in the law's
// meetings 16.7).  Other vocabularies are selected by tiles, their law a launch of its own.
bool guffin::selection_makes_laws(uint32_t vocab, uint32_t retain) { return vocab >= retain && by_threshold(vocab, retain); }

int guffin::select_law(hipStream_t s, const float* logits, uint32_t vocab, uint32_t retain, uint32_t sure, void* workspace, const LawCall& law,
                       bool suppressed_ok) {
    if (reinterpret_cast<uintptr_t>(workspace) & 7u) return fail(GUFFIN_E_ALIGN, "select_candidates: workspace must be 8-byte aligned");
    const uint32_t segs = (vocab + kSeg - 1) / kSeg;
    const float divisor = law.opt.temperature;
    uint32_t* words = static_cast<uint32_t*>(workspace);
    launch(segment_max_kernel, dim3((segs + 3) / 4, 1), dim3(256), 0, s, logits, vocab, segs, divisor, words, law.whole ? law.status : nullptr);
    if (int rc = check_launch("draft_law(segment maxima)")) return rc;
    launch(threshold_select_kernel<true>, dim3((vocab + kCollectTile - 1) / kCollectTile, 1), dim3(1024), 0, s, logits, words, vocab, segs, retain,
           sure, divisor, 1u, nullptr, nullptr, nullptr, 64u, nullptr, law.status, suppressed_ok, law.whole != 0, law);
    return check_launch("draft_law(threshold)");
}

extern "C" int guffin_hip_input_validation(void* stream, const uint32_t* actual, const uint32_t* expected, uint32_t rows,
                                           uint32_t vocab, uint32_t* status) {
    if (!actual || !expected || !status) return fail(GUFFIN_E_ARG, "input_validation: null pointer");
    if (rows == 0 || vocab == 0) return fail(GUFFIN_E_SHAPE, "input_validation: empty shape");
    launch(input_validation_kernel, dim3((rows + 63) / 64), dim3(64), 0, as_stream(stream), actual, expected,
                       rows, vocab, status);
    return check_launch("input_validation");
}

extern "C" int guffin_hip_selection_requests(void* stream, const void* raw, uint32_t rows, uint32_t vocab, uint32_t top_k,
                                             uint32_t repetition_enabled, void* resolved, uint32_t* histories,
                                             uint32_t* status) {
    if (!raw || !resolved) return fail(GUFFIN_E_ARG, "selection_requests: null pointer");
    if (rows == 0 || vocab == 0) return fail(GUFFIN_E_SHAPE, "selection_requests: empty shape");
    if (top_k == 0 || top_k > 256) return fail(GUFFIN_E_CAPACITY, "selection_requests: top_k must be in [1, 256]");
    if ((reinterpret_cast<uintptr_t>(raw) | reinterpret_cast<uintptr_t>(resolved)) & 3u)
        return fail(GUFFIN_E_ALIGN, "selection_requests: rows must be 4-byte aligned");
    launch(selection_requests_kernel, dim3(rows), dim3(64), 0, as_stream(stream),
                       static_cast<const SelectionRow*>(raw), vocab, top_k, repetition_enabled,
                       static_cast<ResolvedRow*>(resolved), histories, status);
    return check_launch("selection_requests");
}

extern "C" int guffin_hip_select_candidates_resolved(void* stream, const float* logits, uint32_t rows, uint32_t vocab,
                                                     uint32_t retain_capacity, const void* resolved, void* workspace,
                                                     void* result, uint32_t* status) {
    if (!resolved) return fail(GUFFIN_E_ARG, "select_candidates_resolved: null pointer");
    const uint32_t* words = static_cast<const uint32_t*>(resolved);
    constexpr uint32_t stride = sizeof(ResolvedRow) / 4;
    // history ids, their count and the row's retain all sit in the record; the ids are 68 words apart too
    return select_candidates_scaled(as_stream(stream), logits, rows, vocab, retain_capacity, 1.0f,
                                    words + offsetof(ResolvedRow, history_token_ids) / 4,
                                    words + offsetof(ResolvedRow, history_count) / 4, workspace, result, status, false,
                                    words + offsetof(ResolvedRow, base_candidate_count) / 4, stride);
}

extern "C" int guffin_hip_argmax(void* stream, const float* logits, uint32_t rows, uint32_t vocab, void* workspace,
                                 uint32_t* token, float* logit, uint32_t* status) {
    if (!logits || !workspace || !token) return fail(GUFFIN_E_ARG, "argmax: null pointer");
    if (rows == 0 || vocab == 0) return fail(GUFFIN_E_SHAPE, "argmax: empty shape");
    if (reinterpret_cast<uintptr_t>(workspace) & 7u) return fail(GUFFIN_E_ALIGN, "argmax: workspace must be 8-byte aligned");
    const uint32_t blocks = vocab / 1024 < 1 ? 1 : (vocab / 1024 > 256 ? 256 : vocab / 1024);
    hipStream_t s = as_stream(stream);
    uint64_t* part = static_cast<uint64_t*>(workspace);  // rows * 256 keys at most
    launch(argmax_tile_kernel, dim3(blocks, rows), dim3(256), 0, s, logits, part, vocab, status);
    if (int rc = check_launch("argmax(tile)")) return rc;
    launch(argmax_final_kernel, dim3(rows), dim3(256), 0, s, part, blocks, token, logit);
    return check_launch("argmax(final)");
}
