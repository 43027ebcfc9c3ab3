// What the resident passes share (resident.hip, drafter_pass.hip).
#pragma once
#include "common.hpp"

namespace guffin {

constexpr uint32_t kGroups = 32;        // workgroups per XCD
constexpr uint32_t kGrid = 256;
constexpr uint32_t kHd = 256;

__device__ __forceinline__ uint32_t xcc_id() {
    uint32_t v;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(v));
    return v & 0xFu;
}

// The pass of a narrow Q8_0 model with one KV head (drafter_pass.hip): whether it covers the model, and all blocks of one pass.
// Up to kRunRows contiguous rows, an XCD each: a later row takes the keys and values of the earlier ones from them, block by block,
// and a row's sums are those of a pass by itself.
// exchange: drafter_pass_bytes of memory; sync: drafter_pass_sync_words cleared words; x, u: the embedded rows and their first
// norm, written over where the model has more blocks than a launch takes; last_hidden: the last row's final state once more, or
// null; out_sums: the receipt of all rows (receipt_rows = rows) or of the last one (1).
bool drafter_pass_fits(const guffin_model_desc& m);
struct DrafterPass {
    uint8_t* exchange; uint32_t* sync;
    const float *rope_local, *rope_global;
    const uint32_t* schedule;
    void *priv_k, *priv_v;
    float *x, *u, *out_hidden, *last_hidden, *out_sums;
    uint32_t receipt_rows;
    uint32_t* status;
};
uint64_t drafter_pass_bytes(const guffin_model_desc& m, uint32_t rows);
uint32_t drafter_pass_sync_words(const guffin_model_desc& m);
int drafter_pass(hipStream_t stream, const guffin_model_desc& m, uint32_t rows, const DrafterPass& p);

}  // namespace guffin
