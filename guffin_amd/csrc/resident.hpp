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
// exchange: resident_scratch_bytes of memory; sync: resident_sync_words cleared words; x, u: the embedded rows and their first
// norm, written over where the model has more blocks than a launch takes.
bool drafter_pass_fits(const guffin_model_desc& m);
struct DrafterPass {
    uint8_t* exchange; uint32_t* sync;
    const float *rope_local, *rope_global;
    const uint32_t *schedule, *ancestors;
    void *priv_k, *priv_v;
    float *x, *u, *out_hidden, *out_sums;
    uint32_t* status;
};
int drafter_pass(hipStream_t stream, const guffin_model_desc& m, uint32_t rows, const DrafterPass& p);

}  // namespace guffin
