// Lifecycle of a drafter between speculation cycles: prefix, pending token and transactions.
//
// Mirrors the state machine of Gemma3DraftPlan (include/local_gguf_engine/engine/gemma3_draft.hpp:56-82;
// src/engine/gemma3_draft.mm:1300-1490; lifecycle cases tests/engine/gemma3_draft_tests.cpp:206-277):
//
//   position       tokens the plan knows, a pending one included
//   materialized   tokens whose K/V rows exist; a pending token (the drafter's last emission, or one restored
//                  by the caller) gets its rows only when the next input needs them
//   transaction    begin .. commit_prefix(p) | abort: rows written in between can be taken back
//
// The reference keeps a transaction's rows in a private arena that attention reads beside the ring.  Here a
// transaction's rows go to the rings at once, where the ring attention of guffin_hip_forward_rows sees them,
// and the ring rows they overwrite (a local layer's slot (position & mask) held position - window) are first
// saved per position in a backup arena per layer (the plan's transaction capacity, a constructor argument as in
// the reference, rounded up to a power of two); abort, truncate and a commit of a shorter prefix copy them back.
// The final normalised row of every position a transaction runs is kept as well (the reference's private_norm,
// gemma3_draft.mm:966-968, 984-992), so that logits can be projected at a frontier a truncate or a shorter commit
// went back to.  Same observable behaviour: an aborted or truncated suffix leaves every ring row as it was, and
// logits after a commit equal those of a plain replay of the kept tokens.
//
// Every call is host-synchronous (it returns when its device work is done), but inside a call the host waits once: the
// passes and laws of up to kBatch tokens are enqueued behind each other, a drafted token passing from law to embedding in
// device memory, and the status word is read when all of them are done (run_batch).  Waiting for every pass and law, and
// a copy launch per block, took 1.4 of the 5.0 ms of six passes and four proposals of an 18-block drafter.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "common.hpp"

#define GUFFIN_TRY(expr) do { if (int rc_ = (expr)) return rc_; } while (0)

namespace guffin {
namespace {

constexpr uint32_t kDefaultTransactionRows = 32;   // when the caller names none (the reference's callers use 96 or 256)
constexpr uint32_t kMaxHorizon = 23;        // external_speculation_max_horizon
constexpr uint64_t kLawBytes = 8 + 256 * 4 + 257 * 8;
constexpr uint32_t kBatch = kMaxHorizon + 1;   // passes between two looks at the status word; no more than a transaction holds
constexpr uint32_t kHistory = 64;              // the sampler's window
struct Draws { uint32_t word, pad; double u_accept, u_residual, u_next; };
// What a call uploads, in one copy: the input tokens of a batch, the draws, and the sampler's window with the drafted tokens
// behind it: chain[kHistory + i] is drafted token i, and the window before it the up to 64 words that precede it
struct Staging { Draws draws[kMaxHorizon]; uint32_t tokens[kBatch]; uint32_t chain[kHistory + kMaxHorizon]; };

struct Carve {
    uint8_t* base; uint64_t used;
    template <typename T> T* take(uint64_t count) {
        used = (used + 255) & ~uint64_t{255};
        T* p = base ? reinterpret_cast<T*>(base + used) : nullptr;
        used += count * sizeof(T);
        return p;
    }
};

struct Buffers {
    uint8_t* forward; uint64_t forward_bytes;
    uint16_t *priv_k, *priv_v, *backup_k, *backup_v;
    float *hidden, *hidden_sums, *hidden_saved, *sums_saved, *txn_hidden, *logits, *parts, *scores;
    Staging* staging;
    uint32_t* status;
    uint8_t *law_ws, *law;
    uint64_t* cdf;
    void **ring_k_table, **ring_v_table;
};

uint32_t arena_rows(uint32_t transaction_rows) {
    uint32_t rows = 1;
    while (rows < transaction_rows) rows <<= 1;
    return rows;
}

Buffers carve(const guffin_model_desc& m, uint32_t arena, void* workspace, uint64_t* total) {
    Carve c {static_cast<uint8_t*>(workspace), 0};
    Buffers b {};
    const uint64_t kvw = uint64_t(m.kv_heads) * m.head_dim;
    b.forward_bytes = std::max(guffin_hip_forward_scratch_bytes(&m, 2, m.ring_global - 2), forward_run_bytes(m));
    b.forward = c.take<uint8_t>(b.forward_bytes);
    b.priv_k = c.take<uint16_t>(uint64_t(m.layer_count) * kRunRows * kvw);
    b.priv_v = c.take<uint16_t>(uint64_t(m.layer_count) * kRunRows * kvw);
    b.backup_k = c.take<uint16_t>(uint64_t(m.layer_count) * arena * kvw);
    b.backup_v = c.take<uint16_t>(uint64_t(m.layer_count) * arena * kvw);
    b.hidden = c.take<float>(2 * uint64_t(m.hidden));
    b.hidden_sums = c.take<float>(guffin_hip_receipt_bytes(2, m.hidden) / 4);
    b.hidden_saved = c.take<float>(2 * uint64_t(m.hidden));
    b.sums_saved = c.take<float>(guffin_hip_receipt_bytes(2, m.hidden) / 4);
    b.txn_hidden = c.take<float>(uint64_t(arena) * m.hidden);
    b.logits = c.take<float>(2 * uint64_t(m.vocab));
    b.parts = c.take<float>(uint64_t(std::max(1u, guffin_hip_gemv_packed_slices(m.head_dtype, m.hidden, m.vocab))) * 2 * m.vocab);
    b.scores = c.take<float>(m.vocab);
    b.staging = c.take<Staging>(1);
    b.status = c.take<uint32_t>(1);
    b.law_ws = c.take<uint8_t>(guffin_hip_draft_law_any_workspace_bytes(m.vocab));
    b.law = c.take<uint8_t>(kLawBytes);
    b.cdf = c.take<uint64_t>(uint64_t(m.vocab) + 1);
    b.ring_k_table = c.take<void*>(m.layer_count);
    b.ring_v_table = c.take<void*>(m.layer_count);
    if (total) *total = (c.used + 255) & ~uint64_t{255};
    return b;
}

Buffers carve(const guffin_draft_plan* p) { return carve(*p->model, p->transaction_arena, p->workspace, nullptr); }

int usable(const guffin_draft_plan* p, const char* what) {
    if (!p || !p->model || !p->workspace) return fail(GUFFIN_E_ARG, what);
    if (p->poisoned) return fail(GUFFIN_E_STATE, "draft_plan: the plan is poisoned (a device status was raised); reset it");
    return GUFFIN_OK;
}

int poison(guffin_draft_plan* p, int code, const char* what) {
    p->poisoned = 1;
    return fail(code, what);
}

// ring rows [first, end) of every layer to the backup arena (save) or back (restore)
int move_rows(hipStream_t s, const guffin_draft_plan* p, const Buffers& b, uint32_t first, uint32_t end, bool save) {
    if (end <= first) return GUFFIN_OK;
    return kv_move_rows(s, *p->model, save ? KvMove::Save : KvMove::Restore, b.backup_k, b.backup_v, p->transaction_arena, first, end - first);
}

// one pass of the `rows` tokens from `token` on (device memory) at the materialized frontier, published to the rings
int forward(hipStream_t s, guffin_draft_plan* p, const Buffers& b, const uint32_t* token, uint32_t rows) {
    const guffin_model_desc& m = *p->model;
    const uint32_t at = p->materialized;
    // a transaction keeps the rows' final normalised states by their place in it
    float* kept = p->transaction_active ? b.txn_hidden + uint64_t(at - p->checkpoint_materialized) * m.hidden : nullptr;
    if (forward_run_chosen(m)) {
        GUFFIN_TRY(forward_run(s, m, token, rows, at, b.forward, b.priv_k, b.priv_v, kept, b.hidden, b.hidden_sums, b.status));
        GUFFIN_TRY(commit_rows_keeping(s, m, b.priv_k, b.priv_v, b.ring_k_table, b.ring_v_table, nullptr, at, rows, nullptr, nullptr));
    } else {
        GUFFIN_TRY(guffin_hip_forward_rows(s, &m, token, 1, at, b.forward, b.forward_bytes, b.priv_k, b.priv_v, b.hidden,
                                           b.hidden_sums, b.status));
        GUFFIN_TRY(commit_rows_keeping(s, m, b.priv_k, b.priv_v, b.ring_k_table, b.ring_v_table, nullptr, at, 1, b.hidden, kept));
        rows = 1;
    }
    p->materialized = at + rows;
    p->last_rows = 1;
    p->logits_valid = 0;
    p->hidden_valid = 1;
    return GUFFIN_OK;
}

int read_status(hipStream_t s, const Buffers& b, uint32_t* status) {
    return hipMemcpyWithStream(status, b.status, 4, hipMemcpyDeviceToHost, s) == hipSuccess ? GUFFIN_OK : GUFFIN_E_HIP;
}

int finish(hipStream_t s, guffin_draft_plan* p, const Buffers& b, const char* what) {
    uint32_t status = 0;
    if (read_status(s, b, &status)) return poison(p, GUFFIN_E_HIP, what);
    if (status != 0) return poison(p, GUFFIN_E_NUMERIC, what);
    return GUFFIN_OK;
}

// the output rows of the pass at the frontier, kept across a transaction so that an abort leaves the plan able to
// draft from (or read the logits of) the prefix it returns to; rows and receipt lie behind each other on both sides
int copy_frontier(hipStream_t s, const guffin_model_desc& m, const Buffers& b, bool save) {
    const size_t bytes = (b.hidden_sums - b.hidden) * 4 + guffin_hip_receipt_bytes(2, m.hidden);
    if (hipMemcpyAsync(save ? b.hidden_saved : b.hidden, save ? b.hidden : b.hidden_saved, bytes, hipMemcpyDeviceToDevice, s) != hipSuccess)
        return fail(GUFFIN_E_HIP, "draft_plan: copying the frontier rows failed");
    return GUFFIN_OK;
}

// the final state at `position`, which the open transaction ran or began on, back to b.hidden / b.hidden_sums
int restore_frontier(hipStream_t s, guffin_draft_plan* p, const Buffers& b, uint32_t position) {
    const guffin_model_desc& m = *p->model;
    p->hidden_valid = p->logits_valid = 0;
    if (position > p->checkpoint_materialized) {
        const float* kept = b.txn_hidden + uint64_t(position - 1 - p->checkpoint_materialized) * m.hidden;
        if (hipMemcpyAsync(b.hidden, kept, uint64_t(m.hidden) * 4, hipMemcpyDeviceToDevice, s) != hipSuccess)
            return fail(GUFFIN_E_HIP, "draft_plan: restoring the frontier's state failed");
        GUFFIN_TRY(guffin_hip_group_sums(s, b.hidden, b.hidden_sums, 1, m.hidden));
        p->last_rows = 1;
        p->hidden_valid = 1;
    } else if (p->checkpoint_hidden_valid) {
        GUFFIN_TRY(copy_frontier(s, m, b, false));
        p->last_rows = p->checkpoint_last_rows;
        p->hidden_valid = 1;
    }
    return GUFFIN_OK;
}

// Enqueues `body` (up to `rows` passes from the materialized frontier on, with the laws between them), waits once and looks at
// the status word.  Two things can make a batch run again, from the ring rows and the final state it began with:
//   - the resident pass gave up a wait (a device shared with other work): its rows, and whatever else it raised in the status
//     word, are not to be trusted; the resident form is switched off for the process and the batch runs one launch per operator;
//   - a law's support did not fit the compact form (status bit 32): body(true) runs the laws with the full-vocabulary kernels
//     behind the compact one, which otherwise are fourteen launches per proposal that find nothing to do.
// The ring rows a batch overwrites go to the backup arena first, inside a transaction (where they may already be) and, for a
// batch that may have to run again, outside one.  poisoned: the plan after an error, as for every pass that fails.
template <typename Body>
int run_batch(hipStream_t s, guffin_draft_plan* p, const Buffers& b, uint32_t rows, const char* what, Body body) {
    const guffin_model_desc& m = *p->model;
    const uint32_t first = p->materialized, end = first + rows;
    const bool watched = resident_chosen(m, 1) && g_forward_mode == 0;
    if (p->transaction_active) {
        if (end > p->backup_end) {   // rows below backup_end already hold the originals
            if (int rc = move_rows(s, p, b, std::max(first, p->backup_end), end, true)) { p->poisoned = 1; return rc; }
            p->backup_end = end;
        }
    } else if (watched) {
        if (int rc = move_rows(s, p, b, first, end, true)) { p->poisoned = 1; return rc; }
    }
    constexpr uint32_t kOverflow = 32u;   // the compact law's support overflow
    bool full_laws = false, given_up = false;
    for (;;) {
        if (int rc = body(full_laws)) { p->poisoned = 1; return rc; }
        uint32_t status = 0;
        if (read_status(s, b, &status)) return poison(p, GUFFIN_E_HIP, what);
        if (status == 0) return GUFFIN_OK;
        const bool again_plain = watched && !given_up && (status & GUFFIN_STATUS_SYNC) != 0;
        const bool again_full = !again_plain && p->transaction_active && !full_laws && (status & kOverflow) != 0;
        if (!again_plain && !again_full) return poison(p, GUFFIN_E_NUMERIC, what);
        if (again_plain) { resident_note_status(status); given_up = true; }
        full_laws |= again_full;
        if (hipMemsetAsync(b.status, 0, 4, s) != hipSuccess) return poison(p, GUFFIN_E_HIP, what);
        if (int rc = move_rows(s, p, b, first, end, false)) { p->poisoned = 1; return rc; }
        p->materialized = first;
        p->hidden_valid = p->logits_valid = 0;
        if (p->transaction_active)
            if (int rc = restore_frontier(s, p, b, first)) { p->poisoned = 1; return rc; }
    }
}

// host tokens through the blocks, a pending token first: a token's rows and logits do not depend on how the caller grouped its
// appends, which is what lets a commit be compared with a replay bit for bit.  The drafter's pass takes eight at a time, an XCD a
// row, each summed as by itself; any other form goes one row per pass (a two-row pass of those sums attention partitions and norms
// in another order than two one-row passes)
int ingest(hipStream_t s, guffin_draft_plan* p, const Buffers& b, const uint32_t* tokens, uint32_t count, const char* what) {
    std::vector<uint32_t> input;
    if (p->has_pending) input.push_back(p->pending_token);
    input.insert(input.end(), tokens, tokens + count);
    for (uint32_t i0 = 0; i0 < input.size(); i0 += kBatch) {
        const uint32_t n = std::min(kBatch, static_cast<uint32_t>(input.size()) - i0);
        if (hipMemcpyWithStream(b.staging->tokens, input.data() + i0, n * 4, hipMemcpyHostToDevice, s) != hipSuccess)
            return poison(p, GUFFIN_E_HIP, "draft_plan: token upload failed");
        GUFFIN_TRY(run_batch(s, p, b, n, what, [&](bool) {
            for (const uint32_t first = p->materialized; p->materialized - first < n;) {
                const uint32_t done = p->materialized - first;
                GUFFIN_TRY(forward(s, p, b, b.staging->tokens + done, std::min(n - done, kRunRows)));
            }
            return int(GUFFIN_OK);
        }));
    }
    p->has_pending = 0;
    p->position = p->materialized;
    return GUFFIN_OK;
}

// logits of the rows of the last pass (the head GEMV runs only when somebody asks)
int ensure_logits(hipStream_t s, guffin_draft_plan* p, const Buffers& b) {
    if (p->logits_valid) return GUFFIN_OK;
    if (!p->hidden_valid) return fail(GUFFIN_E_STATE, "draft_plan: no pass stands at the current frontier (append a token first)");
    const guffin_model_desc& m = *p->model;
    GUFFIN_TRY(guffin_hip_gemv_packed(s, m.head_dtype, m.head_tiles, b.hidden, b.hidden_sums, b.parts, b.logits, p->last_rows,
                                      m.hidden, m.vocab));
    p->logits_valid = 1;
    return GUFFIN_OK;
}

int capacity_check(const guffin_draft_plan* p, uint32_t new_rows, const char* what) {
    const guffin_model_desc& m = *p->model;
    if (uint64_t(p->materialized) + new_rows > m.ring_global) return fail(GUFFIN_E_CAPACITY, what);
    if (p->transaction_active && uint64_t(p->materialized) + new_rows - p->checkpoint_materialized > p->transaction_rows)
        return fail(GUFFIN_E_CAPACITY, "draft_plan: the transaction would write more rows than the plan was prepared for");
    return GUFFIN_OK;
}

}  // namespace
}  // namespace guffin

using namespace guffin;

// transaction_rows: 0 = 32; otherwise at least the largest horizon + 2 (gemma3_draft.mm:654-655) and no more than a ring holds
static bool transaction_rows_fit(const guffin_model_desc& m, uint32_t& transaction_rows) {
    if (transaction_rows == 0) transaction_rows = kDefaultTransactionRows;
    return transaction_rows >= kMaxHorizon + 2 && arena_rows(transaction_rows) <= m.ring_local && arena_rows(transaction_rows) <= m.ring_global;
}

extern "C" uint64_t guffin_hip_draft_plan_bytes(const guffin_model_desc* model, uint32_t transaction_rows) {
    if (!model || !model->layers || !model->head_tiles || model->ring_global < 4 || !transaction_rows_fit(*model, transaction_rows)) return 0;
    uint64_t total = 0;
    carve(*model, arena_rows(transaction_rows), nullptr, &total);
    return total;
}

extern "C" int guffin_hip_draft_plan_init(void* stream, guffin_draft_plan* plan, const guffin_model_desc* model, void* workspace,
                                          uint64_t workspace_bytes, uint32_t transaction_rows) {
    if (!plan || !model || !model->layers || !workspace) return fail(GUFFIN_E_ARG, "draft_plan_init: null pointer");
    if (!model->head_tiles) return fail(GUFFIN_E_ARG, "draft_plan_init: the model needs its head tiles");
    if (model->vocab % 256 != 0) return fail(GUFFIN_E_SHAPE, "draft_plan_init: the law kernels need a vocabulary that is a multiple of 256");
    if (!transaction_rows_fit(*model, transaction_rows))
        return fail(GUFFIN_E_SHAPE, "draft_plan_init: a transaction holds at least 25 rows (the largest horizon + 2) and, rounded up to a power of two, no more than the smallest ring");
    const uint64_t need = guffin_hip_draft_plan_bytes(model, transaction_rows);
    if (need == 0 || workspace_bytes < need) return fail(GUFFIN_E_CAPACITY, "draft_plan_init: workspace below guffin_hip_draft_plan_bytes");
    if (reinterpret_cast<uintptr_t>(workspace) & 255u) return fail(GUFFIN_E_ALIGN, "draft_plan_init: workspace must be 256-byte aligned");
    std::memset(plan, 0, sizeof(*plan));
    plan->model = model;
    plan->workspace = workspace;
    plan->workspace_bytes = workspace_bytes;
    plan->transaction_rows = transaction_rows;
    plan->transaction_arena = arena_rows(transaction_rows);
    const Buffers b = carve(plan);
    std::vector<void*> rk(model->layer_count), rv(model->layer_count);
    for (uint32_t l = 0; l < model->layer_count; ++l) {
        if (!model->layers[l].ring_k || !model->layers[l].ring_v) return fail(GUFFIN_E_ARG, "draft_plan_init: every layer needs its rings");
        rk[l] = model->layers[l].ring_k;
        rv[l] = model->layers[l].ring_v;
    }
    hipStream_t s = as_stream(stream);
    if (hipMemcpyAsync(b.ring_k_table, rk.data(), rk.size() * sizeof(void*), hipMemcpyHostToDevice, s) != hipSuccess
        || hipMemcpyAsync(b.ring_v_table, rv.data(), rv.size() * sizeof(void*), hipMemcpyHostToDevice, s) != hipSuccess
        || hipMemsetAsync(b.status, 0, 4, s) != hipSuccess || hipStreamSynchronize(s) != hipSuccess)
        return fail(GUFFIN_E_HIP, "draft_plan_init: upload failed");
    return GUFFIN_OK;
}

// Forgets the prefix (reset(), gemma3_draft.hpp:63): ring contents stay but no row of them is referenced.
extern "C" int guffin_hip_draft_plan_reset(void* stream, guffin_draft_plan* plan) {
    if (!plan || !plan->model || !plan->workspace) return fail(GUFFIN_E_ARG, "draft_plan_reset: null pointer");
    const Buffers b = carve(plan);
    hipStream_t s = as_stream(stream);
    if (hipMemsetAsync(b.status, 0, 4, s) != hipSuccess || hipStreamSynchronize(s) != hipSuccess)
        return fail(GUFFIN_E_HIP, "draft_plan_reset: clearing the status failed");
    const guffin_model_desc* model = plan->model;
    void* workspace = plan->workspace;
    const uint64_t bytes = plan->workspace_bytes;
    const uint32_t rows = plan->transaction_rows, arena = plan->transaction_arena;
    std::memset(plan, 0, sizeof(*plan));
    plan->model = model; plan->workspace = workspace; plan->workspace_bytes = bytes;
    plan->transaction_rows = rows; plan->transaction_arena = arena;
    return GUFFIN_OK;
}

extern "C" int guffin_hip_draft_plan_begin_transaction(void* stream, guffin_draft_plan* plan) {
    GUFFIN_TRY(usable(plan, "draft_plan_begin_transaction: null pointer"));
    if (plan->transaction_active) return fail(GUFFIN_E_STATE, "draft_plan_begin_transaction: a transaction is already open");
    if (plan->hidden_valid) GUFFIN_TRY(copy_frontier(as_stream(stream), *plan->model, carve(plan), true));
    plan->checkpoint_hidden_valid = plan->hidden_valid;
    plan->checkpoint_last_rows = plan->last_rows;
    plan->checkpoint_position = plan->position;
    plan->checkpoint_materialized = plan->materialized;
    plan->checkpoint_pending = plan->pending_token;
    plan->checkpoint_has_pending = plan->has_pending;
    plan->backup_end = plan->materialized;
    plan->transaction_active = 1;
    return GUFFIN_OK;
}

extern "C" int guffin_hip_draft_plan_abort_transaction(void* stream, guffin_draft_plan* plan) {
    GUFFIN_TRY(usable(plan, "draft_plan_abort_transaction: null pointer"));
    // outside a transaction the reference's abort poisons the plan (gemma3_draft.mm:1305-1312): there is nothing to
    // go back to, and the caller's ledger is out of step with the plan's
    if (!plan->transaction_active) { plan->poisoned = 1; return fail(GUFFIN_E_STATE, "draft_plan_abort_transaction: no transaction is open; the plan is poisoned"); }
    const Buffers b = carve(plan);
    hipStream_t s = as_stream(stream);
    if (int rc = move_rows(s, plan, b, plan->checkpoint_materialized, plan->backup_end, false)) { plan->poisoned = 1; return rc; }
    GUFFIN_TRY(finish(s, plan, b, "draft_plan_abort_transaction: restoring the ring rows failed"));
    plan->position = plan->checkpoint_position;
    plan->materialized = plan->checkpoint_materialized;
    plan->pending_token = plan->checkpoint_pending;
    plan->has_pending = plan->checkpoint_has_pending;
    plan->transaction_active = 0;
    plan->hidden_valid = plan->logits_valid = 0;
    if (plan->checkpoint_hidden_valid) {
        if (int rc = copy_frontier(s, *plan->model, b, false)) { plan->poisoned = 1; return rc; }
        plan->hidden_valid = 1;
        plan->last_rows = plan->checkpoint_last_rows;
    }
    return GUFFIN_OK;
}

// 1 if truncate(position) would be admitted: the current position always (nothing changes), and inside a transaction
// any position down to where it began (gemma3_draft.mm:1283-1288)
extern "C" int guffin_hip_draft_plan_can_truncate(const guffin_draft_plan* plan, uint32_t position) {
    if (!plan || !plan->model || plan->poisoned || position > plan->position) return 0;
    return position == plan->position || (plan->transaction_active && position >= plan->checkpoint_position);
}

extern "C" int guffin_hip_draft_plan_truncate(void* stream, guffin_draft_plan* plan, uint32_t position) {
    GUFFIN_TRY(usable(plan, "draft_plan_truncate: null pointer"));
    if (!guffin_hip_draft_plan_can_truncate(plan, position))
        return fail(GUFFIN_E_STATE, "draft_plan_truncate: only rows written inside the open transaction can be dropped");
    if (position == plan->position) return GUFFIN_OK;
    if (position < plan->materialized) {
        const Buffers b = carve(plan);
        hipStream_t s = as_stream(stream);
        if (int rc = move_rows(s, plan, b, position, plan->backup_end, false)) { plan->poisoned = 1; return rc; }
        plan->backup_end = std::min(plan->backup_end, position);
        plan->materialized = position;
        // the frontier's final state: a row this transaction ran, or the one the transaction began on
        if (int rc = restore_frontier(s, plan, b, position)) { plan->poisoned = 1; return rc; }
        GUFFIN_TRY(finish(s, plan, b, "draft_plan_truncate: restoring the frontier's state failed"));
    }
    plan->has_pending = 0;    // position <= materialized now: whatever was pending lay beyond it
    plan->position = position;
    return GUFFIN_OK;
}

// Keeps the first `position` tokens and closes the transaction.  The prefix may end in the pending token.
extern "C" int guffin_hip_draft_plan_commit_prefix(void* stream, guffin_draft_plan* plan, uint32_t position) {
    GUFFIN_TRY(usable(plan, "draft_plan_commit_prefix: null pointer"));
    if (!plan->transaction_active) return fail(GUFFIN_E_STATE, "draft_plan_commit_prefix: no transaction is open");
    if (position < plan->checkpoint_position || position > plan->position)
        return fail(GUFFIN_E_ARG, "draft_plan_commit_prefix: the prefix must end inside the transaction");
    if (position < plan->position) GUFFIN_TRY(guffin_hip_draft_plan_truncate(stream, plan, position));
    plan->transaction_active = 0;
    return GUFFIN_OK;
}

extern "C" int guffin_hip_draft_plan_append(void* stream, guffin_draft_plan* plan, const uint32_t* tokens, uint32_t count) {
    GUFFIN_TRY(usable(plan, "draft_plan_append: null pointer"));
    if (count == 0) return GUFFIN_OK;
    if (!tokens) return fail(GUFFIN_E_ARG, "draft_plan_append: null pointer");
    for (uint32_t i = 0; i < count; ++i)
        if (tokens[i] >= plan->model->vocab) return fail(GUFFIN_E_ARG, "draft_plan_append: token outside the vocabulary");
    GUFFIN_TRY(capacity_check(plan, count + (plan->has_pending ? 1u : 0u), "draft_plan_append: the context is full"));
    const Buffers b = carve(plan);
    hipStream_t s = as_stream(stream);
    return ingest(s, plan, b, tokens, count, "draft_plan_append: the pass raised the device status");
}

// A saved emission of this drafter put back after its prefix was replayed: known, but not run (:75-77).
extern "C" int guffin_hip_draft_plan_restore_pending_token(guffin_draft_plan* plan, uint32_t token) {
    GUFFIN_TRY(usable(plan, "draft_plan_restore_pending_token: null pointer"));
    if (plan->transaction_active) return fail(GUFFIN_E_STATE, "draft_plan_restore_pending_token: not inside a transaction");
    if (plan->has_pending) return fail(GUFFIN_E_STATE, "draft_plan_restore_pending_token: a token is already pending");
    if (plan->materialized == 0) return fail(GUFFIN_E_STATE, "draft_plan_restore_pending_token: no prefix to follow");
    if (token >= plan->model->vocab) return fail(GUFFIN_E_ARG, "draft_plan_restore_pending_token: token outside the vocabulary");
    if (uint64_t(plan->position) + 1 > plan->model->ring_global) return fail(GUFFIN_E_CAPACITY, "draft_plan_restore_pending_token: the context is full");
    plan->pending_token = token;
    plan->has_pending = 1;
    plan->position += 1;
    return GUFFIN_OK;
}

// Drafts `horizon` tokens inside the open transaction from the given 32-bit words: token i comes from the
// law of the logits after token i-1 (the last appended token for i = 0); all but the last are run through the
// blocks, the last one stays pending (propose, gemma3_draft.mm:1430-1486).  history: the sampler's window in
// chronological order (host), extended by the drafted tokens as the chain grows; used when the options carry
// a repetition penalty.
extern "C" int guffin_hip_draft_plan_propose(void* stream, guffin_draft_plan* plan, const uint32_t* words, uint32_t horizon,
                                             const void* options, const uint32_t* history, uint32_t history_count,
                                             uint32_t* drafted) {
    GUFFIN_TRY(usable(plan, "draft_plan_propose: null pointer"));
    if (!words || !options || !drafted) return fail(GUFFIN_E_ARG, "draft_plan_propose: null pointer");
    if (!plan->transaction_active) return fail(GUFFIN_E_STATE, "draft_plan_propose: proposals are drafted inside a transaction");
    if (horizon == 0 || horizon > kMaxHorizon) return fail(GUFFIN_E_CAPACITY, "draft_plan_propose: the horizon must be in [1, 23]");
    if (history_count > 64 || (history_count && !history)) return fail(GUFFIN_E_ARG, "draft_plan_propose: at most 64 history tokens");
    if (plan->materialized == 0) return fail(GUFFIN_E_STATE, "draft_plan_propose: no prefix to draft from");
    if (!plan->has_pending && !plan->hidden_valid && !plan->logits_valid)   // a state error, not a fault: nothing is poisoned
        return fail(GUFFIN_E_STATE, "draft_plan_propose: no pass stands at the current frontier (append a token first)");
    GUFFIN_TRY(capacity_check(plan, horizon - 1 + (plan->has_pending ? 1u : 0u), "draft_plan_propose: the context is full"));
    struct Options { float temperature; uint32_t top_k; float top_p, min_p, repetition_penalty; };
    Options opt;
    std::memcpy(&opt, options, sizeof(opt));
    const guffin_model_desc& m = *plan->model;
    const Buffers b = carve(plan);
    hipStream_t s = as_stream(stream);
    Staging up {};
    const bool pending = plan->has_pending != 0;
    for (uint32_t i = 0; i < horizon; ++i) up.draws[i] = {words[i], 0, 0.5, 0.5, 0.5};
    if (pending) up.tokens[0] = plan->pending_token;
    for (uint32_t i = 0; i < history_count; ++i) up.chain[kHistory - history_count + i] = history[i];
    if (hipMemcpyWithStream(b.staging, &up, sizeof(up), hipMemcpyHostToDevice, s) != hipSuccess)
        return poison(plan, GUFFIN_E_HIP, "draft_plan_propose: upload failed");
    const bool penalise = opt.repetition_penalty != 1.0f;
    Options law_options = opt;
    law_options.repetition_penalty = 1.0f;   // applied to the scores below, as gd_process does before the law
    // what guffin_hip_draft_law takes; options out of range are guffin_hip_draft_law_any's to refuse
    const bool compact = opt.temperature > 0.f && std::isfinite(opt.temperature) && opt.top_k >= 1 && opt.top_k <= 64 && opt.top_p > 0.f
                      && opt.top_p <= 1.f && opt.min_p >= 0.f && opt.min_p <= 1.f;
    GUFFIN_TRY(run_batch(s, plan, b, horizon - 1 + (pending ? 1u : 0u), "draft_plan_propose: a pass or a law raised the device status", [&](bool full_laws) {
        if (pending) GUFFIN_TRY(forward(s, plan, b, b.staging->tokens, 1));
        for (uint32_t i = 0; i < horizon; ++i) {
            GUFFIN_TRY(ensure_logits(s, plan, b));
            const float* logits = b.logits + uint64_t(plan->last_rows - 1) * m.vocab;
            const uint32_t window = std::min(kHistory, history_count + i);
            uint32_t* token = b.staging->chain + kHistory + i;
            if (penalise && window != 0) {
                GUFFIN_TRY(guffin_hip_draft_process(s, logits, m.vocab, token - window, window, opt.repetition_penalty, b.scores));
                logits = b.scores;
            }
            if (compact && !full_laws)
                GUFFIN_TRY(guffin_hip_draft_law(s, logits, m.vocab, &law_options, 0, 0, b.staging->draws + i, b.law_ws, b.law, token, b.status));
            else
                GUFFIN_TRY(guffin_hip_draft_law_any(s, logits, m.vocab, &law_options, 0, 0, b.staging->draws + i, b.law_ws, b.law, b.cdf,
                                                    token, b.status));
            if (i + 1 < horizon) GUFFIN_TRY(forward(s, plan, b, token, 1));
        }
        return int(GUFFIN_OK);
    }));
    plan->has_pending = 0;
    plan->position = plan->materialized;
    if (hipMemcpyWithStream(drafted, b.staging->chain + kHistory, horizon * 4, hipMemcpyDeviceToHost, s) != hipSuccess)
        return poison(plan, GUFFIN_E_HIP, "draft_plan_propose: read-back failed");
    plan->pending_token = drafted[horizon - 1];
    plan->has_pending = 1;
    plan->position = plan->materialized + 1;
    return GUFFIN_OK;
}

// Logits after the last materialized token (read_logits, :94), to host memory.
extern "C" int guffin_hip_draft_plan_read_logits(void* stream, guffin_draft_plan* plan, float* logits_host) {
    GUFFIN_TRY(usable(plan, "draft_plan_read_logits: null pointer"));
    if (!logits_host) return fail(GUFFIN_E_ARG, "draft_plan_read_logits: null pointer");
    const Buffers b = carve(plan);
    hipStream_t s = as_stream(stream);
    GUFFIN_TRY(ensure_logits(s, plan, b));
    GUFFIN_TRY(finish(s, plan, b, "draft_plan_read_logits: the head raised the device status"));
    const uint64_t V = plan->model->vocab;
    if (hipMemcpy(logits_host, b.logits + uint64_t(plan->last_rows - 1) * V, V * 4, hipMemcpyDeviceToHost) != hipSuccess)
        return poison(plan, GUFFIN_E_HIP, "draft_plan_read_logits: read-back failed");
    return GUFFIN_OK;
}

// fp16 K and V rows of `count` materialized positions of one layer, in position order (read_cache, :95-98).
// Rows a local layer no longer holds (older than its ring) are refused, never made up.
extern "C" int guffin_hip_draft_plan_read_cache(void* stream, const guffin_draft_plan* plan, uint32_t layer, uint32_t first_position,
                                                uint32_t count, void* keys_host, void* values_host) {
    if (!plan || !plan->model || !keys_host || !values_host) return fail(GUFFIN_E_ARG, "draft_plan_read_cache: null pointer");
    const guffin_model_desc& m = *plan->model;
    if (layer >= m.layer_count) return fail(GUFFIN_E_ARG, "draft_plan_read_cache: no such layer");
    if (uint64_t(first_position) + count > plan->materialized) return fail(GUFFIN_E_ARG, "draft_plan_read_cache: rows beyond the materialized prefix");
    const uint32_t capacity = layer_is_local(m.global_period, layer) ? m.ring_local : m.ring_global;
    if (plan->materialized - first_position > capacity) return fail(GUFFIN_E_ARG, "draft_plan_read_cache: rows older than the layer's ring");
    if (hipStreamSynchronize(as_stream(stream)) != hipSuccess) return fail(GUFFIN_E_HIP, "draft_plan_read_cache: the stream failed");
    const uint64_t row_bytes = uint64_t(m.kv_heads) * m.head_dim * 2;
    for (uint32_t i = 0; i < count; ++i) {
        const uint64_t slot = (first_position + i) & (capacity - 1);
        if (hipMemcpy(static_cast<uint8_t*>(keys_host) + i * row_bytes, static_cast<const uint8_t*>(m.layers[layer].ring_k) + slot * row_bytes,
                      row_bytes, hipMemcpyDeviceToHost) != hipSuccess
            || hipMemcpy(static_cast<uint8_t*>(values_host) + i * row_bytes, static_cast<const uint8_t*>(m.layers[layer].ring_v) + slot * row_bytes,
                         row_bytes, hipMemcpyDeviceToHost) != hipSuccess)
            return fail(GUFFIN_E_HIP, "draft_plan_read_cache: read-back failed");
    }
    return GUFFIN_OK;
}
