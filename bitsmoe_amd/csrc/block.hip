// The block's forward as one call: everything between the hidden states and the block output that runs on this library's
// kernels -- the two projections, the router, the routed-expert operator, the super experts' operator call beside it, the
// closing pass -- is launched from here, so that a forward costs its host one call instead of one per kernel.  At decode
// sizes the kernels of a block take 30 to 100 us and the host work of launching them one by one from the framework took as
// long or longer (128-expert layer, one token: 82 us per eager forward for 29 us of kernels).
#include <algorithm>

#include "common.h"

using namespace bitsmoe;

static inline size_t align256(size_t v) { return (v + 255) / 256 * 256; }

// Rows that the few-rows kernel takes: a call of more ends with the projection's operand (and super_out) in the caller's memory.
constexpr int64_t PROJECT_OUT_MAX_ROWS = 64;

// Where the intermediates of a call sit in the workspace.
struct BlockWorkspace {
    size_t selected, weights, rank_accum, operand, forward, forward_bytes, super_forward, super_bytes, super_out, total;
};
static BlockWorkspace carve(const bitsmoe_block_plan* p, int64_t T) {
    BlockWorkspace w;
    size_t at = 0;
    auto take = [&](size_t bytes) { const size_t here = at; at += align256(bytes); return here; };
    w.selected = take((size_t)T * p->top_k * 8);
    w.weights = take((size_t)T * p->top_k * 4);
    w.rank_accum = take((size_t)T * p->rank_out * 4);
    const bool may_project = T <= PROJECT_OUT_MAX_ROWS;
    w.operand = take(may_project ? (size_t)T * (p->rank_out + p->shared_intermediate) * 2 : 0);
    w.forward_bytes = align256(bitsmoe_forward_routed_workspace_bytes(p->gate, p->up, p->down, T, p->top_k, BITSMOE_PATH_AUTO));
    w.forward = take(w.forward_bytes);
    w.super_bytes = p->super_gate ? align256(bitsmoe_forward_routed_workspace_bytes(p->super_gate, p->super_up, p->super_down, T,
                                                                                    p->top_k, BITSMOE_PATH_AUTO)) : 0;
    w.super_forward = take(w.super_bytes);
    w.super_out = take(p->super_gate && may_project ? (size_t)T * p->hidden * 4 : 0);
    w.total = at;
    return w;
}

extern "C" size_t bitsmoe_block_workspace_bytes(const bitsmoe_block_plan* plan, int64_t n_tokens) {
    if (!plan || !plan->gate || !plan->up || !plan->down || n_tokens < 0 || plan->top_k <= 0) return 0;
    return carve(plan, n_tokens).total;
}

// One stream waits for what the other holds so far (an event of this call: calls on other threads share nothing with it).
static int stream_after(hipStream_t later, hipStream_t earlier) {
    hipEvent_t ev;
    BITSMOE_HIP_TRY(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
    hipError_t e = hipEventRecord(ev, earlier);
    if (e == hipSuccess) e = hipStreamWaitEvent(later, ev, 0);
    (void)hipEventDestroy(ev);
    if (e != hipSuccess) return hip_fail(e, "hipStreamWaitEvent");
    return BITSMOE_OK;
}

extern "C" int32_t bitsmoe_block_router_is_beside(const bitsmoe_block_plan* p, int64_t n_tokens, int32_t stages) {
    return p && (stages & BITSMOE_BLOCK_PROJECT_IN) != 0 && p->router_form == BITSMOE_ROUTER_LINEAR &&
           skinny_linear_takes_router(n_tokens, p->hidden, p->w_in_prepared, p->n_global, p->top_k);
}

extern "C" int bitsmoe_block_forward(const bitsmoe_block_plan* p, const void* x, int64_t ld_x, int64_t n_tokens, void* proj,
                                     int32_t stages, void* selected, float* weights, void* out, float* super_out, void* workspace,
                                     size_t workspace_bytes, void* side_stream, void* stream) {
    return bitsmoe_block_forward_tiled(p, x, ld_x, n_tokens, proj, stages, selected, weights, nullptr, out, super_out, workspace,
                                       workspace_bytes, side_stream, stream);
}

extern "C" int bitsmoe_block_forward_tiled(const bitsmoe_block_plan* p, const void* x, int64_t ld_x, int64_t n_tokens, void* proj,
                                           int32_t stages, void* selected, float* weights, void* operand, void* out, float* super_out,
                                           void* workspace, size_t workspace_bytes, void* side_stream, void* stream) {
    BITSMOE_REQUIRE(p && p->gate && p->up && p->down && p->global_to_local && p->local_to_global, "null pointer in the block's plan");
    BITSMOE_REQUIRE(n_tokens >= 0 && p->top_k > 0, "n_tokens must be >= 0 and top_k > 0");
    if (n_tokens == 0) return BITSMOE_OK;
    BITSMOE_REQUIRE(x && proj && out, "null pointer");
    BITSMOE_REQUIRE(p->router_form != BITSMOE_ROUTER_CALLER || (selected && weights), "the caller's routing is missing");
    // (here, not only in the closing pass: the grouped GEMM's combine writes rows of rank_out before that, rank_out + this apart)
    BITSMOE_REQUIRE(p->shared_intermediate >= 0, "negative size");
    const bool tiled_in = (stages & BITSMOE_BLOCK_PROJECT_IN_TILED) != 0, tiled_out = (stages & BITSMOE_BLOCK_PROJECT_OUT_TILED) != 0;
    const bool few_in = (stages & BITSMOE_BLOCK_PROJECT_IN) != 0, few_out = (stages & BITSMOE_BLOCK_PROJECT_OUT) != 0;
    const bool project_out = few_out || tiled_out;
    BITSMOE_REQUIRE(!(few_in && tiled_in) && !(few_out && tiled_out), "one kernel per projection");
    BITSMOE_REQUIRE(!few_out || n_tokens <= PROJECT_OUT_MAX_ROWS, "the output projection takes at most 64 tokens");
    const bool super = p->super_gate != nullptr;
    const bool in_workspace = project_out && n_tokens <= PROJECT_OUT_MAX_ROWS;
    BITSMOE_REQUIRE(!tiled_out || operand || in_workspace, "more than 64 tokens: the operand's memory is the caller's");
    BITSMOE_REQUIRE(!super || in_workspace || super_out, "super_out must not be null where the caller projects");
    const BlockWorkspace w = carve(p, n_tokens);
    if (workspace == nullptr || workspace_bytes < w.total) {
        set_error("workspace too small: need %zu bytes, got %zu", w.total, workspace_bytes);
        return BITSMOE_E_WORKSPACE;
    }
    BITSMOE_REQUIRE(((uintptr_t)workspace & 255) == 0, "workspace must be 256-byte aligned");
    char* ws = (char*)workspace;
    hipStream_t st = (hipStream_t)stream;
    const int64_t ld = p->in_features;
    const uint16_t* big = (const uint16_t*)proj;
#define BITSMOE_TRY(expr)                      \
    do {                                       \
        const int _rc = (expr);                \
        if (_rc != BITSMOE_OK) return _rc;     \
    } while (0)

    if (tiled_in)
        BITSMOE_TRY(bitsmoe_tiled_linear(x, p->act_dtype, ld_x, p->w_in_rows, n_tokens, p->hidden, p->in_features, proj, ld, nullptr, 0, stream));
    if (!selected) selected = ws + w.selected;
    if (!weights) weights = (float*)(ws + w.weights);
    const bool routed = bitsmoe_block_router_is_beside(p, n_tokens, stages) != 0;
    if (routed) {
        const RouterBeside router = {p->w_router, p->n_global, p->top_k, p->renormalize, p->round_dtype, p->weight_scale, (int64_t*)selected, weights};
        BITSMOE_TRY(skinny_linear_with_router(x, p->act_dtype, ld_x, p->w_in, n_tokens, p->hidden, p->in_features, proj, ld, router, stream));
    } else if (few_in) {
        BITSMOE_TRY(bitsmoe_skinny_linear(x, p->act_dtype, 0, ld_x, p->w_in, p->w_in_prepared, n_tokens, p->hidden, p->in_features,
                                          proj, ld, nullptr, 0, stream));
    }
    if (p->router_form == BITSMOE_ROUTER_LOGITS)
        BITSMOE_TRY(bitsmoe_router_softmax_topk_strided(big + p->col_logits, p->act_dtype, ld, n_tokens, p->n_global, p->top_k,
                                                        p->renormalize, p->weight_scale, p->round_dtype, selected, 1, weights, stream));
    else if (p->router_form == BITSMOE_ROUTER_LINEAR && !routed)
        BITSMOE_TRY(bitsmoe_router_linear_topk(x, p->act_dtype, ld_x, p->w_router, 1, n_tokens, p->hidden, p->n_global, p->top_k,
                                               p->renormalize, p->weight_scale, p->round_dtype, selected, 1, weights, stream));
    // The super experts' operator call needs the router's output and the hidden states only: on the side stream it runs
    // beside the packed experts' call (its small launches fill what the packed kernels leave idle).
    float* sup = super_out ? super_out : (float*)(ws + w.super_out);
    auto run_super = [&](hipStream_t on) {
        return bitsmoe_moe_forward_routed(p->super_gate, p->super_up, p->super_down, x, x, p->act_dtype, n_tokens, p->hidden, p->hidden,
                                          ld_x, ld_x, selected, 1, weights, p->top_k, p->super_global_to_local, p->n_global,
                                          p->super_local_to_global, p->hidden, p->super_intermediate, 0, BITSMOE_PATH_AUTO, sup,
                                          ws + w.super_forward, w.super_bytes, nullptr, on);
    };
    int super_rc = BITSMOE_OK;
    if (super && side_stream) {
        BITSMOE_TRY(stream_after((hipStream_t)side_stream, st));
        super_rc = run_super((hipStream_t)side_stream);      // (reported after the join)
    }
    float* rank_accum = (float*)(ws + w.rank_accum);
    // what the output projection reads: the cast sums beside the shared expert's activations; a few fp32 rows without a
    // shared expert go into it as they are
    const bool f32_rows = few_out && p->shared_intermediate == 0 && skinny_f32_rows_possible(n_tokens, p->rank_out, p->w_out_prepared);
    if (!project_out) operand = out;
    else if (few_out || !operand) operand = ws + w.operand;
    const int k_out = p->rank_out + p->shared_intermediate;
    CastRows cast = {operand, k_out, false};
    const int rc = forward_routed_cast(p->gate, p->up, p->down, big + p->col_gate, big + p->col_up, p->act_dtype, n_tokens, p->rank_gate,
                                       p->rank_up, ld, ld, selected, 1, weights, p->top_k, p->global_to_local, p->n_global,
                                       p->local_to_global, p->rank_out, p->intermediate_size, rank_accum, ws + w.forward,
                                       w.forward_bytes, f32_rows ? nullptr : &cast, stream);
    int finish_rc = BITSMOE_OK;
    if (rc == BITSMOE_OK && !f32_rows && !(cast.done && p->shared_intermediate == 0)) {
        const bool shared = p->shared_intermediate > 0;
        finish_rc = block_finish(rank_accum, n_tokens, p->rank_out, shared ? big + p->col_shared_gate : nullptr,
                                 shared ? big + p->col_shared_up : nullptr, ld, p->shared_intermediate,
                                 shared && p->col_shared_logit >= 0 ? big + p->col_shared_logit : nullptr, ld, p->act_dtype,
                                 operand, k_out, cast.done, stream);
    }
    if (super && side_stream)      // (joined whatever happened in between: the side stream may hold launches)
        BITSMOE_TRY(stream_after(st, (hipStream_t)side_stream));
    BITSMOE_TRY(rc);
    BITSMOE_TRY(finish_rc);
    BITSMOE_TRY(super_rc);
    if (super && !side_stream) BITSMOE_TRY(run_super(st));
    if (tiled_out)
        BITSMOE_TRY(bitsmoe_tiled_linear(operand, p->act_dtype, k_out, p->w_out_rows, n_tokens, k_out, p->hidden, out, p->hidden,
                                         super ? sup : nullptr, p->hidden, stream));
    if (few_out)
        BITSMOE_TRY(skinny_linear(f32_rows ? (const void*)rank_accum : operand, p->act_dtype, f32_rows ? 1 : 0, k_out, p->w_out,
                                  p->w_out_prepared, n_tokens, k_out, p->hidden, out, p->hidden, super ? sup : nullptr, p->hidden,
                                  stream));
#undef BITSMOE_TRY
    return BITSMOE_OK;
}
