// The whole layer in one call.  Host code only: it lays out one scratch buffer and enqueues the operators of the
// layer, so that a decode step costs the launches themselves (2 to 3 us each) instead of an interpreter round trip,
// a handful of allocations and three event records around every one of them: a recorded event alone is a 5.6 us gap
// on the GPU, three of them per layer.
#include <mutex>
#include <vector>

#include "gmm_common.h"
#include "gmm_tiled.h"
#include "layer_parts.h"

using namespace moe355;

namespace {

struct Arena {
    char* base;
    size_t used = 0;
    template <typename T>
    T* take(size_t bytes)
    {
        T* p = (T*)(base + used);
        used += (bytes + 255) & ~(size_t)255;
        return p;
    }
};

enum { W_INT8 = 0, W_INT8_LIST = 1, W_INT4 = 2 };

// the buffers of one call, all in the caller's workspace
struct Buffers {
    void* topk_weights;
    int32_t* topk_ids;
    int8_t* xq;
    float* x_scale;
    int64_t* expert_tokens;
    int64_t* one_group;
    float* ymax;  // a few tokens: maxima of the SwiGLU values, 16 at a time
    int32_t* dst;
    int32_t* row_token;
    MeetingPlan plan;
    uint32_t* meet;  // [plan.columns][R], behind them [sh_columns][T]
    int sh_columns, meet_words;  // meet_words: for each of the R pairs
    void* map_ws;
    float* logits;
    void* gate_ws;
    void* mlp_ws;  // fp32 SwiGLU values, behind them the scratch of the gate_up GEMM
    int8_t* q1;
    float* q1_scale;
    void* o;
    void* gmm2_ws;
    int32_t* sh_acc;
    void* sh_ws;
    int8_t* sh_q;
    float* sh_q_scale;
    void* sh_ws2;
    void* sh_out;
    size_t map_bytes, gate_bytes, mlp_bytes, gmm2_bytes, sh_bytes, sh2_bytes, total;
};

struct Forms {
    bool few;      // a few tokens: two or three launches (few.hip), and one in front where few_gates leaves the gating to it
    bool pairs;    // pair order
    bool requant;  // ... with the re-quantisation inside the down GEMM
    bool merged;   // ... and the shared expert in the two GEMM launches
    bool shared_few;  // the shared expert alone on the kernels for a few tokens
    bool small;    // sorted, gating + sort + quantisation in one launch
};

FewArgs few_args(const moe355_layer& l, const Buffers& b, int64_t T)
{
    FewArgs a = {};
    a.xq = b.xq;
    a.x_scale = b.x_scale;
    a.ids = b.topk_ids;
    a.tw = (const uint16_t*)b.topk_weights;
    a.T = (int)T;
    a.k = l.top_k;
    a.R = (int)T * l.top_k;
    a.E = l.num_experts;
    a.H = (int)l.hidden;
    a.I = (int)l.intermediate;
    if (l.weights == W_INT8_LIST) {
        a.w13_list = (const int8_t* const*)l.w13;
        a.s13_list = (const float* const*)l.s13;
        a.w2_list = (const int8_t* const*)l.w2;
        a.s2_list = (const float* const*)l.s2;
    } else {
        a.w13 = (const int8_t*)l.w13;
        a.s13 = (const float*)l.s13;
        a.w2 = (const int8_t*)l.w2;
        a.s2 = (const float*)l.s2;
    }
    a.limit = l.swiglu_limit;
    if (l.shared) {
        a.S = (int)l.shared_intermediate;
        a.sw13 = l.shared_w13;
        a.sw2 = l.shared_w2;
        a.ss13 = l.shared_s13;
        a.ss2 = l.shared_s2;
        a.sh_limit = l.shared_limit;
        a.sh_alpha = l.shared_alpha;
        a.sh_beta = l.shared_beta;
    }
    a.y = (float*)b.mlp_ws;
    a.ymax = b.ymax;
    a.q1 = b.q1;
    a.q1_scale = b.q1_scale;
    a.f16 = l.x_dtype == MOE355_DT_F16;
    a.load = l.load;
    return a;
}

// the shared expert on its own: no pairs
FewArgs shared_args(const moe355_layer& l, const Buffers& b, int64_t T)
{
    FewArgs a = few_args(l, b, T);
    a.R = 0;
    a.k = 0;
    a.load = nullptr;
    a.y = (float*)b.sh_acc;
    a.q1 = b.sh_q;
    a.q1_scale = b.sh_q_scale;
    a.out = (uint16_t*)b.sh_out;
    return a;
}

Forms forms_of(const moe355_layer& l, int64_t T)
{
    Forms f = {};
    f.few = l.weights != W_INT4 && l.pair_order && T <= 64 && l.top_k <= 64 &&
            moe355_gate_quant_supported(T, l.top_k, l.num_experts) && few_supported(few_args(l, Buffers{}, T));
    if (f.few) return f;
    const bool takes_shared = l.weights != W_INT4 && l.shared && l.shared_intermediate == l.intermediate &&
                              l.shared_alpha == 1.0f && l.shared_beta == 0.0f;
    if (l.weights == W_INT4)
        f.pairs = l.pair_order && moe355_gate_quant_supported(T, l.top_k, l.num_experts) &&
                  w4_pairs_supported(T, l.top_k, l.num_experts, l.hidden, l.intermediate, l.group13, l.group2);
    else
        f.pairs = l.pair_order && pair_order_impl(T, l.top_k, l.num_experts, l.num_experts, l.hidden, l.intermediate, takes_shared);
    const bool int8_pairs = f.pairs && l.weights != W_INT4;
    // A shared expert that the two launches can take along saves more (three or four launches) than the re-quantisation inside
    // the second one (a launch, and only without a shared expert in it).  us a call with the re-quantisation inside and the
    // shared expert in launches of its own, in line or on the side stream, against merged: 128 experts of 2048 / 768, eight
    // slots, 10 / 24 / 57 / 64 tokens 74.9 / 110.5 / 130.7 / 132.0 and 78.0 / 104.7 / 122.2 / 123.8 against 71.1 / 96.3 / 114.3 /
    // 115.3, Zipf(1.1) 52.9 / 69.0 / 92.7 / 95.5 and 67.6 / 73.4 / 85.6 / 87.3 against 44.6 / 53.3 / 73.1 / 75.8; 64 experts of
    // 2048 / 512, 64 tokens 71.8 and 73.8 against 57.4.  Nowhere slower between 64 and 128 experts and rows of 512 to 1024 values.
    f.merged = int8_pairs && takes_shared;
    f.requant = int8_pairs && !f.merged &&
                moe355_gmm2_requant_pairs_supported(T, l.top_k, l.hidden, l.intermediate, l.num_experts);
    // Up to 16 tokens the kernels for a few tokens run a shared expert in two or three launches instead of four.  On the
    // side stream that pays from 8 tokens on: below, their many workgroups take more from the routed GEMM beside them
    // than they save.  int4 layer of the DeepSeek-V3 shape, us a call, four launches against these: in line, 2 / 8 / 16
    // tokens 110 / 257 / 405 against 99 / 248 / 397; side stream 97 / 251 / 398 against 100 / 250 / 391.
    f.shared_few = l.shared && !f.merged && T <= 16 && (l.shared == 1 || T >= 8) && few_supported(shared_args(l, Buffers{}, T));
    f.small = !f.pairs && l.sync_counter && moe355_route_quant_small_supported(T, l.top_k, l.num_experts);
    return f;
}

Buffers lay_out(const moe355_layer& l, const Forms& f, int64_t T, void* base)
{
    Arena a = {(char*)base};
    Buffers b = {};
    const int64_t R = T * l.top_k, H = l.hidden, I = l.intermediate;
    const int E = l.num_experts;
    b.topk_weights = a.take<void>((size_t)R * 2);
    b.topk_ids = a.take<int32_t>((size_t)R * 4);
    b.xq = a.take<int8_t>((size_t)T * H);
    b.x_scale = a.take<float>((size_t)T * 4);
    b.expert_tokens = a.take<int64_t>((size_t)E * 8);
    b.one_group = a.take<int64_t>(8);
    if (l.gate_weight) {
        b.logits = a.take<float>((size_t)T * E * 4);
        b.gate_bytes = moe355_router_gate_workspace(T, (int)H, E);
        b.gate_ws = b.gate_bytes ? a.take<void>(b.gate_bytes) : nullptr;
    }
    if (f.few) {
        const size_t values = (size_t)R * I + (l.shared ? (size_t)T * l.shared_intermediate : 0);
        b.ymax = a.take<float>(values / 16 * 4);
        b.mlp_ws = a.take<void>(values * 4);
        b.q1 = a.take<int8_t>(values);
        b.q1_scale = a.take<float>((size_t)(R + T) * 4);
        b.total = a.used;
        return b;
    }
    const int64_t rows = R + (f.merged ? T : 0);
    b.q1 = a.take<int8_t>((size_t)rows * I);
    b.q1_scale = a.take<float>((size_t)rows * 4);
    if (f.pairs) {
        b.mlp_ws = a.take<void>((size_t)rows * I * 4);
        b.o = a.take<void>((size_t)rows * H * 2);
    } else {
        b.dst = a.take<int32_t>((size_t)R * 4);
        b.row_token = a.take<int32_t>((size_t)R * 4);
        if (l.weights != W_INT4 && !f.small) b.plan = meeting_plan(R, H, 2 * I, E);
        // (on a side stream the column workgroups share the chip with other launches and need not run at the same time)
        if (l.shared == 1 && l.shared_alpha == 1.0f && l.shared_beta == 0.0f && !f.small && !f.shared_few && one_launch_map(R, E))
            b.sh_columns = shared_meeting_columns(T, H, 2 * l.shared_intermediate);
        b.meet_words = b.plan.columns + (b.sh_columns + l.top_k - 1) / l.top_k;
        b.meet = a.take<uint32_t>((size_t)R * 4 * b.meet_words);
        b.map_bytes = moe355_init_routing_workspace(T, l.top_k, E);
        b.map_ws = a.take<void>(b.map_bytes);
        // the down GEMM writes its rows where the SwiGLU values were: those are dead once re-quantised
        const size_t y = ((size_t)R * I * 4 + 255) & ~(size_t)255, o = (size_t)R * H * 2;
        b.mlp_bytes = l.weights == W_INT4 ? y : moe355_gmm1_swiglu_quant_workspace(R, 2 * I, H, E);
        b.mlp_ws = a.take<void>(b.mlp_bytes > o ? b.mlp_bytes : o);
        b.o = b.mlp_ws;
        b.gmm2_bytes = l.weights == W_INT4 ? tiled_workspace_bytes(R, E, 64) : moe355_gmm2_dequant_workspace(R, H, I, E);
        b.gmm2_ws = a.take<void>(b.gmm2_bytes);
    }
    if (f.merged) {
        b.sh_out = (char*)b.o + (size_t)R * H * 2;
    } else if (l.shared) {
        const int64_t S = l.shared_intermediate;
        if (f.shared_few) b.ymax = a.take<float>((size_t)T * (S / 16) * 4);
        b.sh_acc = a.take<int32_t>((size_t)T * 2 * S * 4);
        b.sh_bytes = moe355_gmm_i32_workspace(T, 2 * S, H, 1);
        b.sh_ws = a.take<void>(b.sh_bytes);
        b.sh_q = a.take<int8_t>((size_t)T * S);
        b.sh_q_scale = a.take<float>((size_t)T * 4);
        b.sh2_bytes = moe355_gmm2_dequant_workspace(T, H, S, 1);
        b.sh_ws2 = a.take<void>(b.sh2_bytes);
        b.sh_out = a.take<void>((size_t)T * H * 2);
    }
    b.total = a.used;
    return b;
}

int check_layer(const moe355_layer* l)
{
    if (!l || l->hidden <= 0 || l->intermediate <= 0 || l->num_experts <= 0 || l->top_k <= 0) return MOE355_E_ARG;
    if (l->weights < W_INT8 || l->weights > W_INT4 || l->shared < 0 || l->shared > 2) return MOE355_E_ARG;
    if (!l->w13 || !l->s13 || !l->w2 || !l->s2) return MOE355_E_ARG;
    if (l->shared && l->shared_intermediate <= 0) return MOE355_E_ARG;
    if (l->shared && (!l->shared_w13 || !l->shared_s13 || !l->shared_w2 || !l->shared_s2)) return MOE355_E_ARG;
    if (l->x_dtype != MOE355_DT_BF16 && l->x_dtype != MOE355_DT_F16) return MOE355_E_UNSUPPORTED;
    return MOE355_OK;
}

// Events that order the side stream's work against the caller's stream.  A wait takes the state of the event at the
// time of the call, so a pair is free again once its waits are enqueued: it goes back to the list then, and the list
// is as long as there were calls at the same time.  They live as long as the process (there is no safe moment to
// destroy them after the runtime has gone).
struct ForkJoin {
    hipEvent_t fork = nullptr, join = nullptr;
    int dev = -1;
};
constexpr int kDevices = 64;
std::mutex g_events_mutex;
std::vector<ForkJoin> g_events[kDevices];

struct ForkJoinLease {
    ForkJoin fj;
    bool take()
    {
        int dev = -1;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kDevices) return false;
        {
            std::lock_guard<std::mutex> lock(g_events_mutex);
            if (!g_events[dev].empty()) {
                fj = g_events[dev].back();
                g_events[dev].pop_back();
                return true;
            }
        }
        if (hipEventCreateWithFlags(&fj.fork, hipEventDisableTiming) != hipSuccess) return false;
        if (hipEventCreateWithFlags(&fj.join, hipEventDisableTiming) != hipSuccess) {
            (void)hipEventDestroy(fj.fork);
            return false;
        }
        fj.dev = dev;
        return true;
    }
    ~ForkJoinLease()
    {
        if (fj.dev < 0) return;
        std::lock_guard<std::mutex> lock(g_events_mutex);
        g_events[fj.dev].push_back(fj);
    }
};

// dense W8A8 MLP over all tokens, on the rows the routed experts quantised
// cleared: the words for its meeting are
int shared_expert(const moe355_layer& l, const Forms& f, const Buffers& b, int64_t T, void* st, bool beside, bool cleared)
{
    if (f.shared_few) return few_forward(shared_args(l, b, T), nullptr, (hipStream_t)st);
    const int64_t H = l.hidden, I = l.shared_intermediate;
    int rc;
    if (cleared && b.sh_columns) {
        rc = shared_meeting_impl(b.xq, l.shared_w13, l.shared_s13, b.x_scale, b.one_group, T, H, 2 * I, l.shared_limit,
                                 b.meet + (size_t)b.plan.columns * T * l.top_k, b.plan.looks, b.sh_q, b.sh_q_scale, st);
        if (rc != MOE355_OK) return rc;
        return gmm2_impl(b.sh_q, l.shared_w2, nullptr, l.shared_s2, nullptr, b.sh_q_scale, b.one_group, MOE355_GL_CUMSUM, T, I, H,
                         1, b.sh_out, l.x_dtype, b.sh_ws2, b.sh2_bytes, st, false, beside);
    }
    rc = gmm_i32_impl(b.xq, l.shared_w13, b.one_group, MOE355_GL_CUMSUM, T, H, 2 * I, 1, b.sh_acc, b.sh_ws, b.sh_bytes,
                          st, beside);
    if (rc != MOE355_OK) return rc;
    rc = moe355_dequant_swiglu_quant_grouped(b.sh_acc, l.shared_s13, b.x_scale, nullptr, 0, nullptr, 1, T, 2 * I, 1, 1,
                                             l.shared_limit, l.shared_alpha, l.shared_beta, 1, nullptr, 0, nullptr,
                                             b.sh_q, b.sh_q_scale, st);
    if (rc != MOE355_OK) return rc;
    return gmm2_impl(b.sh_q, l.shared_w2, nullptr, l.shared_s2, nullptr, b.sh_q_scale, b.one_group, MOE355_GL_CUMSUM, T, I, H,
                     1, b.sh_out, l.x_dtype, b.sh_ws2, b.sh2_bytes, st, false, beside);
}

int routed_pairs(const moe355_layer& l, const Forms& f, const Buffers& b, int64_t T, void* st)
{
    const int64_t H = l.hidden, I = l.intermediate;
    if (l.weights == W_INT4) {
        int rc = gmm1_w4_pairs(b.xq, b.x_scale, b.topk_ids, T, l.top_k, (const uint8_t*)l.w13, (const float*)l.s13,
                               l.group13, H, 2 * I, l.num_experts, l.swiglu_limit, (float*)b.mlp_ws, b.q1, b.q1_scale,
                               (hipStream_t)st);
        if (rc != MOE355_OK) return rc;
        return gmm2_w4_pairs(b.q1, b.q1_scale, b.topk_ids, T, l.top_k, (const uint8_t*)l.w2, (const float*)l.s2, l.group2,
                             I, H, l.num_experts, b.o, l.x_dtype, (hipStream_t)st);
    }
    PairWeights w13 = {}, w2 = {};
    if (l.weights == W_INT8_LIST) {
        w13.list = (const int8_t* const*)l.w13;
        w13.scale_list = (const float* const*)l.s13;
        w2.list = (const int8_t* const*)l.w2;
        w2.scale_list = (const float* const*)l.s2;
    } else {
        w13.one = (const int8_t*)l.w13;
        w13.scale = (const float*)l.s13;
        w2.one = (const int8_t*)l.w2;
        w2.scale = (const float*)l.s2;
    }
    float* y = (float*)b.mlp_ws;
    const PairShared sh13 = {l.shared_w13, l.shared_s13, l.shared_limit}, sh2 = {l.shared_w2, l.shared_s2};
    int rc = gmm1_pairs_impl(b.xq, b.x_scale, b.topk_ids, T, l.top_k, w13, H, 2 * I, l.num_experts, l.swiglu_limit, y,
                             f.requant ? nullptr : b.q1, b.q1_scale, st, f.merged ? &sh13 : nullptr);
    if (rc != MOE355_OK) return rc;
    return gmm2_pairs_impl(b.q1, b.q1_scale, f.requant ? y : nullptr, w2, b.topk_ids, T, l.top_k, I, H, l.num_experts,
                           b.o, l.x_dtype, st, f.merged ? &sh2 : nullptr);
}

int routed_sorted(const moe355_layer& l, const Buffers& b, int64_t T, bool tiles_ready, void* st)
{
    const int64_t H = l.hidden, I = l.intermediate, R = T * l.top_k;
    const int E = l.num_experts;
    int rc;
    if (l.weights == W_INT4) {
        const TileMap chunks = w4_chunk_spec(R, E, b.gmm2_ws).tm;
        const TileMap* tm = tiles_ready ? &chunks : nullptr;
        rc = gmm1_w4_impl(b.xq, (const uint8_t*)l.w13, (const float*)l.s13, l.group13, nullptr, b.x_scale, b.expert_tokens,
                          MOE355_GL_COUNT, R, H, 2 * I, E, l.swiglu_limit, b.q1, b.q1_scale, b.mlp_ws, b.mlp_bytes, st,
                          b.row_token, tm);
        if (rc != MOE355_OK) return rc;
        return gmm2_w4_impl(b.q1, (const uint8_t*)l.w2, (const float*)l.s2, l.group2, nullptr, b.q1_scale, b.expert_tokens,
                            MOE355_GL_COUNT, R, I, H, E, b.o, l.x_dtype, st, tm);
    }
    const bool list = l.weights == W_INT8_LIST;
    rc = gmm1_impl(b.xq, list ? nullptr : (const int8_t*)l.w13, list ? (const int8_t* const*)l.w13 : nullptr,
                   list ? nullptr : (const float*)l.s13, list ? (const float* const*)l.s13 : nullptr, b.x_scale,
                   b.expert_tokens, MOE355_GL_COUNT, R, H, 2 * I, E, l.swiglu_limit, b.q1, b.q1_scale, b.mlp_ws,
                   b.mlp_bytes, st, b.row_token, tiles_ready, b.plan, b.meet);
    if (rc != MOE355_OK) return rc;
    return gmm2_impl(b.q1, list ? nullptr : (const int8_t*)l.w2, list ? (const int8_t* const*)l.w2 : nullptr,
                     list ? nullptr : (const float*)l.s2, list ? (const float* const*)l.s2 : nullptr, b.q1_scale,
                     b.expert_tokens, MOE355_GL_COUNT, R, I, H, E, b.o, l.x_dtype, b.gmm2_ws, b.gmm2_bytes, st,
                     tiles_ready);
}

}  // namespace

extern "C" size_t moe355_layer_workspace(const moe355_layer* layer, int64_t num_tokens)
{
    if (check_layer(layer) != MOE355_OK || num_tokens <= 0) return 256;
    return lay_out(*layer, forms_of(*layer, num_tokens), num_tokens, nullptr).total;
}

extern "C" const char* moe355_layer_kernel_name(const moe355_layer* layer, int64_t num_tokens)
{
    if (check_layer(layer) != MOE355_OK || num_tokens <= 0) return "";
    const moe355_layer& l = *layer;
    const Forms f = forms_of(l, num_tokens);
    if (f.few) return l.shared ? "few_up_kernel with the shared expert" : "few_up_kernel";
    if (l.weights == W_INT4) return f.pairs ? "gmm_w4_pairs_kernel" : "gmm_w4_stream_kernel";
    if (f.pairs) return f.merged ? "gmm_stream_kernel with the shared expert" : "gmm_stream_kernel";
    return moe355_gmm_kernel_name(1, num_tokens * l.top_k, l.hidden, 2 * l.intermediate, l.num_experts);
}

extern "C" int moe355_layer_gates_inside(const moe355_layer* layer, int64_t num_tokens)
{
    if (check_layer(layer) != MOE355_OK || num_tokens <= 0) return 0;
    return forms_of(*layer, num_tokens).few && few_gates(few_args(*layer, Buffers{}, num_tokens));
}

extern "C" int moe355_layer_forward(const moe355_layer* layer, const void* x, const void* logits, int logits_dtype,
                                    int64_t num_tokens, void* out, void* workspace, size_t workspace_bytes,
                                    void* stream)
{
    int rc = check_layer(layer);
    if (rc != MOE355_OK) return rc;
    if (num_tokens < 0) return MOE355_E_ARG;
    if (num_tokens == 0) return MOE355_OK;
    const moe355_layer& l = *layer;
    const int64_t T = num_tokens, R = T * l.top_k;
    if (!x || !out || (!logits && !l.gate_weight)) return MOE355_E_ARG;
    if (R >= 0x7fffffffLL) return MOE355_E_SHAPE;
    const Forms f = forms_of(l, T);
    Buffers b = lay_out(l, f, T, workspace);
    b.plan.looks = take_meeting_looks();
    if (!workspace || ((uintptr_t)workspace & 255) || workspace_bytes < b.total) return MOE355_E_WORKSPACE;

    // measurement hook: the armed events are the routed gate_up product's, whatever is launched in front of it
    hipEvent_t ev0, ev1;
    take_profile_events(ev0, ev1);
    GateCall g = {x, logits, l.bias, l.x_dtype, logits_dtype, T, l.hidden, l.num_experts, l.top_k, l.k_group,
                  l.group_count, 1, l.renorm, l.norm_type, l.routed_scaling_factor, l.eps};
    if (l.gate_weight) {
        rc = router_gate_impl(x, l.x_dtype, l.gate_weight, l.gate_bias, T, (int)l.hidden, l.num_experts, b.logits, b.gate_ws,
                              b.gate_bytes, &g.n_planes, stream);
        if (rc != MOE355_OK) return rc;
        g.logits = g.n_planes ? b.gate_ws : b.logits;
        g.plane_bias = g.n_planes ? l.gate_bias : nullptr;
        g.logits_dtype = MOE355_DT_F32;
    }
    FewArgs few = {};
    if (f.few) {
        few = few_args(l, b, T);
        few.out = (uint16_t*)out;
    }
    const bool gates_itself = f.few && few_gates(few);
    if (!gates_itself) {
        rc = gate_quant_impl(f.small, g, 1, b.topk_weights, b.topk_ids, b.xq, b.x_scale, b.dst, b.row_token,
                             b.expert_tokens, l.sync_counter, l.shared ? b.one_group : nullptr, stream);
        if (rc != MOE355_OK) return rc;
    }
    if (f.few) {
        // the shared expert rides in the same two launches, whatever stream it was meant for
        (void)moe355_profile_next_gemm(ev0, ev1);
        return few_forward(few, gates_itself ? &g : nullptr, (hipStream_t)stream);
    }

    ForkJoinLease lease;
    bool joined = true;
    if (f.merged) {
        // in the GEMM launches of the routed experts, whatever stream it was meant for: 45 us of launches of its own
        // become the time of its weights
    } else if (l.shared == 2) {
        hipStream_t side = (hipStream_t)l.shared_stream, main = (hipStream_t)stream;
        if (!lease.take() || hipEventRecord(lease.fj.fork, main) != hipSuccess ||
            hipStreamWaitEvent(side, lease.fj.fork, 0) != hipSuccess)
            return MOE355_E_LAUNCH;
        // Products of the routed experts that end after some 50 us do not cover a dense product that leaves most of the chip
        // idle.  Experts of 4096 / 2048, two slots, us a call with `beside` / without: 8 experts, 200 / 256 / 320 / 600 tokens
        // 159 / 174 / 130 / 171 against 100 / 107 / 113 / 166; 16 experts, 700 tokens 156 against 173.
        const int64_t routed_bytes = 3 * l.num_experts * l.hidden * l.intermediate / (l.weights == W_INT4 ? 2 : 1);
        rc = shared_expert(l, f, b, T, side, routed_bytes >= (1ll << 28), false);
        // joined below even if a launch was refused: the caller frees the scratch in the order of its own stream
        if (hipEventRecord(lease.fj.join, side) != hipSuccess) return MOE355_E_LAUNCH;
        joined = false;
    }
    bool tiles_ready = false;
    if (rc == MOE355_OK && !f.pairs && !f.small) {
        TileSpec specs[2];
        int n = 0;
        if (l.weights == W_INT4) {
            specs[n++] = w4_chunk_spec(R, l.num_experts, b.gmm2_ws);
        } else {
            n = gemm_tile_specs(R, l.hidden, 2 * l.intermediate, l.num_experts,
                                gmm1_tile_ws(b.mlp_ws, R, 2 * l.intermediate), specs, b.plan.tile_rows);
            n += gemm_tile_specs(R, l.intermediate, l.hidden, l.num_experts, b.gmm2_ws, specs + n);
        }
        rc = route_map_impl(b.topk_ids, T, l.top_k, l.num_experts, 1, b.dst, b.row_token, b.expert_tokens, b.map_ws,
                            b.map_bytes, specs, n, &tiles_ready, stream, b.meet, b.meet_words);
    }
    // behind the maps, whose launch clears the words that its workgroups meet at
    if (rc == MOE355_OK && l.shared == 1 && !f.merged) rc = shared_expert(l, f, b, T, stream, false, tiles_ready);
    if (rc == MOE355_OK) {
        (void)moe355_profile_next_gemm(ev0, ev1);
        rc = f.pairs ? routed_pairs(l, f, b, T, stream) : routed_sorted(l, b, T, tiles_ready, stream);
    }
    if (!joined && hipStreamWaitEvent((hipStream_t)stream, lease.fj.join, 0) != hipSuccess) return MOE355_E_LAUNCH;
    if (rc != MOE355_OK) return rc;
    const void* residual = l.shared ? b.sh_out : nullptr;
    return unpermute_impl(b.o, l.x_dtype, f.pairs ? nullptr : b.dst, b.topk_weights, T, l.top_k, l.hidden, R, residual,
                          out, f.pairs ? b.topk_ids : nullptr, l.num_experts, nullptr, b.expert_tokens, l.load, stream);
}
