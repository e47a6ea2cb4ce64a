// Host entries that the layer call (layer.hip) shares with the exported operators: the same launches, with the
// options that only a whole layer has (per-expert weight tables in pair order, the group list of a dense product
// written by the routing launch, expert loads added up by the combine).
#pragma once

#include "tile_map.h"

namespace moe355 {

// Chunk results of the router gate that the gating launch adds up itself, all of them in flight at once.  With more of them
// the reduction in a launch of its own is faster: us a call with it / without, 8 planes (H = 1024, 8 experts) 1000 tokens 57 /
// 53.8; 16 planes (128 experts) 1 / 4 / 60 / 777 tokens 24.9 / 46.9 / 117.4 / 154.3 against 24.1 / 46.2 / 116.8 / 153.7; 56
// planes (256 experts; eight in flight at a time) one token 79 against 91.
constexpr int kGatePlanes = 16;

// hidden states and logits of a batch, and how the router scores and groups the experts
struct GateCall {
    const void* x;       // [T, H] bf16 / fp16
    const void* logits;  // [T, E]
    const void* bias;    // [E] in the dtype of the logits, or null
    int x_dtype, logits_dtype;
    int64_t num_tokens, hidden;
    int num_experts, top_k, k_group, group_count, group_select_mode, renorm, norm_type;
    float routed_scaling_factor, eps;
    // (at most kGatePlanes:) fp32 logits that are still the router gate's chunk results: n_planes planes [T, E] at `logits`, to be added in
    // ascending order from +0, and plane_bias [E] last (or null); 0: `logits` holds the logits
    int n_planes;
    const float* plane_bias;
};

// moe355_router_gate; with n_planes, a launch that leaves the logits as chunk results says how many there are (0: none,
// `logits` holds them) instead of adding them up: the gating launch behind it does that while it reads them
int router_gate_impl(const void* x, int x_dtype, const float* weight, const float* bias, int64_t num_tokens, int hidden,
                     int num_experts, float* logits, void* workspace, size_t workspace_bytes, int* n_planes, void* stream);

// what the gating launches take of such a call, and what they refuse (num_tokens > 0)
int check_gate(const GateCall& g);

// sort: the whole of moe355_route_quant_small; otherwise gating and quantisation only (any number of tokens).
// one_group: receives num_tokens on the device, or null.
int gate_quant_impl(bool sort, const GateCall& g, int tokens_num_type, void* topk_weights, int32_t* topk_ids,
                    int8_t* xq, float* x_scale, int32_t* expanded_row_idx, int32_t* row_token, int64_t* expert_tokens,
                    int32_t* sync_counter, int64_t* one_group, void* stream);

// sorted_indices null: pair order (hist_ids = the ids, counts to hist_out unless that is null).  load [hist_experts]: the counts of this
// batch are added to it (from hist_ids, or load_counts where the rows are sorted).
int unpermute_impl(const void* permuted, int dtype, const int32_t* sorted_indices, const void* probs,
                   int64_t num_tokens, int top_k, int64_t hidden, int64_t permuted_rows, const void* residual,
                   void* out, const int32_t* hist_ids, int hist_experts, int64_t* hist_out, const int64_t* load_counts,
                   int64_t* load, void* stream);

// Weights of a pair-order GEMM: one tiled tensor with its scales, or device tables of per-expert tensors.
struct PairWeights {
    const int8_t* one;
    const float* scale;
    const int8_t* const* list = nullptr;
    const float* const* scale_list = nullptr;
    bool complete() const { return (one && scale) || (list && scale_list); }
    bool aligned() const { return !((uintptr_t)one & 15) && !((uintptr_t)scale & 15); }
};

// The shared expert in the two pair-order launches (one GEMM each): tensors of a routed expert's shape.
struct PairShared {
    const int8_t* w;
    const float* scale;
    float limit = 0.0f;
    bool aligned() const { return !((uintptr_t)w & 15) && !((uintptr_t)scale & 15); }
    template <typename Args>
    void into(Args& a, int num_tokens) const
    {
        a.sh_w = w;
        a.sh_scale = scale;
        a.sh_limit = limit;
        a.sh_rows = num_tokens;
        a.sh_blocks = (num_tokens + 31) / 32;
    }
};

// moe355_pair_order; with_shared: the launches take a shared expert of a routed expert's shape along
bool pair_order_impl(int64_t num_tokens, int top_k, int num_logits, int num_experts, int64_t hidden, int64_t intermediate,
                     bool with_shared);
// with `shared`, y, out and out_scale hold num_tokens more rows (the shared expert's, in token order); the same for x,
// per_token_scale and out of the second
int gmm1_pairs_impl(const int8_t* x, const float* x_scale, const int32_t* topk_ids, int64_t num_tokens, int top_k,
                    const PairWeights& w, int64_t k, int64_t n, int num_experts, float swiglu_limit, float* y,
                    int8_t* out, float* out_scale, void* stream, const PairShared* shared = nullptr);
int gmm2_pairs_impl(const int8_t* x, const float* per_token_scale, const float* y, const PairWeights& w,
                    const int32_t* topk_ids, int64_t num_tokens, int top_k, int64_t k, int64_t n, int num_experts,
                    void* out, int out_dtype, void* stream, const PairShared* shared = nullptr);
// the gate_up product whose tiles' workgroups exchange the rows' maxima: rows of its tiles and workgroups of a tile (0: they do not),
// a word for each of them and every row in `meet`, cleared before the launch
struct MeetingPlan {
    int tile_rows = 0, columns = 0, looks = 0;
};
int take_meeting_looks();  // how often the workgroups of this thread's next call look for the others' maxima
MeetingPlan meeting_plan(int64_t rows, int64_t k, int64_t n, int num_experts);
// the same for the shared expert's, one expert that owns every row: columns, or 0; meet: [columns][rows], cleared before the launch
int shared_meeting_columns(int64_t rows, int64_t k, int64_t n);
int shared_meeting_impl(const int8_t* x, const int8_t* weight_nz, const float* weight_scale, const float* x_scale,
                        const int64_t* group_list, int64_t rows, int64_t k, int64_t n, float limit, uint32_t* meet, int looks,
                        int8_t* out, float* out_scale, void* stream);
// plan, meet: used where the tile map is ready, which it is where there is a plan and the layer sorts
int gmm1_impl(const int8_t* x, const int8_t* weight_nz, const int8_t* const* weight_list, const float* weight_scale,
              const float* const* scale_list, const float* x_scale, const int64_t* group_list, int group_list_type,
              int64_t rows, int64_t k, int64_t n, int num_experts, float swiglu_limit, int8_t* out, float* out_scale,
              void* workspace, size_t workspace_bytes, void* stream, const int32_t* row_src = nullptr,
              bool tiles_ready = false, const MeetingPlan& plan = {}, uint32_t* meet = nullptr);
// beside: the launch runs on a side stream, beside long products of the routed experts
int gmm2_impl(const int8_t* x, const int8_t* weight_nz, const int8_t* const* weight_list, const float* scale,
              const float* const* scale_list, const float* per_token_scale, const int64_t* group_list,
              int group_list_type, int64_t rows, int64_t k, int64_t n, int num_experts, void* out, int out_dtype,
              void* workspace, size_t workspace_bytes, void* stream, bool tiles_ready = false, bool beside = false);
int gmm_i32_impl(const int8_t* x, const int8_t* weight_nz, const int64_t* group_list, int group_list_type, int64_t rows,
                 int64_t k, int64_t n, int num_experts, int32_t* acc, void* workspace, size_t workspace_bytes, void* stream,
                 bool beside);
void* gmm1_tile_ws(void* workspace, int64_t rows, int64_t n);
// the tile map (0 or 1) that a grouped product will look for in its workspace
int gemm_tile_specs(int64_t rows, int64_t k, int64_t n, int num_experts, void* tile_ws, TileSpec* specs, int tile_rows = 0);

// int4 weights, sorted rows (gmm_w4.hip): the chunks of both products in the order they run in, for the routing launch to build
// in a workspace of tiled_workspace_bytes(rows, E, 64); without it (null) every workgroup finds its chunk from the group list
TileSpec w4_chunk_spec(int64_t rows, int num_experts, void* workspace);
int gmm1_w4_impl(const int8_t* x, const uint8_t* weight_nz4, const float* weight_scale, int64_t group_size,
                 const float* bias, const float* x_scale, const int64_t* group_list, int group_list_type, int64_t rows,
                 int64_t k, int64_t n, int num_experts, float swiglu_limit, int8_t* out, float* out_scale, void* workspace,
                 size_t workspace_bytes, void* stream, const int32_t* row_src, const TileMap* chunks);
int gmm2_w4_impl(const int8_t* x, const uint8_t* weight_nz4, const float* scale, int64_t group_size, const float* bias,
                 const float* per_token_scale, const int64_t* group_list, int group_list_type, int64_t rows, int64_t k,
                 int64_t n, int num_experts, void* out, int out_dtype, void* stream, const TileMap* chunks);

// int4 weights, pair order (gmm_w4.hip)
bool w4_pairs_supported(int64_t num_tokens, int top_k, int num_experts, int64_t hidden, int64_t intermediate,
                        int64_t group13, int64_t group2);
int gmm1_w4_pairs(const int8_t* x, const float* x_scale, const int32_t* topk_ids, int64_t num_tokens, int top_k,
                  const uint8_t* w, const float* scale, int64_t group, int64_t k, int64_t n, int num_experts,
                  float swiglu_limit, float* y, int8_t* out, float* out_scale, hipStream_t st);
int gmm2_w4_pairs(const int8_t* x, const float* x_scale, const int32_t* topk_ids, int64_t num_tokens, int top_k,
                  const uint8_t* w, const float* scale, int64_t group, int64_t k, int64_t n, int num_experts, void* out,
                  int out_dtype, hipStream_t st);

// moe355_route_map with the tile maps of the two products (nspecs of them, at most 2) built by the same launch where it
// is one launch (one_launch_map; returns 1 in *built then), which also clears zeros_per_pair words for every pair
bool one_launch_map(int64_t pairs, int num_experts);
int route_map_impl(const int32_t* expert_idx, int64_t num_tokens, int top_k, int num_experts, int tokens_num_type,
                   int32_t* expanded_row_idx, int32_t* row_token, int64_t* expert_tokens, void* workspace,
                   size_t workspace_bytes, const TileSpec* specs, int nspecs, bool* built, void* stream, uint32_t* zeros = nullptr,
                   int zeros_per_pair = 0);

// ------------------------------------------------------------------ a few tokens (few.hip)
// n / d for n and d below 2^16 in one multiplication (an integer division is about 25 instructions, one after the other)
struct SmallDivisor {
    uint32_t m = 0;
    SmallDivisor() = default;
    explicit SmallDivisor(uint32_t d) : m(d > 1 ? (uint32_t)(((1ull << 32) + d - 1) / d) : 0) {}
    __device__ int operator()(int n) const { return m ? (int)__umulhi((uint32_t)n, m) : n; }
};

struct FewArgs {
    const int8_t* xq;        // [T, H]
    const float* x_scale;    // [T]
    const int32_t* ids;      // [T, k]
    const uint16_t* tw;      // [T, k] routing weights, 16 bits
    int T, k, R, E, H, I, S; // R = T * k; S: width of the shared expert
    const int8_t *w13, *w2;  // tiled tensors with their scales, or device tables of per-expert tensors
    const float *s13, *s2;
    const int8_t* const* w13_list;
    const float* const* s13_list;
    const int8_t* const* w2_list;
    const float* const* s2_list;
    float limit;
    const int8_t *sw13, *sw2;  // shared expert, or null
    const float *ss13, *ss2;
    float sh_limit, sh_alpha, sh_beta;
    float* y;                // [R, I] SwiGLU values, then [T, S]
    float* ymax;             // [R, I / 16] maxima of 16 values each, then [T, S / 16]
    int8_t* q1;              // [R, I] then [T, S]
    float* q1_scale;         // [R + T]
    uint16_t* out;           // [T, H]
    int f16;
    int64_t* load;           // [E] or null: the rows of every expert are added
    // divisions by k, I / 4, I / 16, S / 4, S / 16 and the items of an expert's K range (few_forward)
    SmallDivisor by_k, by_i4, by_i16, by_s4, by_s16, by_parts;
};

bool few_supported(const FewArgs& a);
// whether few_forward takes the gating and the token quantisation of such a call as well
bool few_gates(const FewArgs& a);
// gate: the call that few_forward gates and quantises for itself (ids and weights go to a.ids and a.tw), or null
int few_forward(const FewArgs& a, const GateCall* gate, hipStream_t st);

}  // namespace moe355
