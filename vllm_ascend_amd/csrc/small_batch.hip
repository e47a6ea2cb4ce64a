// Small batches (decode): router and dispatch in one launch.
//
// The reference runs the gating op, then the init-routing op (histogram, stable sort, gather with the first int8
// quantisation), and the expert GEMM reads the gathered copy.  For a few hundred (token, slot) pairs that is two
// launches of a few microseconds each in front of a weight stream of some tens of microseconds.  Here one launch
// does both:
//   - ceil(T / 4) workgroups (every fifth of the grid) gate four token rows each (one per wavefront, the arithmetic of the gating
//     kernel) and then count themselves on a counter; the one that finds all the others done sorts the T * k pairs
//     by expert, stably: per-chunk histograms in LDS (a chunk = 64 consecutive pairs), a scan over (chunk, expert),
//     ballot-matched ranks inside a chunk.  Nobody waits for anybody: a workgroup that is not the last one ends;
//   - the other T workgroups quantise one token row each, ONCE, in token order.  The rows are not copied k times
//     into the expert-sorted order: the expert GEMM reads row r of that order through row_token[r].
// The results are the ones the two separate ops give: topk weights and ids, expanded_row_idx, the per-expert
// counts, and (through row_token) the int8 rows and scales of the expert-sorted activation.
// The counter is one int32 that the caller keeps at zero between calls (the sorting workgroup puts it back).
#include <type_traits>

#include "gating_body.h"
#include "layer_parts.h"

namespace moe355 {

constexpr int kSmallThreads = 256;
constexpr int kSmallWaves = kSmallThreads / 64;
constexpr int kSmallMaxPairs = 1024;
constexpr int kSmallChunks = kSmallMaxPairs / 64;
constexpr int kSmallMaxExperts = 256;  // the sorting workgroup's tables stay well below 64 KiB of LDS

struct SmallRouteArgs {
    const void* x;        // [T, H] bf16 / fp16
    const void* logits;   // [T, E]
    const void* bias;     // [E] or null (logits dtype)
    int T, H, E, k, k_group, G, mode, renorm, norm_type;
    float rsf, eps;
    int tokens_num_type;
    void* topk_weights;   // [T, k] in the dtype of x
    int x_dtype;
    int32_t* topk_ids;    // [T, k]
    int8_t* xq;           // [T, H]
    float* x_scale;       // [T]
    int32_t* dst;         // [T * k] expanded_row_idx
    int32_t* row_token;   // [T * k] token of every expert-sorted row
    int64_t* expert_tokens;  // [E]
    int32_t* arrived;     // one int32, zero between calls
    int64_t* one_group;   // or null: receives T (the group list of a dense product over all tokens)
    int n_planes;         // GateCall
    const float* plane_bias;
    int wave_rows;        // the quantising workgroups take four rows each, one per wavefront
};

// 16-byte pieces of a row that a thread of its workgroup requests at once and holds: rows of up to 8192 values are read
// once.  The launch of rows of 7168 values, 256 experts without groups, 1 / 64 / 512 / 4096 tokens, us with one piece
// held and the others read twice / so: 3.78 / 4.15 / 5.20 / 20.24 against 3.29 / 3.92 / 4.43 / 17.24.
constexpr int kHeld = 4;

// LDS of a gating wavefront (gate_row_wave)
__host__ __device__ constexpr int gate_row_floats(int E) { return E <= 192 ? 192 : (E + 3) & ~3; }

// the quantiser of the layer on one row, by the whole workgroup
template <int DT>
__device__ __forceinline__ void quantise_token_row(const SmallRouteArgs& a, int t, float* lds16)
{
    const int tid = threadIdx.x;
    const int64_t nv = a.H >> 3;
    const v8u16* xv = (const v8u16*)((const uint16_t*)a.x + (int64_t)t * a.H);
    v8u16 held[kHeld];  // requested at once
#pragma unroll
    for (int i = 0; i < kHeld; ++i)
        held[i] = i * kSmallThreads + tid < nv ? xv[i * kSmallThreads + tid] : (v8u16){0, 0, 0, 0, 0, 0, 0, 0};
    float amax = 0.0f;
    auto largest = [&](v8u16 v) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float f = __builtin_fabsf(half_to_f32<DT>(v[j]));
            amax = f > amax ? f : amax;
        }
    };
#pragma unroll
    for (int i = 0; i < kHeld; ++i) largest(held[i]);
    for (int64_t i = kHeld * kSmallThreads + tid; i < nv; i += kSmallThreads) largest(xv[i]);
    amax = wave_max(amax);
    if ((tid & 63) == 0) lds16[tid >> 6] = amax;
    __syncthreads();
    amax = lds16[0];
#pragma unroll
    for (int w = 1; w < kSmallWaves; ++w) amax = lds16[w] > amax ? lds16[w] : amax;
    const float s = amax / 127.0f;
    const RowDivisor d = row_divisor(s);
    if (tid == 0) a.x_scale[t] = (amax == 0.0f) ? 0.0f : s;
    uint2* qv = (uint2*)(a.xq + (int64_t)t * a.H);
    auto emit = [&](auto fast) {
#pragma unroll
        for (int i = 0; i < kHeld; ++i)
            if (i * kSmallThreads + tid < nv)
                qv[i * kSmallThreads + tid] = quantise_by_row<decltype(fast)::value, DT>(held[i], d);
        for (int64_t i = kHeld * kSmallThreads + tid; i < nv; i += kSmallThreads)
            qv[i] = quantise_by_row<decltype(fast)::value, DT>(xv[i], d);
    };
    if (d.fast) emit(std::true_type{});
    else emit(std::false_type{});
}

// The same on one row by a wavefront (H <= 2048): a lane requests up to four pieces at once and there is no barrier.
template <int DT>
__device__ __forceinline__ void quantise_token_row_wave(const SmallRouteArgs& a, int t, int lane)
{
    if (t >= a.T) return;
    const int nv = a.H >> 3;
    const v8u16* xv = (const v8u16*)((const uint16_t*)a.x + (int64_t)t * a.H);
    v8u16 held[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) held[i] = i * 64 + lane < nv ? xv[i * 64 + lane] : (v8u16){0, 0, 0, 0, 0, 0, 0, 0};
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float f = __builtin_fabsf(half_to_f32<DT>(held[i][j]));
            amax = f > amax ? f : amax;
        }
    amax = wave_max(amax);
    const float s = amax / 127.0f;
    const RowDivisor d = row_divisor(s);
    if (lane == 0) a.x_scale[t] = (amax == 0.0f) ? 0.0f : s;
    uint2* qv = (uint2*)(a.xq + (int64_t)t * a.H);
    auto emit = [&](auto fast) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (i * 64 + lane < nv) qv[i * 64 + lane] = quantise_by_row<decltype(fast)::value, DT>(held[i], d);
    };
    if (d.fast) emit(std::true_type{});
    else emit(std::false_type{});
}

// LDT: dtype of the logits; XDT: dtype of the hidden states (and of the weights that are returned)
template <int LDT, int PER, int XDT>
__global__ __launch_bounds__(kSmallThreads) void route_quant_small_kernel(SmallRouteArgs a)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int gate_wgs = (a.T + kSmallWaves - 1) / kSmallWaves;
    if ((int)blockIdx.x >= gate_wgs) {
        const int wg = (int)blockIdx.x - gate_wgs;
        if (a.wave_rows) quantise_token_row_wave<XDT>(a, wg * kSmallWaves + (int)(threadIdx.x >> 6), threadIdx.x & 63);
        else quantise_token_row<XDT>(a, wg, lds);
        return;
    }
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int E = a.E, k = a.k, R = a.T * a.k;
    if (a.one_group && blockIdx.x == 0 && tid == 0) *a.one_group = a.T;
    // ---------------- gating: one row per wavefront
    {
        const int row = (int)blockIdx.x * kSmallWaves + wave;
        if (row < a.T)
            gate_row_wave<LDT, PER>(RowLogits<LDT>{a.logits, (int64_t)row * E, (int64_t)a.T * E, a.n_planes, a.plane_bias},
                                    a.bias, E, k,
                                    a.k_group, a.G, a.mode, a.renorm, a.norm_type, a.rsf, a.eps, (int64_t)row * k,
                                    a.topk_weights, a.x_dtype, a.topk_ids, lds + wave * gate_row_floats(E), lane);
    }
    if (!a.arrived) return;  // gating and quantisation only (moe355_gate_quant): the maps come from another launch
    // This workgroup's ids have reached memory before it is counted: every thread waits for its own stores, the
    // barrier collects the workgroup, and the counting thread issues a device-scope release fence in front of the
    // atomic (the ids are written with device-scope stores already; the fence is what the memory model asks for,
    // so that the hand-off does not rest on how those stores happen to be compiled).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int32_t* flag = (int32_t*)lds;
    if (tid == 0) {
        __threadfence();
        *flag = atomicAdd(a.arrived, 1) == gate_wgs - 1;
    }
    __syncthreads();
    if (!*flag) return;
    __threadfence();  // acquire side: the reads below come after the count that this workgroup has observed
    __syncthreads();
    // ---------------- the last gating workgroup sorts the R pairs (stable counting sort by expert)
    int32_t* ids_l = (int32_t*)lds;             // [kSmallMaxPairs]
    int32_t* hist = ids_l + kSmallMaxPairs;     // [16][E]: chunk histograms, then rows of the expert in earlier chunks
    int32_t* total = hist + kSmallChunks * E;   // [E]: rows of each expert, then its first row
    int32_t* partial = total + E;               // [16] scan scratch
    for (int i = tid; i < kSmallChunks * E; i += kSmallThreads) hist[i] = 0;
    for (int f = tid; f < R; f += kSmallThreads)
        ids_l[f] = __hip_atomic_load(a.topk_ids + f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int passes = (R + kSmallThreads - 1) / kSmallThreads;  // pair f = pass * 256 + tid, chunk = f / 64
    for (int ps = 0; ps < passes; ++ps) {
        const int f = ps * kSmallThreads + tid;
        if (f < R) {
            const int e = ids_l[f];
            if (e >= 0 && e < E) atomicAdd(&hist[(f >> 6) * E + e], 1);
        }
    }
    __syncthreads();
    for (int e = tid; e < E; e += kSmallThreads) {
        int32_t run = 0;
#pragma unroll
        for (int c = 0; c < kSmallChunks; ++c) {
            const int32_t n = hist[c * E + e];
            hist[c * E + e] = run;
            run += n;
        }
        total[e] = run;
    }
    __syncthreads();
    const int32_t mine = tid < E ? total[tid] : 0;  // E <= 256 = the number of threads
    int32_t all;
    const int32_t first = block_scan_exclusive_i32(mine, partial, all);
    if (tid < E) {
        total[tid] = first;
        a.expert_tokens[tid] = a.tokens_num_type == 1 ? (int64_t)mine : (int64_t)(first + mine);
    }
    __syncthreads();
    // rank inside the chunk: lanes with the same expert find each other with ballots
    int nbits = 0;
    while ((1 << nbits) < E) ++nbits;
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int ps = 0; ps < passes; ++ps) {
        const int f = ps * kSmallThreads + tid;
        int e = -1;
        if (f < R) {
            e = ids_l[f];
            if (e < 0 || e >= E) e = -1;  // cannot happen for ids that the gate chose; kept for symmetry with the op
        }
        const bool valid = e >= 0;
        unsigned long long same = __ballot(valid);
        for (int b = 0; b < nbits; ++b) {
            const bool bit = (e >> b) & 1;
            const unsigned long long bal = __ballot(valid && bit);
            same &= bit ? bal : ~bal;
        }
        if (f < R) {
            int32_t d = R;  // a dropped pair points one past the last row
            if (valid) {
                d = total[e] + hist[(f >> 6) * E + e] + __popcll(same & below);
                a.row_token[d] = f / k;
            }
            a.dst[f] = d;
        }
    }
    if (tid == 0) *a.arrived = 0;  // ready for the next call
}

}  // namespace moe355

using namespace moe355;

extern "C" int moe355_gate_quant_supported(int64_t num_tokens, int top_k, int num_experts)
{
    return num_tokens > 0 && num_tokens < (1 << 30) && top_k > 0 && top_k <= 64 && num_experts > 0 &&
           num_experts <= kSmallMaxExperts && top_k <= num_experts;
}

extern "C" int moe355_route_quant_small_supported(int64_t num_tokens, int top_k, int num_experts)
{
    return num_tokens > 0 && top_k > 0 && top_k <= 64 && num_tokens * top_k <= kSmallMaxPairs && num_experts > 0 &&
           num_experts <= kSmallMaxExperts && top_k <= num_experts;
}

int moe355::check_gate(const GateCall& g)
{
    if (g.num_tokens < 0 || g.hidden <= 0 || g.num_experts <= 0 || g.top_k <= 0) return MOE355_E_ARG;
    if (g.norm_type != 0 && g.norm_type != 1) return MOE355_E_ARG;
    if (g.group_select_mode != 0 && g.group_select_mode != 1) return MOE355_E_ARG;
    if (g.group_count <= 0 || g.k_group <= 0 || g.k_group > g.group_count) return MOE355_E_ARG;
    if (g.x_dtype != MOE355_DT_BF16 && g.x_dtype != MOE355_DT_F16) return MOE355_E_UNSUPPORTED;
    if (g.logits_dtype < MOE355_DT_F32 || g.logits_dtype > MOE355_DT_F16) return MOE355_E_ARG;
    if (g.num_tokens == 0) return MOE355_OK;
    if (!moe355_gate_quant_supported(g.num_tokens, g.top_k, g.num_experts)) return MOE355_E_SHAPE;
    if (g.group_count > 64 || g.num_experts % g.group_count != 0) return MOE355_E_SHAPE;
    if (g.hidden % 8 != 0 || ((uintptr_t)g.x & 15)) return MOE355_E_SHAPE;
    if (!g.x || !g.logits) return MOE355_E_ARG;
    return MOE355_OK;
}

int moe355::gate_quant_impl(bool sort, const GateCall& g, int tokens_num_type, void* topk_weights, int32_t* topk_ids,
                            int8_t* xq, float* x_scale, int32_t* expanded_row_idx, int32_t* row_token,
                            int64_t* expert_tokens, int32_t* sync_counter, int64_t* one_group, void* stream)
{
    const void *x = g.x, *logits = g.logits, *bias = g.bias;
    const int x_dtype = g.x_dtype, logits_dtype = g.logits_dtype, num_experts = g.num_experts, k = g.top_k;
    const int k_group = g.k_group, group_count = g.group_count, group_select_mode = g.group_select_mode;
    const int renorm = g.renorm, norm_type = g.norm_type;
    const int64_t num_tokens = g.num_tokens, hidden = g.hidden;
    if (tokens_num_type != 0 && tokens_num_type != 1) return MOE355_E_UNSUPPORTED;
    int rc = check_gate(g);
    if (rc != MOE355_OK || num_tokens == 0) return rc;
    if (sort && !moe355_route_quant_small_supported(num_tokens, k, num_experts)) return MOE355_E_SHAPE;
    if ((uintptr_t)xq & 7) return MOE355_E_SHAPE;
    if (!topk_weights || !topk_ids || !xq || !x_scale) return MOE355_E_ARG;
    if (sort && (!expanded_row_idx || !row_token || !expert_tokens || !sync_counter)) return MOE355_E_ARG;
    SmallRouteArgs a = {};
    a.x = x;
    a.logits = logits;
    a.bias = bias;
    a.n_planes = g.n_planes;
    a.plane_bias = g.plane_bias;
    a.T = (int)num_tokens;
    a.H = (int)hidden;
    a.E = num_experts;
    a.k = k;
    a.k_group = k_group;
    a.G = group_count;
    a.mode = group_select_mode;
    a.renorm = renorm;
    a.norm_type = norm_type;
    a.rsf = g.routed_scaling_factor;
    a.eps = g.eps;
    a.tokens_num_type = tokens_num_type;
    a.topk_weights = topk_weights;
    a.x_dtype = x_dtype;
    a.topk_ids = topk_ids;
    a.xq = xq;
    a.x_scale = x_scale;
    a.dst = expanded_row_idx;
    a.row_token = row_token;
    a.expert_tokens = expert_tokens;
    a.arrived = sort ? sync_counter : nullptr;
    a.one_group = one_group;
    const int E = num_experts;
    int per = 1;
    while (64 * per < E) per *= 2;
    // LDS: the sorting tables; the gating rows need gate_row_floats(E) per wavefront and the quantiser 4 floats (less)
    const size_t lds_bytes = sort ? ((size_t)kSmallMaxPairs + (size_t)kSmallChunks * E + E + 16) * 4
                                  : ((size_t)kSmallWaves * gate_row_floats(E) + 16) * 4;
    const int64_t quads = (num_tokens + kSmallWaves - 1) / kSmallWaves;
    // A workgroup per row has 16 bytes per thread in flight and a barrier in the middle; at 8192 tokens the launch takes 25.0 us
    // against 19.8 with a row per wavefront (H = 2048; H = 1024 14.7 against 10.9), at 2048 9.3 against 8.3, the same at 512
    // to 1024.  Below that, and for longer rows, the workgroup per row has more threads on a row.
    a.wave_rows = hidden <= 2048 && num_tokens >= 512;
    const dim3 grid((unsigned)(quads + (a.wave_rows ? quads : num_tokens)));
    hipStream_t st = (hipStream_t)stream;
#define MOE355_SMALL(L_, P_, X_)                                                                                  \
    hipLaunchKernelGGL((route_quant_small_kernel<L_, P_, X_>), grid, dim3(kSmallThreads), lds_bytes, st, a)
#define MOE355_SMALL_PER(L_, X_)                    \
    switch (per) {                                  \
        case 1: MOE355_SMALL(L_, 1, X_); break;     \
        case 2: MOE355_SMALL(L_, 2, X_); break;     \
        default: MOE355_SMALL(L_, 4, X_); break;    \
    }
#define MOE355_SMALL_X(L_)                                             \
    if (x_dtype == MOE355_DT_F16) { MOE355_SMALL_PER(L_, MOE355_DT_F16) } \
    else { MOE355_SMALL_PER(L_, MOE355_DT_BF16) }
    if (logits_dtype == MOE355_DT_F32) { MOE355_SMALL_X(MOE355_DT_F32) }
    else if (logits_dtype == MOE355_DT_BF16) { MOE355_SMALL_X(MOE355_DT_BF16) }
    else { MOE355_SMALL_X(MOE355_DT_F16) }
#undef MOE355_SMALL_X
#undef MOE355_SMALL_PER
#undef MOE355_SMALL
    return launch_status();
}

extern "C" int moe355_route_quant_small(const void* x, int x_dtype, const void* logits, int logits_dtype,
                                        const void* bias, int64_t num_tokens, int64_t hidden, int num_experts, int k,
                                        int k_group, int group_count, int group_select_mode, int renorm,
                                        int norm_type, float routed_scaling_factor, float eps, int tokens_num_type,
                                        void* topk_weights, int32_t* topk_ids, int8_t* xq, float* x_scale,
                                        int32_t* expanded_row_idx, int32_t* row_token, int64_t* expert_tokens,
                                        int32_t* sync_counter, void* stream)
{
    const GateCall g = {x, logits, bias, x_dtype, logits_dtype, num_tokens, hidden, num_experts, k, k_group, group_count,
                        group_select_mode, renorm, norm_type, routed_scaling_factor, eps};
    return gate_quant_impl(true, g, tokens_num_type, topk_weights, topk_ids, xq, x_scale, expanded_row_idx, row_token,
                           expert_tokens, sync_counter, nullptr, stream);
}

extern "C" int moe355_gate_quant(const void* x, int x_dtype, const void* logits, int logits_dtype, const void* bias,
                                 int64_t num_tokens, int64_t hidden, int num_experts, int k, int k_group,
                                 int group_count, int group_select_mode, int renorm, int norm_type,
                                 float routed_scaling_factor, float eps, void* topk_weights, int32_t* topk_ids,
                                 int8_t* xq, float* x_scale, void* stream)
{
    const GateCall g = {x, logits, bias, x_dtype, logits_dtype, num_tokens, hidden, num_experts, k, k_group, group_count,
                        group_select_mode, renorm, norm_type, routed_scaling_factor, eps};
    return gate_quant_impl(false, g, 1, topk_weights, topk_ids, xq, x_scale, nullptr, nullptr, nullptr, nullptr, nullptr,
                           stream);
}
