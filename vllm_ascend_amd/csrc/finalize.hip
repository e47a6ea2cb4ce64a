// Weighted un-permute (finalize routing): one workgroup per token, each lane
// owns runs of 8 hidden elements (16-byte loads), accumulating the k expert
// rows in fp32 in slot order.
#include "layer_parts.h"

namespace moe355 {

// TOPK > 0: the slot loop is unrolled and all TOPK row loads are issued before the first add,
// so their latencies overlap; TOPK == 0: generic loop.
// The rows are read once, past the caches: 8192 tokens of 8 x 2048 values (301 MB) 59.5 -> 54.5 us, 4096 of 8 x 7168 (587 MB)
// 117 -> 101, 512 of 8 x 7168 14.9 -> 14.1.  (Non-temporal stores as well: 54 and 111; rows in pieces: the same.)
// DT: bf16 or fp16 (rows, weights, residual and result share it).
constexpr int kHistMaxExperts = 2048;

// idx == nullptr: the rows lie in pair order (row of token t, slot s = t * top_k + s) and hist_ids holds their ids.
// hist_out [hist_experts] or load: one more workgroup (the last of the grid's x range) counts the pairs of every expert
// into the one and adds them to the other, next to the others instead of in a launch of its own.
struct UnpermuteArgs {
    int T, top_k, pieces, hist_experts;  // (gridDim would be a load of its own in front of everything else)
    const uint16_t* permuted;
    const int32_t* idx;
    const uint16_t* probs;
    const uint16_t* residual;
    uint16_t* out;
    const int32_t* hist_ids;
    int64_t H, permuted_rows;
    int64_t* hist_out;
    const int64_t* load_counts;
    int64_t* load;
};

// |index| as a row; INT32_MIN stays negative (no overflow that the compiler may build on), and a negative row is none
__device__ __forceinline__ int32_t row_of(int32_t index) { return index < 0 ? (int32_t)(0u - (uint32_t)index) : index; }

template <int TOPK, int DT = MOE355_DT_BF16>
__global__ __launch_bounds__(256) void token_unpermute_kernel(UnpermuteArgs a)
{
    const uint16_t* __restrict__ permuted = a.permuted;
    const int32_t* __restrict__ idx = a.idx;
    const uint16_t* __restrict__ probs = a.probs;
    const uint16_t* __restrict__ residual = a.residual;
    uint16_t* __restrict__ out = a.out;
    const int32_t* __restrict__ hist_ids = a.hist_ids;
    const int64_t H = a.H, permuted_rows = a.permuted_rows;
    const int hist_experts = a.hist_experts;
    if ((int)blockIdx.x == a.T) {
        int64_t* hist_out = a.hist_out;
        int64_t* load = a.load;
        __shared__ int32_t hcnt[kHistMaxExperts];
        if (blockIdx.y != 0) return;
        if (!hist_ids) {
            for (int e = threadIdx.x; e < hist_experts; e += 256) load[e] += a.load_counts[e];
            return;
        }
        for (int e = threadIdx.x; e < hist_experts; e += 256) hcnt[e] = 0;
        __syncthreads();
        for (int64_t f = threadIdx.x; f < permuted_rows; f += 256) {
            const int32_t e = hist_ids[f];
            if (e >= 0 && e < hist_experts) atomicAdd(&hcnt[e], 1);
        }
        __syncthreads();
        for (int e = threadIdx.x; e < hist_experts; e += 256) {
            if (hist_out) hist_out[e] = (int64_t)hcnt[e];
            if (load) load[e] += (int64_t)hcnt[e];
        }
        return;
    }
    const int64_t t = blockIdx.x;
    const int64_t nv = H >> 3;
    // few tokens: a row is cut into pieces, one workgroup each
    const int64_t first = (int64_t)blockIdx.y * 256 + threadIdx.x, step = 256 * (int64_t)a.pieces;
    auto load_residual = [&](int64_t i) {
        return residual ? ((const v8u16*)(residual + t * H))[i] : (v8u16){0, 0, 0, 0, 0, 0, 0, 0};
    };
    auto finish = [&](int64_t i, float (&acc)[8], v8u16 r) {
        if (residual) {
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] = acc[j] + half_to_f32<DT>(r[j]);
        }
        v8u16 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = f32_to_half<DT>(acc[j]);
        ((v8u16*)(out + t * H))[i] = o;
    };
    if constexpr (TOPK > 0) {
        // Rows, weights and ids of the slots are the same for the whole workgroup: every wavefront reads them into lanes, one load
        // each, in front of the rows.  In pair order the rows' addresses wait for nothing (a row that nobody computed is read
        // and left out).  With a barrier and LDS between the two, 64 tokens of 2 x 1024 values took 2.9 us and take 1.7; calls of
        // both in turn: the small layer, 64 tokens, 24.7 and 24.4 us, others the same within noise.
        const int lane = threadIdx.x & 63;
        const int64_t mine = t * TOPK + (lane < TOPK ? lane : TOPK - 1);
        int32_t d = idx ? idx[mine] : (int32_t)mine;
        int32_t e = !idx && hist_ids ? hist_ids[mine] : -1;
        uint32_t p16 = probs ? probs[mine] : 0u;
        int32_t row[TOPK];
        if (idx) {
            d = row_of(d);
            const int32_t r = d >= 0 && (int64_t)d < permuted_rows ? d : 0;
#pragma unroll
            for (int s = 0; s < TOPK; ++s) row[s] = __builtin_amdgcn_readlane(r, s);
        } else {
#pragma unroll
            for (int s = 0; s < TOPK; ++s) row[s] = t * TOPK + s < permuted_rows ? (int32_t)(t * TOPK + s) : 0;
        }
        // Whole wavefronts go round: lane s holds slot s, also where the row ends in front of that lane.
        for (int64_t at = first; at - lane < nv; at += step) {
            const int64_t i = at < nv ? at : nv - 1;
            v8u16 v[TOPK];
            if (permuted_rows > 0) {
#pragma unroll
                for (int s = 0; s < TOPK; ++s) v[s] = __builtin_nontemporal_load((const v8u16*)(permuted + (int64_t)row[s] * H) + i);
            }
            const v8u16 r = load_residual(i);
            asm volatile("" : "+v"(d), "+v"(e), "+v"(p16));  // used from here on: what is made of them stays behind the rows' loads
            // pair order: a pair whose expert id is out of range was computed by nobody
            const unsigned long long use = __ballot(d >= 0 && (int64_t)d < permuted_rows && (idx || !hist_ids || (e >= 0 && e < hist_experts)));
            const float w_lane = probs ? half_to_f32<DT>((uint16_t)p16) : 1.0f;
            float acc[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] = 0.0f;
#pragma unroll
            for (int s = 0; s < TOPK; ++s) {
                if (!((use >> s) & 1)) continue;
                const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w_lane), s));
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    float pr = w * half_to_f32<DT>(v[s][j]);
                    acc[j] = acc[j] + pr;
                }
            }
            if (at < nv) finish(i, acc, r);
        }
    } else {
        __shared__ int32_t srow[64];
        __shared__ float sw[64];
        const int top_k = a.top_k;
        if (threadIdx.x < top_k) {
            int32_t d = idx ? idx[t * top_k + threadIdx.x] : (int32_t)(t * top_k + threadIdx.x);
            d = row_of(d);
            if (!idx && hist_ids) {
                const int32_t e = hist_ids[t * top_k + threadIdx.x];
                if (e < 0 || e >= hist_experts) d = 0x7fffffff;
            }
            srow[threadIdx.x] = ((int64_t)d < permuted_rows) ? d : -1;
            sw[threadIdx.x] = probs ? half_to_f32<DT>(probs[t * top_k + threadIdx.x]) : 1.0f;
        }
        __syncthreads();
        for (int64_t i = first; i < nv; i += step) {
            float acc[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] = 0.0f;
            for (int s = 0; s < top_k; ++s) {
                const int32_t d = srow[s];
                if (d < 0) continue;
                const float w = sw[s];
                const v8u16 v = ((const v8u16*)(permuted + (int64_t)d * H))[i];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    float pr = w * half_to_f32<DT>(v[j]);
                    acc[j] = acc[j] + pr;
                }
            }
            finish(i, acc, load_residual(i));
        }
    }
}

}  // namespace moe355

using namespace moe355;

int moe355::unpermute_impl(const void* permuted, int dtype, const int32_t* sorted_indices, const void* probs,
                           int64_t num_tokens, int top_k, int64_t hidden, int64_t permuted_rows, const void* residual,
                           void* out, const int32_t* hist_ids, int hist_experts, int64_t* hist_out,
                           const int64_t* load_counts, int64_t* load, void* stream)
{
    if (num_tokens < 0 || top_k <= 0 || hidden <= 0 || permuted_rows < 0) return MOE355_E_ARG;
    if (dtype != MOE355_DT_BF16 && dtype != MOE355_DT_F16) return MOE355_E_UNSUPPORTED;
    if (top_k > 64 || hidden % 8 != 0 || num_tokens > 0x7ffffffeLL) return MOE355_E_SHAPE;
    if (num_tokens == 0) return MOE355_OK;
    if (!permuted || (!sorted_indices && !hist_ids) || !out) return MOE355_E_ARG;
    if (((uintptr_t)permuted & 15) || ((uintptr_t)out & 15) || ((uintptr_t)residual & 15)) return MOE355_E_SHAPE;
    // one workgroup per token when the tokens alone fill the chip; otherwise the rows are cut into pieces of 256
    // 16-byte vectors until there are about 1024 workgroups
    unsigned pieces = 1;
    if (num_tokens < 512) {
        const int64_t per_row = (hidden / 8 + 255) / 256;
        const int64_t want = (1024 + num_tokens - 1) / num_tokens;
        pieces = (unsigned)(per_row < want ? per_row : want);
        if (pieces < 1) pieces = 1;
    }
    const UnpermuteArgs a = {(int)num_tokens, top_k, (int)pieces, hist_experts, (const uint16_t*)permuted, sorted_indices,
                             (const uint16_t*)probs, (const uint16_t*)residual, (uint16_t*)out, hist_ids, hidden, permuted_rows,
                             hist_out, load_counts, load};
    const dim3 grid((unsigned)num_tokens + (hist_out || load ? 1u : 0u), pieces);
#define MOE355_UNPERMUTE(K, D) hipLaunchKernelGGL((token_unpermute_kernel<K, D>), grid, dim3(256), 0, (hipStream_t)stream, a)
    if (dtype == MOE355_DT_F16) {
        // fp16 models: the common fan-outs unrolled, the rest through the generic loop
        if (top_k == 8) MOE355_UNPERMUTE(8, MOE355_DT_F16);
        else if (top_k == 2) MOE355_UNPERMUTE(2, MOE355_DT_F16);
        else MOE355_UNPERMUTE(0, MOE355_DT_F16);
        return launch_status();
    }
    switch (top_k) {
        case 1: MOE355_UNPERMUTE(1, MOE355_DT_BF16); break;
        case 2: MOE355_UNPERMUTE(2, MOE355_DT_BF16); break;
        case 4: MOE355_UNPERMUTE(4, MOE355_DT_BF16); break;
        case 6: MOE355_UNPERMUTE(6, MOE355_DT_BF16); break;
        case 8: MOE355_UNPERMUTE(8, MOE355_DT_BF16); break;
        default: MOE355_UNPERMUTE(0, MOE355_DT_BF16); break;
    }
#undef MOE355_UNPERMUTE
    return launch_status();
}

extern "C" int moe355_token_unpermute(const void* permuted, int dtype, const int32_t* sorted_indices,
                                      const void* probs, int64_t num_tokens, int top_k, int64_t hidden,
                                      int64_t permuted_rows, const void* residual, void* out, void* stream)
{
    if (num_tokens > 0 && !sorted_indices) return MOE355_E_ARG;
    return unpermute_impl(permuted, dtype, sorted_indices, probs, num_tokens, top_k, hidden, permuted_rows, residual, out,
                          nullptr, 0, nullptr, nullptr, nullptr, stream);
}

extern "C" int moe355_token_unpermute_pairs(const void* rows, int dtype, const void* probs, const int32_t* topk_ids,
                                            int64_t num_tokens, int top_k, int64_t hidden, int num_experts,
                                            const void* residual, void* out, int64_t* expert_tokens, void* stream)
{
    if (num_experts <= 0) return MOE355_E_ARG;
    if (num_experts > kHistMaxExperts) return MOE355_E_SHAPE;
    if (num_tokens > 0 && (!topk_ids || !expert_tokens)) return MOE355_E_ARG;
    return unpermute_impl(rows, dtype, nullptr, probs, num_tokens, top_k, hidden, num_tokens * top_k, residual, out,
                          topk_ids, num_experts, expert_tokens, nullptr, nullptr, stream);
}

extern "C" int moe355_abi_version(void) { return MOE355_ABI_VERSION; }

extern "C" const char* moe355_strerror(int code)
{
    switch (code) {
        case MOE355_OK: return "ok";
        case MOE355_E_ARG: return "invalid argument (null pointer, negative size or unknown enum value)";
        case MOE355_E_SHAPE: return "shape or alignment outside what the kernels support";
        case MOE355_E_WORKSPACE: return "workspace missing, misaligned or too small";
        case MOE355_E_LAUNCH: return "the HIP runtime refused the kernel launch";
        case MOE355_E_UNSUPPORTED: return "option not supported by this build";
        default: return "unknown error code";
    }
}
