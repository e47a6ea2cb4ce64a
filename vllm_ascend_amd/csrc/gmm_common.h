// Pieces shared by the grouped-GEMM kernels: tiled weight addressing, the
// MFMA accumulator <-> (row, channel) mapping and the three epilogues.
//
// MFMA of the streaming kernel: v_mfma_i32_32x32x32_i8 (the tiles of many rows use mfma_i8_16 below).
// Operand A (4 VGPRs = 16 int8 per lane) carries WEIGHTS: lane l supplies channel l%32, K slice 16*(l/32)..+15 of the
// 32-wide K step.  Operand B carries TOKENS with the same K mapping.  The
// 32x32 int32 result sits in 16 VGPRs: lane l, register v holds
//   token   = l % 32
//   channel = 8*(v/4) + 4*(l/32) + v%4
// so every lane owns one token and four runs of four consecutive channels.
#pragma once

#include "moe355_common.h"

namespace moe355 {

enum { EPI_I32 = 0, EPI_SWIGLU = 1, EPI_DEQUANT = 2, EPI_MEET = 3, EPI_MEET_SHARED = 4 };

// EPI_MEET: SwiGLU and the rows' quantisation; the workgroups of a tile exchange the maxima of its rows (gmm_tiled.hip)
// EPI_MEET_SHARED: the same with the shared expert's arithmetic (dequant_swiglu_quant_kernel, form_b): the channel's scale before the
// row's, scale = maximum * (1 / 127), values divided by it
constexpr bool meets(int epi) { return epi == EPI_MEET || epi == EPI_MEET_SHARED; }
constexpr bool gated(int epi) { return epi == EPI_SWIGLU || meets(epi); }

struct GmmArgs {
    const int8_t* x;        // [R, K]
    const int8_t* w;        // tiled [E][N/32][K/32][1024]
    const int64_t* gl;      // [E]
    int gl_type;
    int64_t R;
    int K, N, E;
    const float* row_scale; // [R]     token scale
    // when set: row r of the expert-sorted activation is row row_src[r] of x, and its scale is
    // row_scale[row_src[r]] (the rows were quantised once, in token order, and never copied)
    const int32_t* row_src;
    const float* ch_scale;  // [E, N]  channel scale
    // per-expert tensors (weights that can be swapped expert by expert): device arrays of E pointers;
    // when set they replace w / ch_scale
    const int8_t* const* w_list;
    const float* const* s_list;
    // Pair order (small batches, streaming kernel only): no group list and no sorted copy.  pair_ids[f] is the
    // expert of pair f = token * pair_k + slot; R pairs.  Every workgroup collects the pairs of its expert itself;
    // row i of the expert is pair f: its values lie in row f / pair_k of x (pair_gather: x and row_scale in token
    // order) or in row f, and its result goes to row f.
    const int32_t* pair_ids;
    int pair_k, pair_gather;
    // The grid has a place for each of the experts [0, pair_first), and pair_slots places behind them: slot s works on
    // the s-th of the other experts that have pairs (the idle ones cost nothing).  pair_extra > 0: those work on the
    // first 32 rows of their expert, and as many more places on further blocks of 32 rows: pair_early of them in front of
    // the slots, the others at the end of the grid.
    int pair_first, pair_slots, pair_extra, pair_early;
    // Pair order with the shared expert in the same launch: sh_blocks places in front of the others, place b on rows
    // 32 b .. of the sh_rows tokens.  Token t's values lie in row t (pair_gather) or R + t of x, its result goes to row
    // R + t.  Its weights have the shape of a routed expert's.
    int sh_blocks, sh_rows;
    const int8_t* sh_w;
    const float* sh_scale;
    float sh_limit;
    // the same for a sorted activation with fewer rows than experts: place s works on the s-th expert whose group
    // is not empty
    int gl_slots;
    // pair order, down GEMM with the re-quantisation inside (REQ): the SwiGLU values [R, K] fp32 that the gate_up
    // GEMM wrote; the workgroup quantises the rows of its expert itself (x and row_scale are not read)
    const float* y_in;
    int beside;             // dense product on a side stream: few workgroups that hide, not many that finish early
    float limit;            // swiglu clamp
    int tiles_ready;        // the tile maps of this call are in its workspace already (built by the routing launch)
    // EPI_MEET: [columns][R] the maximum of a row over a column block, its bits with the sign set; zero before the launch
    uint32_t* meet;
    int meet_looks;         // at the others' maxima before a workgroup computes them itself
    int8_t* q;              // [R, N/2]
    float* q_scale;         // [R]
    // outputs
    int32_t* acc;           // EPI_I32   [R, N]
    int32_t* acc_part;      // EPI_I32 with K cut into slabs: [slabs][R, N] partial sums (or null: atomics into acc)
    float* y;               // EPI_SWIGLU [R, N/2] fp32 SwiGLU values
    uint16_t* out;          // EPI_DEQUANT [R, N] bf16, or fp16 when out_f16 is set
    int out_f16;
};

// tiled weights / channel scales of expert e
__device__ __forceinline__ const int8_t* expert_weights(const GmmArgs& a, int e)
{
    return a.w_list ? a.w_list[e] : a.w + (int64_t)e * a.N * a.K;
}
__device__ __forceinline__ const float* expert_scales(const GmmArgs& a, int e)
{
    return a.s_list ? a.s_list[e] : a.ch_scale + (int64_t)e * a.N;
}

// Loads through pointers that may come out of a per-expert pointer table.  The compiler cannot prove that
// such a pointer is global memory and would emit FLAT loads, which count against the LDS counter as well:
// every s_waitcnt after them becomes a full drain (vmcnt(0) lgkmcnt(0)) and the software pipeline of the
// GEMM kernels collapses to one batch in flight.  Saying "global" keeps the waits partial.
typedef const v4i __attribute__((address_space(1))) * gv4i_ptr;
typedef const v4f __attribute__((address_space(1))) * gv4f_ptr;
__device__ __forceinline__ v4i gload16(const void* p) { return *(gv4i_ptr)(uintptr_t)p; }
__device__ __forceinline__ v4i gload16_nt(const void* p) { return __builtin_nontemporal_load((gv4i_ptr)(uintptr_t)p); }
__device__ __forceinline__ v4f gload4f(const float* p) { return *(gv4f_ptr)(uintptr_t)p; }

// 16 bytes written through the L2, for the outputs of the large products.  A read stream of weights with 128-byte row pieces
// written beside it, non-temporal / plain / written through, us: 1611 + 75 MB 292 / 296 / 282, 805 + 101 MB 156 / 155 / 148, 201 +
// 25 MB 37.7 / 39.1 / 34.7, 1611 + 200 MB 324 / 316 / 304 (sc0 sc1 as sc1; with nt beside either as non-temporal; pieces of 128
// bytes to 1 KiB the same).  The down products 2 to 5 % faster than with non-temporal stores.
__device__ __forceinline__ void store16_through(void* p, v4i v)
{
    // (behind a store of 16 bytes the next two wait states may not write its data)
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}

__device__ __forceinline__ v16i mfma_i8(v4i a, v4i b, v16i c)
{
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
}

// v_mfma_i32_16x16x64_i8: A = 16 channels x 64 K (lane l: channel l%16, K slice 16*(l/16)..+15),
// B = 16 tokens x 64 K with the same K mapping; result 4 VGPRs: token l%16, channels 4*(l/16)+0..3.
__device__ __forceinline__ v4i mfma_i8_16(v4i a, v4i b, v4i c)
{
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}

// Weights of 16 channels x 64 K values for it, out of the storage tiles (32 channels x 32 K in 1 KiB: lane l of that tile
// holds channel l % 32, K half l / 32): this lane's byte offset inside the 2 KiB of 64 K values; the second 16 channels
// lie 256 bytes further.
__device__ __forceinline__ int weight_lane(int lane) { return (lane >> 4) * 512 + (lane & 15) * 16; }

// One token row, one run of four consecutive channels starting at c0 (tile 0) and c1 (tile 1).
// rs: the row's token scale; s0 / s1: the channel scales of the two runs.  The caller loads them before its
// K loop: a load issued here, behind the stores of an earlier run, would wait for those stores (the memory
// counter retires in order), one store round trip per run.
// shared (SwiGLU only): the shared expert's operator multiplies by the channel scale first, then by the token scale.
template <int EPI>
__device__ __forceinline__ void epilogue_run(const GmmArgs& a, int64_t row, bool valid, int c0, int c1, const int* g,
                                             const int* u, float rs, v4f s0, v4f s1, bool shared = false)
{
    if (!valid) return;
    if constexpr (EPI == EPI_I32) {
        v4i o0 = {g[0], g[1], g[2], g[3]};
        v4i o1 = {u[0], u[1], u[2], u[3]};
        *(v4i*)(a.acc + row * a.N + c0) = o0;
        *(v4i*)(a.acc + row * a.N + c1) = o1;
    } else if constexpr (EPI == EPI_DEQUANT) {
        v4u16 o0, o1;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float v0 = ((float)g[j] * rs) * s0[j], v1 = ((float)u[j] * rs) * s1[j];
            o0[j] = a.out_f16 ? f32_to_f16(v0) : f32_to_bf16(v0);
            o1[j] = a.out_f16 ? f32_to_f16(v1) : f32_to_bf16(v1);
        }
        *(v4u16*)(a.out + row * a.N + c0) = o0;
        *(v4u16*)(a.out + row * a.N + c1) = o1;
    } else {
        // tile 0 = gate, tile 1 = the matching up tile (c1 = c0 + N/2)
        const int I = a.N >> 1;
        const float limit = shared ? a.sh_limit : a.limit;
        v4f yv;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float gg = ((float)g[j] * (shared ? s0[j] : rs)) * (shared ? rs : s0[j]);
            float uu = ((float)u[j] * (shared ? s1[j] : rs)) * (shared ? rs : s1[j]);
            if (limit > 0.0f) {
                gg = gg > limit ? limit : gg;
                uu = uu > limit ? limit : uu;
                uu = uu < -limit ? -limit : uu;
            }
            yv[j] = m_silu(gg) * uu;
        }
        *(v4f*)(a.y + row * I + c0) = yv;
    }
}

// First channel, inside a 32-channel tile, of the run that quarter q of a 32x32 accumulator tile holds in
// this lane: 8*q + 4*(lane/32), four consecutive channels.
__device__ __forceinline__ int quad_channel(int q, int lane) { return 8 * q + 4 * (lane >> 5); }

// Measurement hook (gmm.hip): hands out, once, the events that moe355_profile_next_gemm armed on this thread
// (both null when nothing is armed); the caller records them around exactly one kernel launch.
void take_profile_events(hipEvent_t& start, hipEvent_t& stop);

// SwiGLU values y fp32 [R, I] -> per-row absmax -> int8 + scale (defined in gmm.hip).
// Rows from shared_from on are the shared expert's: its operator's quantiser (scale = max * float(1/127), q = rint(v /
// scale)) instead of the routed experts'.
void launch_swiglu_requant(const float* y, const int64_t* gl, int gl_type, int E, int64_t R, int I, int8_t* q,
                           float* qs, hipStream_t st, int64_t shared_from = INT64_MAX);

}  // namespace moe355
