// Group-limited top-k gating of one token row by one wavefront (shared by the gating kernel and the fused
// small-batch routing kernel).
//
// Lane l holds experts l, l+64, l+128, ... (PER of them) in registers, so the
// logits row is read with coalesced loads and the softmax sum follows the
// contract order: strided per-lane partials, then a butterfly.  Group scores
// go through a per-wavefront LDS copy of the selection scores (a group's
// experts are spread over lanes).  The order is always "larger value, then lower
// index".  Groups: repeated arg-max reductions in gate_row, a count of the groups
// in front of each in row_scores.  Experts: repeated arg-max reductions, or ranks
// counted by several wavefronts (rank_row) where a launch waits for one row.
#pragma once

#include "layer_parts.h"
#include "moe355_common.h"

namespace moe355 {

// DPP step: combine every lane with the lane `ctrl` names (row shift / row broadcast).  Lanes
// without a source keep their own value, which is harmless for max.
#define MOE355_DPP(v, ctrl, rmask) __builtin_amdgcn_update_dpp((int)(v), (int)(v), ctrl, rmask, 0xf, false)

// Maximum of an unsigned value over the wavefront; every lane returns it.  Six DPP steps, each one v_max_u32 that
// reads its first operand through the lane permutation (the compiler keeps the permutation and the maximum apart:
// copy, v_mov_dpp, compare, select).  A lane without a source in a step (shifted in from outside its row, or a row
// outside the row mask) is left as it is.  The s_nop in front of every step is the wait that a DPP read of a
// register needs after a vector instruction has written it.
__device__ __forceinline__ unsigned wave_max_u32(unsigned v)
{
    asm volatile(
        "s_nop 1\n\tv_max_u32_dpp %0, %0, %0 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\tv_max_u32_dpp %0, %0, %0 row_shr:2 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\tv_max_u32_dpp %0, %0, %0 row_shr:4 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\tv_max_u32_dpp %0, %0, %0 row_shr:8 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\tv_max_u32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
        "s_nop 1\n\tv_max_u32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
        "s_nop 1"
        : "+v"(v));
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// Maximum of a 64-bit key over the wavefront; every lane returns it: the largest high word, and the largest low
// word among the lanes that hold it.  One lane that holds it alone (scores rarely tie) is read instead.
__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long v)
{
    const unsigned hi = (unsigned)(v >> 32);
    const unsigned m = wave_max_u32(hi);
    const unsigned long long holders = __ballot(hi == m);
    unsigned lo;
    if ((holders & (holders - 1)) == 0ull) lo = (unsigned)__builtin_amdgcn_readlane((int)v, __builtin_ctzll(holders));
    else lo = wave_max_u32(hi == m ? (unsigned)v : 0u);
    return ((unsigned long long)m << 32) | lo;
}

__device__ __forceinline__ float wave_max_dpp(float v)
{
#define MOE355_STEP(ctrl, rmask)                                                 \
    {                                                                            \
        float o = __int_as_float(MOE355_DPP(__float_as_int(v), ctrl, rmask));    \
        v = o > v ? o : v;                                                       \
    }
    MOE355_STEP(0x111, 0xf)
    MOE355_STEP(0x112, 0xf)
    MOE355_STEP(0x114, 0xf)
    MOE355_STEP(0x118, 0xf)
    MOE355_STEP(0x142, 0xa)
    MOE355_STEP(0x143, 0xc)
#undef MOE355_STEP
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// Selection key: larger score first, ties to the lower index.  The float is mapped to an
// unsigned integer with the same order (-0 is folded into +0 first, so equal scores compare
// equal), the index is stored inverted in the low word.  0 never occurs as a key of a real
// candidate and stands for "none".
__device__ __forceinline__ unsigned long long make_key(float score, int index)
{
    score = score + 0.0f;
    unsigned u = __float_as_uint(score);
    u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    return ((unsigned long long)u << 32) | (unsigned)(0xffffffffu - (unsigned)index);
}

__device__ __forceinline__ int key_index(unsigned long long key) { return (int)(0xffffffffu - (unsigned)key); }

// Score of one expert group from its gs selection scores: the best one (mode 0) or the sum of the best two, best
// first ("larger value, then lower index").  One pass that keeps the two leaders.
__device__ __forceinline__ float group_score(const float* s, int gs, int mode)
{
    int i1 = 0, i2 = -1;
    float v1 = s[0], v2 = 0.0f;
    for (int j = 1; j < gs; ++j) {
        const float v = s[j];
        if (ranks_before(v, j, v1, i1)) {
            v2 = v1;
            i2 = i1;
            v1 = v;
            i1 = j;
        } else if (i2 < 0 || ranks_before(v, j, v2, i2)) {
            v2 = v;
            i2 = j;
        }
    }
    return (mode != 0 && gs >= 2) ? v1 + v2 : v1;
}

// The scores of all groups of one row at once, for groups of a power of two of at most 64 experts: such a group is
// a run of gs lanes in one of the row's registers (expert e = lane + 64 i), so a butterfly over the lanes of the
// run leaves the group's two largest selection scores in every one of them.  The same two values as the pass of
// group_score (a tie is two equal values either way; the order of a +0 and a -0 does not change their sum), the
// same sum; a row that holds a NaN takes group_score instead, whose treatment of it depends on the position.
// Lane g (< G) returns the score of group g, the other lanes anything.
// The exchanges are register permutations (a step of lane reads through LDS is a chain of some 150 cycles): behind the
// steps of 1 and 2 the lanes of a quad agree, so a mirrored half row or row names a lane of the partner as well as lane
// ^ 4 or ^ 8.  With the divisions of row_scores by shifts, the routing launch of 256 experts in 8 groups and rows of
// 7168 values, 1 / 64 / 512 / 4096 tokens 4.93 / 5.96 / 6.42 / 19.95 -> 4.76 / 5.35 / 5.85 / 18.93 us.
template <int PER>
__device__ __forceinline__ float group_scores_butterfly(const float (&sel)[PER], int gs, int mode, int lane)
{
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    float t1[PER], t2[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        t1[i] = sel[i];
        t2[i] = -__builtin_inff();
    }
    auto merge = [&](int i, float a1, float a2, float b1, float b2) {
        const bool gt = a1 > b1;
        const float lo = gt ? b1 : a1;
        const float second = a2 > b2 ? a2 : b2;
        t1[i] = gt ? a1 : b1;
        t2[i] = lo > second ? lo : second;
    };
#define MOE355_STEP(ctrl)                                                                      \
    _Pragma("unroll") for (int i = 0; i < PER; ++i)                                            \
        merge(i, t1[i], t2[i], __int_as_float(MOE355_DPP(__float_as_int(t1[i]), ctrl, 0xf)),   \
              __int_as_float(MOE355_DPP(__float_as_int(t2[i]), ctrl, 0xf)))
#define MOE355_SWAP(swap)                                                                                    \
    _Pragma("unroll") for (int i = 0; i < PER; ++i)                                                          \
    {                                                                                                        \
        const v2u a = swap(__float_as_uint(t1[i]), __float_as_uint(t1[i]), false, false);                    \
        const v2u b = swap(__float_as_uint(t2[i]), __float_as_uint(t2[i]), false, false);                    \
        merge(i, __uint_as_float(a[0]), __uint_as_float(b[0]), __uint_as_float(a[1]), __uint_as_float(b[1])); \
    }
    if (gs > 1) MOE355_STEP(0xb1);  // quad_perm 1 0 3 2
    if (gs > 2) MOE355_STEP(0x4e);  // quad_perm 2 3 0 1
    if (gs > 4) MOE355_STEP(0x141);  // row_half_mirror
    if (gs > 8) MOE355_STEP(0x140);  // row_mirror
    if (gs > 16) MOE355_SWAP(__builtin_amdgcn_permlane16_swap)
    if (gs > 32) MOE355_SWAP(__builtin_amdgcn_permlane32_swap)
#undef MOE355_SWAP
#undef MOE355_STEP
    const int shift = __builtin_ctz(gs), runs = 64 >> shift;  // groups per register
    const int src = (lane & (runs - 1)) << shift;
    float out = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const float sc = (mode != 0 && gs >= 2) ? t1[i] + t2[i] : t1[i];
        const float v = __shfl(sc, src);
        if (lane >> (6 - shift) == i) out = v;
    }
    return out;
}

template <int PER>
__device__ __forceinline__ bool butterfly_groups(const float (&sel)[PER], int gs)
{
    if (gs > 64 || (gs & (gs - 1)) != 0) return false;
    bool nan = false;
#pragma unroll
    for (int i = 0; i < PER; ++i) nan = nan || (sel[i] != sel[i]);
    return __ballot(nan) == 0ull;
}

// One token row by one wavefront.  Every wavefront of the workgroup calls this the same number of times (it
// contains workgroup barriers); a call with live == false computes a valid row and stores nothing.
// sc_lds: E floats, w_lds: 64 floats, both private to the wavefront.  y may be null (only y_alt wanted);
// idx_lds (LDS, may be null) receives the k chosen experts as well.
template <int DT, int PER>
__device__ __forceinline__ void gate_row(const void* __restrict__ x, const void* __restrict__ bias, int64_t row,
                                         bool live, int E, int k, int k_group, int G, int mode, int renorm,
                                         int norm_type, float rsf, float eps, void* __restrict__ y,
                                         int32_t* __restrict__ idx, float* __restrict__ out, int out_flag,
                                         void* __restrict__ y_alt, int y_alt_dtype, float* sc_lds, float* w_lds,
                                         int32_t* idx_lds, int lane)
{
    float p[PER];
    float sel[PER];
    // ---- normalise
    float m = -__builtin_inff();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        int e = lane + 64 * i;
        p[i] = (e < E) ? load_as_f32<DT>(x, row * E + e) : -__builtin_inff();
        m = p[i] > m ? p[i] : m;
    }
    if (norm_type == 0) {
        m = wave_max_dpp(m);
        float part = 0.0f;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            int e = lane + 64 * i;
            if (e < E) {
                p[i] = m_expf(p[i] - m);
                part = part + p[i];
            }
        }
        float s = wave_tree_sum(part);
        float inv = 1.0f / s;
#pragma unroll
        for (int i = 0; i < PER; ++i) p[i] = p[i] * inv;
    } else {
#pragma unroll
        for (int i = 0; i < PER; ++i) p[i] = 1.0f / (1.0f + m_expf(-p[i]));
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        int e = lane + 64 * i;
        if (e < E) {
            if (out_flag && live) out[row * E + e] = p[i];
            sel[i] = bias ? p[i] + load_as_f32<DT>(bias, e) : p[i];
        } else {
            sel[i] = -__builtin_inff();
        }
    }

    // ---- group limit
    if (G > 1) {
        const int gs = E / G;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            int e = lane + 64 * i;
            if (e < E) sc_lds[e] = sel[i];
        }
        __syncthreads();
        unsigned long long gkey = 0ull;
        if (butterfly_groups<PER>(sel, gs)) {
            const float sc = group_scores_butterfly<PER>(sel, gs, mode, lane);
            if (lane < G) gkey = make_key(sc, lane);
        } else if (lane < G) {
            const float* s = sc_lds + lane * gs;
            gkey = make_key(group_score(s, gs, mode), lane);
        }
        unsigned long long keep = 0ull;
        for (int c = 0; c < k_group; ++c) {
            const int g = key_index(wave_max_u64(gkey));
            keep |= 1ull << g;
            if (lane == g) gkey = 0ull;
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            int e = lane + 64 * i;
            if (e < E && !((keep >> (e / gs)) & 1ull)) sel[i] = -__builtin_inff();
        }
        __syncthreads();
    }

    // ---- top-k over the (masked) selection scores; the unbiased scores wait in LDS
    unsigned long long key[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        int e = lane + 64 * i;
        key[i] = (e < E) ? make_key(sel[i], e) : 0ull;
        if (e < E) sc_lds[e] = p[i];
    }
    int my_i = 0;
    for (int c = 0; c < k; ++c) {
        unsigned long long best = 0ull;
#pragma unroll
        for (int i = 0; i < PER; ++i) best = key[i] > best ? key[i] : best;
        const int win = key_index(wave_max_u64(best));
        if ((win & 63) == lane) {
#pragma unroll
            for (int i = 0; i < PER; ++i)
                if (i == (win >> 6)) key[i] = 0ull;
        }
        if (lane == c) my_i = win;
    }
    __syncthreads();
    float my_p = (lane < k) ? sc_lds[my_i] : 0.0f;
    if (norm_type == 1 || renorm == 1) {
        if (lane < k) w_lds[lane] = my_p;
        __syncthreads();
        float wsum = 0.0f;
        for (int c = 0; c < k; ++c) wsum = wsum + w_lds[c];
        float d = wsum + eps;
        my_p = my_p / d;
    }
    my_p = my_p * rsf;
    if (idx_lds && lane < k) idx_lds[lane] = my_i;
    if (live && lane < k) {
        if (y) store_from_f32<DT>(y, row * k + lane, my_p);
        idx[row * k + lane] = my_i;
        if (y_alt) {
            // second copy of the weights in another dtype: the value stored in y, narrowed again
            float stored = my_p;
            if constexpr (DT == MOE355_DT_BF16) stored = bf16_to_f32(f32_to_bf16(my_p));
            if constexpr (DT == MOE355_DT_F16) stored = f16_to_f32(f32_to_f16(my_p));
            if (y_alt_dtype == MOE355_DT_BF16) ((uint16_t*)y_alt)[row * k + lane] = f32_to_bf16(stored);
            else if (y_alt_dtype == MOE355_DT_F16) ((uint16_t*)y_alt)[row * k + lane] = f32_to_f16(stored);
            else ((float*)y_alt)[row * k + lane] = stored;
        }
    }
}

// The order of a selection score as an unsigned integer (the high word of make_key).
__device__ __forceinline__ unsigned score_order(float score) { return (unsigned)(make_key(score, 0) >> 32); }

// A row's logits as fp32: read from [T, E], or (fp32 only) added up from the router gate's chunk results, at most
// kGatePlanes planes of T x E, in ascending order from +0 and the bias last, which is what its own reduction does.
template <int DT>
struct RowLogits {
    const void* logits;
    int64_t at, plane;  // first value of the row; values of a plane
    int n_planes;
    const float* bias;
    // lane l: the logits of experts l, l + 64, ... (-inf past the last one)
    template <int PER>
    __device__ __forceinline__ void load(float (&p)[PER], int E, int lane) const
    {
        if constexpr (DT == MOE355_DT_F32) {
            if (n_planes > 0) {
                const float* from = (const float*)logits + at + lane;
                float v[kGatePlanes][PER], sum[PER];
#pragma unroll
                for (int c = 0; c < kGatePlanes; ++c)
#pragma unroll
                    for (int i = 0; i < PER; ++i)
                        v[c][i] = c < n_planes && lane + 64 * i < E ? from[c * plane + 64 * i] : 0.0f;
#pragma unroll
                for (int i = 0; i < PER; ++i) sum[i] = 0.0f;
#pragma unroll
                for (int c = 0; c < kGatePlanes; ++c)
#pragma unroll
                    for (int i = 0; i < PER; ++i)
                        if (c < n_planes) sum[i] = sum[i] + v[c][i];
#pragma unroll
                for (int i = 0; i < PER; ++i) {
                    const int e = lane + 64 * i;
                    p[i] = e >= E ? -__builtin_inff() : bias ? sum[i] + bias[e] : sum[i];
                }
                return;
            }
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = lane + 64 * i;
            p[i] = e < E ? load_as_f32<DT>(logits, at + e) : -__builtin_inff();
        }
    }
};

// The scores of one token row by one wavefront, the arithmetic of gate_row without a workgroup barrier: p, the values the
// weights come from, and sel, what the experts are chosen by (groups that are not kept at -inf).  What the row needs from
// other lanes travels by lane reads, the group scores through grp_lds (E floats private to the wavefront; only touched
// when G > 1).
template <int DT, int PER>
__device__ __forceinline__ void row_scores(const RowLogits<DT>& logits, const void* __restrict__ bias, int E, int k_group, int G, int mode,
                                           int norm_type, float* grp_lds, int lane, float (&p)[PER], float (&sel)[PER])
{
    float m = -__builtin_inff();
    logits.load(p, E, lane);
#pragma unroll
    for (int i = 0; i < PER; ++i) m = p[i] > m ? p[i] : m;
    if (norm_type == 0) {
        m = wave_max_dpp(m);
        float part = 0.0f;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (lane + 64 * i < E) {
                p[i] = m_expf(p[i] - m);
                part = part + p[i];
            }
        }
        const float inv = 1.0f / wave_tree_sum(part);
#pragma unroll
        for (int i = 0; i < PER; ++i) p[i] = p[i] * inv;
    } else {
#pragma unroll
        for (int i = 0; i < PER; ++i) p[i] = 1.0f / (1.0f + m_expf(-p[i]));
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = lane + 64 * i;
        if (e < E) sel[i] = bias ? p[i] + load_as_f32<DT>(bias, e) : p[i];
        else sel[i] = -__builtin_inff();
    }
    if (G > 1) {
        // a division by a number of the call is some 150 cycles
        const bool powers = (G & (G - 1)) == 0 && (E & (E - 1)) == 0;
        const int gs = powers ? E >> __builtin_ctz(G) : E / G;
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (lane + 64 * i < E) grp_lds[lane + 64 * i] = sel[i];
        wave_lds_order();
        unsigned gu = 0u;
        if (butterfly_groups<PER>(sel, gs)) gu = score_order(group_scores_butterfly<PER>(sel, gs, mode, lane));
        else if (lane < G) gu = score_order(group_score(grp_lds + lane * gs, gs, mode));
        // a group stays if fewer than k_group others come before it
        int before = 0;
        for (int g = 0; g < G; ++g) {
            const unsigned v = (unsigned)__builtin_amdgcn_readlane((int)gu, g);
            before += (v > gu || (v == gu && g < lane)) ? 1 : 0;
        }
        const unsigned long long keep = __ballot(lane < G && before < k_group);
        auto cut = [&](auto group_of) {
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int e = lane + 64 * i;
                if (e < E && !((keep >> group_of(e)) & 1ull)) sel[i] = -__builtin_inff();
            }
        };
        const int shift = __builtin_ctz(gs);
        if (powers) cut([&](int e) { return e >> shift; });
        else cut([&](int e) { return e / gs; });
    }
}

// The chosen experts of a row, in order, and their weights: lane c (< k) holds the c-th, my_p its unnormalised value.
// Weights are written to weights[o ..] in w_dtype after rounding to DT (the cast chain of the reference's caller: gate
// output in the logits dtype, then .to(hidden dtype)) and ids to idx[o ..].
template <int DT>
__device__ __forceinline__ void store_choice(int my_i, float my_p, int k, int renorm, int norm_type, float rsf, float eps,
                                             int64_t o, void* __restrict__ weights, int w_dtype,
                                             int32_t* __restrict__ idx, int lane)
{
    if (norm_type == 1 || renorm == 1) {
        float wsum = 0.0f;
        for (int c = 0; c < k; ++c) wsum = wsum + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_p), c));
        const float d = wsum + eps;
        my_p = my_p / d;
    }
    my_p = my_p * rsf;
    if (lane >= k) return;
    // a store that is visible to the whole device when it completes (a workgroup on another part of the chip may be the
    // one that sorts the pairs)
    __hip_atomic_store(idx + o + lane, my_i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    float stored = my_p;
    if constexpr (DT == MOE355_DT_BF16) stored = bf16_to_f32(f32_to_bf16(stored));
    if constexpr (DT == MOE355_DT_F16) stored = f16_to_f32(f32_to_f16(stored));
    if (w_dtype == MOE355_DT_BF16) ((uint16_t*)weights)[o + lane] = f32_to_bf16(stored);
    else if (w_dtype == MOE355_DT_F16) ((uint16_t*)weights)[o + lane] = f32_to_f16(stored);
    else ((float*)weights)[o + lane] = stored;
}

constexpr int kChooseFrom = 6;  // see choose_row

// The k first of a row's experts by one wavefront, without the chain of k maxima over the wavefront (about 430 cycles each):
// an expert can only be among them if fewer than k lanes hold a larger score than its own lane's largest, so every lane counts
// those lanes, and the experts of the few that are left (k PER of them, more where scores tie) are ranked by counting again.
// scratch: 192 floats private to the wavefront.  false where ties leave more than 64 experts.
// The routing launch of 1 / 64 / 512 / 4096 tokens, us with k rounds / so: 128 experts, k = 8, 3.37 / 4.23 / 4.36 /
// 7.43 against 2.84 / 3.46 / 3.58 / 7.19; 256 experts 4.13 / 4.72 / 4.89 / 8.58 against 3.58 / 4.06 / 4.21 / 8.02, in
// groups 5.76 / 6.55 / 7.08 / 23.06 against 5.16 / 5.99 / 6.40 / 23.07; 128 experts, k = 4, 2.59 / 3.36 / 3.49 / 6.58
// against 2.59 / 3.27 / 3.41 / 6.98, so from 6 on.
template <int PER>
__device__ __forceinline__ bool choose_row(const unsigned long long (&key)[PER], const float (&p)[PER], int k, float* scratch,
                                           int lane, int& my_i, float& my_p)
{
    unsigned* orders = (unsigned*)scratch;
    unsigned long long* keys = (unsigned long long*)scratch;
    float* values = scratch + 128;
    unsigned long long best = key[0];
#pragma unroll
    for (int i = 1; i < PER; ++i) best = key[i] > best ? key[i] : best;
    const unsigned mine = (unsigned)(best >> 32);
    wave_lds_order();
    orders[lane] = mine;
    wave_lds_order();
    int ahead[4] = {0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const uint4 v = ((const uint4*)orders)[j];
        ahead[0] += v.x > mine ? 1 : 0;
        ahead[1] += v.y > mine ? 1 : 0;
        ahead[2] += v.z > mine ? 1 : 0;
        ahead[3] += v.w > mine ? 1 : 0;
    }
    const bool in = ahead[0] + ahead[1] + ahead[2] + ahead[3] < k;
    const unsigned long long lanes = __ballot(in);
    const int n = __popcll(lanes) * PER;
    if (n > 64) return false;
    wave_lds_order();
    if (in) {
        const int slot = PER * __popcll(lanes & ((1ull << lane) - 1));
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            keys[slot + i] = key[i];
            values[slot + i] = p[i];
        }
    }
    wave_lds_order();
    const unsigned long long own = lane < n ? keys[lane] : 0ull;
    const float value = values[lane < n ? lane : 0];
    int rank = 0;
#pragma unroll 8
    for (int j = 0; j < n; ++j) rank += keys[j] > own ? 1 : 0;
    wave_lds_order();
    if (own != 0ull && rank < k) {
        orders[rank] = (unsigned)key_index(own);
        values[rank] = value;
    }
    wave_lds_order();
    if (lane < k) {
        my_i = (int)orders[lane];
        my_p = values[lane];
    }
    return true;
}

// One token row by one wavefront.  grp_lds: E floats and at least 192, 16-byte aligned.
template <int DT, int PER>
__device__ __forceinline__ void gate_row_wave(const RowLogits<DT>& logits, const void* __restrict__ bias, int E, int k, int k_group,
                                              int G, int mode, int renorm, int norm_type, float rsf, float eps,
                                              int64_t o, void* __restrict__ weights, int w_dtype,
                                              int32_t* __restrict__ idx, float* grp_lds, int lane)
{
    float p[PER], sel[PER];
    row_scores<DT, PER>(logits, bias, E, k_group, G, mode, norm_type, grp_lds, lane, p, sel);
    unsigned long long key[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) key[i] = (lane + 64 * i < E) ? make_key(sel[i], lane + 64 * i) : 0ull;
    int my_i = 0;
    float my_p = 0.0f;
    const bool chosen = k >= kChooseFrom && choose_row<PER>(key, p, k, grp_lds, lane, my_i, my_p);
    for (int c = chosen ? k : 0; c < k; ++c) {
        unsigned long long best = 0ull;
#pragma unroll
        for (int i = 0; i < PER; ++i) best = key[i] > best ? key[i] : best;
        const int win = key_index(wave_max_u64(best));
        float cand = 0.0f;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (i == (win >> 6)) {
                cand = p[i];
                if ((win & 63) == lane) key[i] = 0ull;
            }
        }
        const float pw = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cand), win & 63));
        if (lane == c) {
            my_i = win;
            my_p = pw;
        }
    }
    store_choice<DT>(my_i, my_p, k, renorm, norm_type, rsf, eps, o, weights, w_dtype, idx, lane);
}

// The ranks of one token row's experts by W wavefronts of a workgroup.  The k rounds of a maximum over the wavefront are a
// chain of about 430 cycles each: eight of them 1.5 us of one token's call, with everything else waiting (a bound for the
// k-th best by bisection of the bits takes as long).  Here one wavefront leaves the order of the scores in LDS, and every
// wavefront counts, for all experts, how many of its share of the experts come before them (larger score, then lower
// index); the counts add up to the ranks.  orders [E rounded up to 4]: score_order of every expert, at least 1; ranks [E]:
// zeroes.
template <int PER>
__device__ __forceinline__ void rank_row(const unsigned* orders, int E, int w, int W, int* ranks, int lane)
{
    unsigned u[PER];
    int count[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        u[i] = lane + 64 * i < E ? orders[lane + 64 * i] : 0xffffffffu;
        count[i] = 0;
    }
    const int quads = (E + 3) >> 2, q0 = quads * w / W, q1 = quads * (w + 1) / W;
    for (int qd = q0; qd < q1; ++qd) {
        const uint4 four = *(const uint4*)(orders + 4 * qd);
        const unsigned v[4] = {four.x, four.y, four.z, four.w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int from = 4 * qd + c;
            if (from >= E) break;
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                // at the same score the lower index comes first: v >= u there, which is v > u - 1 (no order is 0)
                count[i] += v[c] > u[i] - (from < lane + 64 * i ? 1u : 0u) ? 1 : 0;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < PER; ++i)
        if (lane + 64 * i < E) atomicAdd(ranks + lane + 64 * i, count[i]);
}

// the k first of the ranked experts into idx_lds (and their values into p_lds), in order
template <int PER>
__device__ __forceinline__ void place_row(const float (&p)[PER], const int* ranks, int E, int k, int* idx_lds, float* p_lds,
                                          int lane)
{
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = lane + 64 * i;
        const int r = e < E ? ranks[e] : k;
        if (r < k) {
            idx_lds[r] = e;
            p_lds[r] = p[i];
        }
    }
}

}  // namespace moe355
