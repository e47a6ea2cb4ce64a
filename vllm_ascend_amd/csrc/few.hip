// The expert MLPs of a few tokens (at most 64 (token, slot) pairs): what the first tokens of a decode
// batch cost is not the weight stream (38 MB of the Qwen3 shape are 5.5 us) but launches, each of them 3 to 6 us with
// its dispatch, its first look at the ids and its last store.  There are two here (three where the up kernel would repeat
// the gating too often, few_gates):
//
//   few_up_kernel    gate_up GEMM + SwiGLU of the routed experts AND of the shared expert, and the maxima of every row
//                    piece (atomics on one maximum per row meet at the memory side: 1536 of them cost 12 us);
//   few_down_kernel  re-quantisation, down GEMM and the weighted combine: a workgroup owns 16 (or 8) output channels of ALL
//                    pairs, so the k rows of a token meet in its LDS and leave as one finished row.
//
// From about 12 K SwiGLU values on every workgroup re-quantising all rows costs more than a launch (few_quant_kernel).
// The ids of at most 64 pairs are one load of one wavefront: every wavefront knows the distinct experts, its expert's
// rows and its share of the work from ballots, without LDS tables or barriers.  Tokens are the 16-column operand of
// v_mfma_i32_16x16x64_i8, so an accumulator is four registers and 8 wavefronts cutting K meet in 2 KB of LDS.
#include <hip/hip_ext.h>

#include <type_traits>

#include "gating_body.h"
#include "gmm_common.h"
#include "layer_parts.h"

namespace moe355 {

constexpr int kFewThreads = 512;
constexpr int kFewWaves = kFewThreads / 64;
constexpr int kFewItem = 8;            // K steps of 64 of an item of the down GEMM
constexpr int kFewInside = 12 * 1024;  // SwiGLU values that the workgroups of the down GEMM quantise themselves

struct FewExperts {
    int id;                     // this lane's pair's expert, or -1
    unsigned long long lead;    // lanes that are the first pair of their expert
};

// id: the expert of pair `lane` (lanes past the last pair: anything)
__device__ __forceinline__ FewExperts few_experts(const FewArgs& a, int id, int lane)
{
    FewExperts f;
    f.id = lane < a.R ? id : -1;
    if (f.id >= a.E) f.id = -1;
    bool lead = f.id >= 0;
    for (int i = 0; i + 1 < a.R; ++i) {
        const int v = __builtin_amdgcn_readlane(f.id, i);
        if (v == f.id && i < lane) lead = false;
    }
    f.lead = __ballot(lead);
    return f;
}

__device__ __forceinline__ unsigned long long lanes_below(int lane)
{
    return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// the lane of the n-th bit of m (n < number of bits)
__device__ __forceinline__ int nth_lane(unsigned long long m, int n, int lane)
{
    const bool it = ((m >> lane) & 1) && __popcll(m & lanes_below(lane)) == n;
    return __builtin_ctzll(__ballot(it));
}

// lane i receives the index of the i-th set bit of m (lanes past the last one: other indices, each once)
__device__ __forceinline__ int compacted(unsigned long long m, int lane)
{
    const int before = __popcll(m & lanes_below(lane));
    const int to = ((m >> lane) & 1) ? before : __popcll(m) + lane - before;
    return __builtin_amdgcn_ds_permute(to * 4, lane);
}

// A storage tile holds 32 channels x 32 K; the operand of the 16-channel instruction is 16 channels x 64 K: lane l
// takes channel l % 16 and K slice l / 16, i.e. half `half` of two neighbouring tiles, 256 bytes at a time.
__device__ __forceinline__ int64_t operand_offset(int half, int lane)
{
    return (int64_t)(lane >> 5) * 1024 + ((lane & 15) + ((lane >> 4) & 1) * 32 + half * 16) * 16;
}

// ------------------------------------------------------------------ gate_up
// LDS of a workgroup that gates and quantises by itself, behind the int8 rows (H + 16 bytes apart)
constexpr int kFewGateTokens = 4;
struct FewGateLds {
    int32_t ids[64];
    float p[64];
    float scale[kFewGateTokens];
    float amax[kFewWaves];
};

// Gating and quantisation of at most four tokens by one workgroup.  Wavefront t < T computes the scores of row t, the others
// share the rows' values; then all of them rank the experts.  (All wavefronts computing all of it for themselves, without
// the first barrier, took 0.7 us longer: the two workgroups of a compute unit share its vector ALUs.)  ids and the int8 rows
// stay in LDS.  orders, ranks: [T][E rounded up to 4]; groups [T][E].
template <int DT, int PER, int XDT>
__device__ __forceinline__ void few_gate(const FewArgs& a, const GateCall& g, int8_t* xs, FewGateLds& l, unsigned* orders,
                                         int* ranks, float* groups, int wave, int lane)
{
    const int T = a.T, E4 = (a.E + 3) & ~3, H = a.H, nv = H >> 3;
    float p[PER];
    // wavefront T + i takes every step-th 512 values of row i % T, from the (i / T)-th on
    const int xi = wave < T ? 0 : wave - T, t = xi % T, part = xi / T, step = (kFewWaves - T - t + T - 1) / T;
    const v8u16* xv = (const v8u16*)((const uint16_t*)g.x + (int64_t)t * H);
    v8u16 held = {0, 0, 0, 0, 0, 0, 0, 0};
    float amax = 0.0f;
    if (wave < T) {
        float sel[PER];
        row_scores<DT, PER>(RowLogits<DT>{g.logits, (int64_t)wave * a.E, (int64_t)T * a.E, g.n_planes, g.plane_bias}, g.bias, a.E,
                            g.k_group, g.group_count, g.group_select_mode, g.norm_type, groups + wave * a.E, lane, p, sel);
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const unsigned u = score_order(sel[i]);
            if (lane + 64 * i < a.E) orders[wave * E4 + lane + 64 * i] = u > 1u ? u : 1u;
        }
    } else {
        for (int i = threadIdx.x - 64 * T; i < T * E4; i += kFewThreads - 64 * T) ranks[i] = 0;
        const int at = part * 64 + lane;
        if (at < nv) held = xv[at];
        for (int i = at; i < nv; i += step * 64) {
            const v8u16 v = i == at ? held : xv[i];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float f = __builtin_fabsf(half_to_f32<XDT>(v[j]));
                amax = f > amax ? f : amax;
            }
        }
        amax = wave_max_dpp(amax);
        if (lane == 0) l.amax[wave] = amax;
    }
    __syncthreads();
    {
        const int W = T == 1 ? 8 : T == 2 ? 4 : 2, r = wave / W;  // T = 3: two wavefronts without a row
        if (r < T) rank_row<PER>(orders + r * E4, a.E, wave - r * W, W, ranks + r * E4, lane);
    }
    if (wave >= T) {
        for (int v = T + t; v < kFewWaves; v += T) amax = l.amax[v] > amax ? l.amax[v] : amax;
        const float s = amax / 127.0f;
        const RowDivisor d = row_divisor(s);
        if (part == 0 && lane == 0) l.scale[t] = (amax == 0.0f) ? 0.0f : s;
        int8_t* q = xs + t * (H + 16);
        const int at = part * 64 + lane;
        for (int i = at; i < nv; i += step * 64) {
            const v8u16 v = i == at ? held : xv[i];
            *(uint2*)(q + i * 8) = d.fast ? quantise_by_row<true, XDT>(v, d) : quantise_by_row<false, XDT>(v, d);
        }
    }
    __syncthreads();
    if (wave < T) place_row<PER>(p, ranks + wave * E4, a.E, a.k, l.ids + wave * a.k, l.p + wave * a.k, lane);
    __syncthreads();
}

// ... and what the down GEMM wants of it, by the first workgroup when its weights are on their way
template <int DT>
__device__ __forceinline__ void few_store_choice(const FewArgs& a, const GateCall& g, const FewGateLds& l, int wave, int lane)
{
    if (wave < a.T)
        store_choice<DT>(lane < a.k ? l.ids[wave * a.k + lane] : 0, lane < a.k ? l.p[wave * a.k + lane] : 0.0f, a.k, g.renorm,
                         g.norm_type, g.routed_scaling_factor, g.eps, (int64_t)wave * a.k, (void*)a.tw, g.x_dtype,
                         (int32_t*)a.ids, lane);
}

// ids and token scales: in LDS if the workgroup gates by itself
__device__ __forceinline__ int few_id(const FewArgs&, const FewGateLds& l, int i) { return l.ids[i]; }
__device__ __forceinline__ int few_id(const FewArgs& a, int, int i) { return a.ids[i]; }
__device__ __forceinline__ float few_x_scale(const FewArgs&, const FewGateLds& l, int t) { return l.scale[t]; }
__device__ __forceinline__ float few_x_scale(const FewArgs& a, int, int t) { return a.x_scale[t]; }

// Workgroup = (expert, 16 gate channels and their 16 up channels), K cut over 8 wavefronts.  UN K steps of 64 are
// requested together (K = 2048: the whole share of a wavefront).  PER > 0: gating and quantisation are done here as
// well, by every workgroup for itself (E <= 64 PER); 0: they came from a launch in front of this one.
template <int UN, int PER, int DT, int XDT>
__global__ __launch_bounds__(kFewThreads, 4) void few_up_kernel(FewArgs a, GateCall gate)
{
    constexpr bool GATE = PER > 0;
    extern __shared__ __attribute__((aligned(16))) int8_t few_lds[];
    __shared__ int32_t acc[16 * 33];
    __shared__ std::conditional_t<GATE, FewGateLds, int> gl;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int units = a.I >> 4, places = a.R < a.E ? a.R : a.E;
    const int b = blockIdx.x;
    const bool shared = b >= places * units;
    const int K = a.H, KB = K >> 6;
    if constexpr (GATE) {
        unsigned* orders = (unsigned*)(few_lds + a.T * (K + 16));
        int* ranks = (int*)(orders + a.T * ((a.E + 3) & ~3));
        few_gate<DT, PER, XDT>(a, gate, few_lds, gl, orders, ranks, (float*)(ranks + a.T * ((a.E + 3) & ~3)), wave, lane);
    }
    int e = 0, rows = a.T, list = lane, p, width;
    unsigned long long mine_mask = 0;
    const int8_t* w;
    const float* sc;
    if (!shared) {
        const int slot = a.by_i16(b);
        p = b - slot * units;
        width = a.I;
        const FewExperts f = few_experts(a, lane < a.R ? few_id(a, gl, lane) : -1, lane);
        if (slot >= __popcll(f.lead)) return;
        e = __builtin_amdgcn_readlane(f.id, nth_lane(f.lead, slot, lane));
        mine_mask = __ballot(f.id == e);
        rows = __popcll(mine_mask) < 16 ? __popcll(mine_mask) : 16;  // the slots of a token are different experts: at most T
        w = a.w13_list ? a.w13_list[e] : a.w13 + (int64_t)e * 2 * a.I * K;
        sc = a.s13_list ? a.s13_list[e] : a.s13 + (int64_t)e * 2 * a.I;
    } else {
        p = b - places * units;
        width = a.S;
        w = a.sw13;
        sc = a.ss13;
    }
    const int64_t tile_row = (int64_t)(K >> 5) * 1024;
    const int8_t* wg = w + (int64_t)(p >> 1) * tile_row + operand_offset(p & 1, lane);
    const int8_t* wu = wg + (int64_t)(width >> 5) * tile_row;
    const int kb0 = KB * wave / kFewWaves, kb1 = KB * (wave + 1) / kFewWaves;

    v4i g[UN], u[UN], t[UN];
    auto request = [&](int kb) {
#pragma unroll
        for (int i = 0; i < UN; ++i) {
            const bool in = kb + i < kb1;
            g[i] = in ? gload16_nt(wg + (int64_t)(kb + i) * 2048) : (v4i){0, 0, 0, 0};
            u[i] = in ? gload16_nt(wu + (int64_t)(kb + i) * 2048) : (v4i){0, 0, 0, 0};
        }
    };
    request(kb0);  // before anything that does not have to be known for it
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (GATE)
        if (b == 0) few_store_choice<DT>(a, gate, gl, wave, lane);
    // token rows: lane l holds row l % 16 of the expert, pair `pair`, token pair / k (shared expert: the token)
    if (!shared) list = compacted(mine_mask, lane);
    const int tok = lane & 15;
    const int pair = __shfl(list, tok, 64);
    const bool valid = tok < rows;
    const int xrow = valid ? (shared ? pair : a.by_k(pair)) : 0;
    const int8_t* xr = GATE ? few_lds + xrow * (K + 16) + (lane >> 4) * 16 : a.xq + (int64_t)xrow * K + (lane >> 4) * 16;
    auto request_tokens = [&](int kb) {
#pragma unroll
        for (int i = 0; i < UN; ++i)
            t[i] = (valid && kb + i < kb1) ? *(const v4i*)(xr + (kb + i) * 64) : (v4i){0, 0, 0, 0};
    };
    request_tokens(kb0);
    // epilogue operands, requested behind the first weights: thread (row, channel)
    const int row = tid >> 4, ch = tid & 15;
    const int epair = __shfl(list, row & 63, 64);
    const bool mine = row < rows;
    float rs = 0.0f, s0 = 0.0f, s1 = 0.0f;
    if (mine) {
        const int t = shared ? epair : a.by_k(epair);
        rs = few_x_scale(a, gl, t);
        s0 = sc[p * 16 + ch];
        s1 = sc[width + p * 16 + ch];
    }
    for (int i = tid; i < rows * 33; i += kFewThreads) acc[i] = 0;
    __syncthreads();
    v4i cg = {0, 0, 0, 0}, cu = {0, 0, 0, 0};
    for (int kb = kb0; kb < kb1; kb += UN) {
#pragma unroll
        for (int i = 0; i < UN; ++i) {
            cg = mfma_i8_16(g[i], t[i], cg);
            cu = mfma_i8_16(u[i], t[i], cu);
        }
        if (kb + UN < kb1) {
            request(kb + UN);
            request_tokens(kb + UN);
        }
    }
    if (valid) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            atomicAdd(&acc[tok * 33 + 4 * (lane >> 4) + j], cg[j]);
            atomicAdd(&acc[tok * 33 + 16 + 4 * (lane >> 4) + j], cu[j]);
        }
    }
    __syncthreads();
    if (row >= 16) return;
    float v = 0.0f;
    if (mine) {
        const int gi = acc[row * 33 + ch], ui = acc[row * 33 + 16 + ch];
        if (!shared) {
            float gg = ((float)gi * rs) * s0, uu = ((float)ui * rs) * s1;
            if (a.limit > 0.0f) {
                gg = gg > a.limit ? a.limit : gg;
                uu = uu > a.limit ? a.limit : uu;
                uu = uu < -a.limit ? -a.limit : uu;
            }
            v = m_silu(gg) * uu;
            a.y[(int64_t)epair * a.I + p * 16 + ch] = v;
        } else {
            // the SwiGLU of the shared expert's operator (dequant_swiglu_quant, swiglu_mode 1)
            float gg = ((float)gi * s0) * rs, uu = ((float)ui * s1) * rs;
            if (a.sh_limit > 0.0f) {
                gg = gg > a.sh_limit ? a.sh_limit : gg;
                uu = uu > a.sh_limit ? a.sh_limit : uu;
                uu = uu < -a.sh_limit ? -a.sh_limit : uu;
            }
            if (a.sh_alpha == 1.0f && a.sh_beta == 0.0f) v = m_silu(gg) * uu;
            else v = (uu + a.sh_beta) * (gg / (1.0f + m_expf(gg * -a.sh_alpha)));
            a.y[(int64_t)a.R * a.I + (int64_t)epair * a.S + p * 16 + ch] = v;
        }
    }
    const float ab = __builtin_fabsf(v);
    float m = ab > 0.0f ? ab : 0.0f;
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) {
        const float o = __shfl_xor(m, off, 64);
        m = o > m ? o : m;
    }
    if (mine && ch == 0) a.ymax[(shared ? a.R * (a.I >> 4) + epair * (a.S >> 4) : epair * (a.I >> 4)) + p] = m;
}

// ------------------------------------------------------------------ re-quantisation
struct FewQuant {
    float amax, inv, s;
    bool shared;
};

__device__ __forceinline__ FewQuant few_quant(const FewArgs& a, int row, float amax)
{
    FewQuant q;
    q.shared = row >= a.R;
    q.amax = amax;
    q.s = q.shared ? q.amax * (float)(1.0 / 127.0) : q.amax / 127.0f;
    q.inv = 1.0f / q.s;
    return q;
}

// the maxima of row `row` (routed pairs, then the shared expert's tokens) that this lane requests: rows of up to 2048
// values are two of them
struct FewMax {
    float m0, m1;
};

__device__ __forceinline__ const float* few_row_maxima(const FewArgs& a, int row, int& n)
{
    const bool shared = row >= a.R;
    n = (shared ? a.S : a.I) >> 4;
    return a.ymax + (shared ? a.R * (a.I >> 4) + (row - a.R) * n : row * n);
}

__device__ __forceinline__ FewMax few_row_pieces(const FewArgs& a, int row, int lane)
{
    int n;
    const float* m = few_row_maxima(a, row, n);
    return FewMax{lane < n ? m[lane] : 0.0f, lane + 64 < n ? m[lane + 64] : 0.0f};
}

// the maximum of the row, in every lane of the wavefront; LONG: of a row that may have more than 2048 values
template <bool LONG>
__device__ __forceinline__ float few_row_max(const FewArgs& a, int row, const FewMax& f, int lane)
{
    int n;
    const float* m = few_row_maxima(a, row, n);
    float v = 0.0f;
    v = f.m0 > v ? f.m0 : v;
    v = f.m1 > v ? f.m1 : v;
    if constexpr (LONG)
        for (int i = lane + 128; i < n; i += 64) v = m[i] > v ? m[i] : v;
    return wave_max_dpp(v);
}

// routed rows multiply by the reciprocal of their scale, the shared expert's rows divide by it
template <bool SHARED>
__device__ __forceinline__ uint32_t few_pack(v4f v, float d)
{
    if constexpr (SHARED) return pack_low_bytes(sat_rint(v[0] / d), sat_rint(v[1] / d), sat_rint(v[2] / d), sat_rint(v[3] / d));
    return quantise_times(v, d);
}

// ... by this.  A row of zeros: 0 * 0, 0 / inf (what else it holds is NaN, which quantises to zero)
__device__ __forceinline__ float few_divisor(const FewQuant& q)
{
    if (q.shared) return q.amax == 0.0f ? __builtin_inff() : q.s;
    return q.amax == 0.0f ? 0.0f : q.inv;
}

// rows of y -> int8 and scale, one workgroup per row
__global__ __launch_bounds__(256) void few_quant_kernel(FewArgs a)
{
    const int row = blockIdx.x;
    const int lane = threadIdx.x & 63;
    const FewQuant q = few_quant(a, row, few_row_max<true>(a, row, few_row_pieces(a, row, lane), lane));
    const float d = few_divisor(q);
    const int width = q.shared ? a.S : a.I;
    const int64_t at = q.shared ? (int64_t)a.R * a.I + (int64_t)(row - a.R) * a.S : (int64_t)row * a.I;
    if (threadIdx.x == 0) a.q1_scale[row] = q.amax == 0.0f ? 0.0f : q.s;
    for (int i = threadIdx.x; i < width >> 2; i += 256)
        ((uint32_t*)(a.q1 + at))[i] = q.shared ? few_pack<true>(((const v4f*)(a.y + at))[i], d)
                                               : few_pack<false>(((const v4f*)(a.y + at))[i], d);
}

// ------------------------------------------------------------------ down GEMM + combine
// Workgroup = CH output channels of every pair.  The int8 rows lie in LDS (quantised here, or copied when
// few_quant_kernel ran); the K ranges of all touched experts (and of the shared expert) are one list of items of UN
// operands, cut evenly over the wavefronts; a wavefront always has the next item's weights in flight.
// CH = 16: the operand of v_mfma_i32_16x16x64_i8 is 16 channels of one K step.  CH = 8 (at most 8 tokens): its rows 8..15
// are the same channels one K step later, and so are its columns; of the product only the quarters with equal halves
// mean anything.  Twice as many workgroups then read whole 128-byte lines each.
template <int CH>
__device__ __forceinline__ int64_t down_offset(int p, int lane)
{
    if constexpr (CH == 16) return operand_offset(p & 1, lane);
    return (int64_t)((lane >> 3) & 1) * 2048 + (int64_t)(lane >> 5) * 1024 + (((lane >> 4) & 1) * 32 + (p & 3) * 8 + (lane & 7)) * 16;
}

// At most 96 registers, as for five wavefronts of a SIMD: beside the four of its own, a workgroup of the routed experts'
// gate_up product (128) has room in the compute unit then.  One register more (104 are taken for 97) and a shared expert on
// the side stream has the compute units to itself: 64 experts of 2048 / 1024, eight slots, shared expert of 2048 values, 9 / 12 /
// 16 tokens 75.5 / 79.4 / 85.2 us with room, 80.8 / 85.3 / 91.4 without.
template <bool QUANT, int NT, int CH>
__global__ __launch_bounds__(NT, 5) void few_down_kernel(FewArgs a)
{
    extern __shared__ __attribute__((aligned(16))) int8_t few_lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nrows = a.R + (a.sw2 ? a.T : 0);
    const int pitch = a.I + 16, pitch_s = a.S + 16;  // rows 16 bytes apart in the banks
    int8_t* q = few_lds;
    int8_t* q_s = q + (int64_t)a.R * pitch;
    int32_t* acc = (int32_t*)(q_s + (a.sw2 ? a.T * pitch_s : 0));  // [nrows][CH + 1]
    float* chs = (float*)(acc + nrows * (CH + 1));                 // [R + 1][CH] channel scales of every pair's expert
    float* qsc = chs + (a.R + 1) * CH;                             // [nrows] scales of the quantised rows
    float* wts = qsc + nrows;                                      // [R] routing weights
    int32_t* idl = (int32_t*)(wts + a.R);                          // [R] ids
    float* qdv = (float*)(idl + a.R);                              // [nrows] QUANT: what the values are multiplied (shared: divided) by
    constexpr int STEPS = 16 / CH;                                 // K steps of an operand
    const int p = blockIdx.x;                                      // channel group
    int my_id = lane < a.R ? a.ids[lane] : -1;
    // What does not depend on the ids is requested before their answer is waited for: the fp32 values, their maxima, the
    // routing weights.  All of it has arrived before the weights are requested: these sit behind conditions, and a wait
    // behind them for anything older would be a wait for every one of them.
    constexpr int NV = QUANT ? kFewInside / 4 / NT : 1;
    v4f yv[NV];
    const int n_y = (a.R * a.I + (a.sw2 ? a.T * a.S : 0)) >> 2;
    FewMax fm = {};
    uint16_t tw = 0;
    if (tid < a.R) tw = a.tw[tid];
    float row_max = 0.0f;
    if constexpr (QUANT) {
        fm = few_row_pieces(a, wave < nrows ? wave : 0, lane);
#pragma unroll
        for (int j = 0; j < NV; ++j)
            yv[j] = tid + j * NT < n_y ? ((const v4f*)a.y)[tid + j * NT] : (v4f){0.0f, 0.0f, 0.0f, 0.0f};
        row_max = few_row_max<false>(a, wave < nrows ? wave : 0, fm, lane);
        for (int r = wave + NT / 64; r < nrows; r += NT / 64) {  // more rows than wavefronts: the maxima wait in LDS
            const float m = few_row_max<false>(a, r, few_row_pieces(a, r, lane), lane);
            if (lane == 0) qdv[r] = m;
        }
        wave_lds_order();
#pragma unroll
        for (int j = 0; j < NV; ++j) asm volatile("" : "+v"(yv[j]));
    }
    asm volatile("" : "+v"(my_id), "+v"(tw));
    const FewExperts f = few_experts(a, my_id, lane);
    const int distinct = __popcll(f.lead);
    constexpr int UN = CH == 16 ? 8 : 4;
    constexpr int ITEM = kFewItem;
    static_assert(ITEM == UN * STEPS, "an item is UN operands");
    const int KB = a.I >> 6, parts = (KB + ITEM - 1) / ITEM;
    const int KBs = a.S >> 6, parts_s = a.sw2 ? (KBs + ITEM - 1) / ITEM : 0;
    const int items = distinct * parts + parts_s;
    const int first = items * wave / (NT / 64), last = items * (wave + 1) / (NT / 64);
    const int64_t lane_off = down_offset<CH>(p, lane);
    const int part = CH == 16 ? 0 : (lane >> 3) & 1;  // which K step of an operand this lane's row and column are

    // item -> weights and K range
    auto request = [&](int it, v4i* w) {
        if (it >= last) return;
        const int8_t* base;
        int kb, end;
        if (it < distinct * parts) {
            const int j = a.by_parts(it);
            kb = (it - j * parts) * ITEM;
            end = KB;
            const int e = __builtin_amdgcn_readlane(f.id, nth_lane(f.lead, j, lane));
            base = a.w2_list ? a.w2_list[e] : a.w2 + (int64_t)e * a.H * a.I;
            base += (int64_t)(p / (32 / CH)) * (a.I >> 5) * 1024;
        } else {
            kb = (it - distinct * parts) * ITEM;
            end = KBs;
            base = a.sw2 + (int64_t)(p / (32 / CH)) * (a.S >> 5) * 1024;
        }
        base += lane_off;
#pragma unroll
        for (int i = 0; i < UN; ++i)
            w[i] = kb + i * STEPS + part < end ? gload16_nt(base + (int64_t)(kb + i * STEPS) * 2048) : (v4i){0, 0, 0, 0};
    };
    v4i wa[UN], wb[UN];
    request(first, wa);

    // channel scales of every pair's expert, behind the weights; they wait in registers until the rows are quantised
    constexpr int NS = (64 * CH + NT - 1) / NT;  // at most 64 pairs
    float chv[NS], chv_s = 0.0f;
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        const int i = tid + j * NT;
        int e = __shfl(f.id, (i / CH) & 63, 64);
        if (e < 0) e = 0;  // a dropped pair: nothing of it is used
        chv[j] = 0.0f;
        if (i < a.R * CH) chv[j] = (a.s2_list ? a.s2_list[e] : a.s2 + (int64_t)e * a.H)[p * CH + i % CH];
    }
    if (a.sw2 && tid < CH) chv_s = a.ss2[p * CH + tid];

    // the zeroed sums, the int8 rows
    for (int i = tid; i < nrows * (CH + 1); i += NT) acc[i] = 0;
    if (tid < a.R) idl[tid] = f.id;  // tid < 64: the first wavefront's lanes
    if (tid < a.R) wts[tid] = a.f16 ? f16_to_f32(tw) : bf16_to_f32(tw);
    if constexpr (QUANT) {
        for (int r = wave; r < nrows; r += NT / 64) {
            const FewQuant fq = few_quant(a, r, r == wave ? row_max : qdv[r]);
            if (lane == 0) {
                qsc[r] = fq.amax == 0.0f ? 0.0f : fq.s;
                qdv[r] = few_divisor(fq);
            }
        }
        __syncthreads();
        const int per = a.I >> 2, per_s = a.S >> 2, n = a.R * per;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int i = tid + j * NT;
            if (i >= n_y) break;
            const bool sh = i >= n;
            const int ii = sh ? i - n : i;
            const int r = sh ? a.by_s4(ii) : a.by_i4(ii), c = ii - r * (sh ? per_s : per);
            const float dv = qdv[sh ? a.R + r : r];
            *(uint32_t*)((sh ? q_s + r * pitch_s : q + r * pitch) + c * 4) = sh ? few_pack<true>(yv[j], dv) : few_pack<false>(yv[j], dv);
        }
    } else {
        const int per = a.I >> 4, per_s = a.S >> 4, n = a.R * per, n_s = a.sw2 ? a.T * per_s : 0;
        for (int i = tid; i < n + n_s; i += NT) {
            const bool sh = i >= n;
            const int ii = sh ? i - n : i;
            const int r = sh ? a.by_s16(ii) : a.by_i16(ii), c = ii - r * (sh ? per_s : per);
            *(v4i*)((sh ? q_s + r * pitch_s : q + r * pitch) + c * 16) = ((const v4i*)a.q1)[i];
        }
        if (tid < nrows) qsc[tid] = a.q1_scale[tid];
    }
#pragma unroll
    for (int j = 0; j < NS; ++j)
        if (tid + j * NT < a.R * CH) chs[tid + j * NT] = chv[j];
    if (a.sw2 && tid < CH) chs[a.R * CH + tid] = chv_s;
    __syncthreads();

    const int tok = lane & (CH - 1), slice = (lane >> 4) * 16;
    const bool means = CH == 16 || (lane >> 5) == part;
    v4i c = {0, 0, 0, 0};
    int held = -1, held_row = 0;  // expert slot whose sums c holds; this lane's row of it
    bool held_valid = false;
    auto flush = [&]() {
        if (held >= 0 && held_valid && means) {
#pragma unroll
            for (int j = 0; j < 4; ++j) atomicAdd(&acc[held_row * (CH + 1) + ((4 * (lane >> 4) + j) & (CH - 1))], c[j]);
        }
        c = (v4i){0, 0, 0, 0};
    };
    auto compute = [&](int it, const v4i* w) {
        const bool sh = it >= distinct * parts;
        const int j = sh ? distinct : a.by_parts(it);
        const int kb = (sh ? it - distinct * parts : it - j * parts) * ITEM;
        if (j != held) {
            flush();
            held = j;
            if (sh) {
                held_valid = tok < a.T;
                held_row = a.R + (held_valid ? tok : 0);
            } else {
                const int e = __builtin_amdgcn_readlane(f.id, nth_lane(f.lead, j, lane));
                const unsigned long long m = __ballot(f.id == e);
                held_valid = tok < __popcll(m);
                held_row = __shfl(compacted(m, lane), held_valid ? tok : 0, 64);
            }
        }
        const int8_t* rowp = (sh ? q_s + (held_row - a.R) * pitch_s : q + held_row * pitch) + kb * 64 + slice;
        const int n = (sh ? KBs : KB) - kb;
#pragma unroll
        for (int i = 0; i < UN; ++i) {
            const int step = i * STEPS + part;
            const v4i t = step < n ? *(const v4i*)(rowp + step * 64) : (v4i){0, 0, 0, 0};
            c = mfma_i8_16(w[i], t, c);
        }
    };
    for (int it = first; it < last; it += 2) {
        request(it + 1, wb);
        compute(it, wa);
        if (it + 1 >= last) break;
        request(it + 2, wa);
        compute(it + 1, wb);
    }
    flush();
    __syncthreads();

    // combine: the weighted value of every (row, channel) by a thread of its own, in the place of its sum, and then a
    // thread per (token, channel): slots in order, the shared expert last, one rounding at the end.  A dropped pair adds
    // +0, which changes no sum that started at +0.
    float* val = (float*)acc;
    for (int i = tid; i < nrows * CH; i += NT) {
        const int r = i / CH, ch = i % CH, at = r * (CH + 1) + ch;
        const bool sh = r >= a.R;
        const float v = ((float)acc[at] * qsc[r]) * chs[(sh ? a.R : r) * CH + ch];
        const float o = a.f16 ? f16_to_f32(f32_to_f16(v)) : bf16_to_f32(f32_to_bf16(v));
        val[at] = sh ? o : idl[r] < 0 ? 0.0f : wts[r] * o;
    }
    __syncthreads();
    for (int i = tid; i < a.T * CH; i += NT) {
        const int t = i / CH, ch = i % CH;
        const float* row = val + t * a.k * (CH + 1) + ch;
        float sum = 0.0f;
        for (int s0 = 0; s0 < a.k; s0 += 8) {
            float v[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) v[s] = s0 + s < a.k ? row[(s0 + s) * (CH + 1)] : 0.0f;
#pragma unroll
            for (int s = 0; s < 8; ++s) sum = sum + v[s];
        }
        if (a.sw2) sum = sum + val[(a.R + t) * (CH + 1) + ch];
        a.out[(int64_t)t * a.H + p * CH + ch] = a.f16 ? f32_to_f16(sum) : f32_to_bf16(sum);
    }
    if (a.load && p == 0 && tid < a.R) {
        const int id = a.ids[tid];
        if (id >= 0 && id < a.E) atomicAdd((unsigned long long*)(a.load + id), 1ull);
    }
}

static size_t few_lds_bytes(const FewArgs& a)
{
    const size_t rows = a.R + (a.sw2 ? a.T : 0);
    return (size_t)a.R * (a.I + 16) + (a.sw2 ? (size_t)a.T * (a.S + 16) : 0) + rows * 17 * 4 + (size_t)(a.R + 1) * 64 +
           rows * 8 + (size_t)a.R * 8;
}

// At most 64 pairs (a lane each) of at most 16 tokens (the columns of the MFMA), whole 64-wide K steps, and int8 rows
// that leave room for two workgroups in a compute unit's LDS.  Measured against pair order (us a layer call, 2 GEMM
// launches of its own, and 4 more for a shared expert): Qwen3 shape, 3 / 4 / 5 / 6 / 8 tokens 34.1 / 39.4 / 47.7 / 54.0 / 70.0
// against 38.6 / 41.5 / 46.7 / 50.4 / 57.3 (every workgroup of the down GEMM has to read all touched experts by itself),
// Zipf(1.1) 27.3 / 32.3 / 36.8 / 40.9 / 53.3 against 34.0 / 35.0 / 36.6 / 37.8 / 40.4; small layer of 8 experts, 10 / 12 / 16
// tokens of two slots 22.2 / 23.1 / 24.2 against 26.3 / 26.3 / 26.5; DeepSeek-V3 shape without a shared expert, 3 / 4 tokens
// 162 / 216 against 167 / 217, with one on its side stream, 1 / 2 / 3 / 4 tokens 78 / 132 / 186 / 229 against 97 / 150 / 204 /
// 240.  So: up to 32 pairs, and with a shared expert as many as fit.
bool few_supported(const FewArgs& a)
{
    return a.T > 0 && a.T <= 16 && a.R <= (a.sw2 ? 64 : 32) && a.H % 64 == 0 && a.I % 64 == 0 && (!a.sw2 || a.S % 64 == 0) &&
           few_lds_bytes(a) <= 80 * 1024 - 512;
}

// up to here every workgroup of the down GEMM re-quantises all rows itself, beyond it a launch of 4.7 us does (one
// token of the DeepSeek-V3 shape, 18 K values: 82 us inside, 78 us with the launch)
static bool few_quant_inside(const FewArgs& a)
{
    return a.I <= 2048 && (!a.sw2 || a.S <= 2048) && (int64_t)a.R * a.I + (a.sw2 ? a.T * a.S : 0) <= kFewInside;
}

// Whether the up kernel gates and quantises by itself (few_up_kernel<., PER > 0>).  Every workgroup does, in front of its
// weights, against a launch in front of it with its hand-over, 3.2 us.  What it costs is the chain of its slowest wavefront:
// the experts that it compares (its share of all of them, 64 at a time, about 25 ns each) and its rounds over a row's values
// (the first of them hides behind the scores, the others take about 30 comparisons each).  Two workgroups of a compute unit
// take turns at its vector ALUs, so beyond one for every unit all of it counts twice, and beyond (nearly) two the others wait.
// us a call inside / in a launch of its own (in brackets the workgroups and the sum below):
//   E =   8, H = 1024, 1 / 2 / 3 / 4 tokens (176 to 704; 1, 4, 68, -)      14.0 / 14.3 / 15.7 / 17.7   17.2 / 16.7 / 16.7 / 17.0
//   E =  32, H = 2048, 1 / 2 / 3 / 4 tokens (128 to 512; 4, 38, 212, 212)  14.1 / 15.7 / 19.2 / 20.9   17.0 / 16.9 / 18.3 / 20.0
//   E =  64, H = 2048, 1 / 2 tokens (256, 512; 8, 92)                      14.9 / 19.8                 17.0 / 20.8
//   E =  64, H = 1024, 3 / 4 tokens of two slots (384, 512; 124)           16.6 / 18.0                 17.1 / 17.4
//   E = 128, H = 2048, 1 token of eight slots (384; 64)                    18.1                        19.5
//                      2 / 3 tokens of four (384, 576; 188, 436)           19.1 / 28.5                 18.4 / 22.1
//   E = 128, H =  512, 2 / 3 tokens (256, 384; 64, 256)                    15.9 / 22.1                 17.1 / 19.4
//   E = 256, H = 2048, 1 / 2 / 3 / 4 tokens (128 to 512; 128, 286, ..)     17.0 / 21.9 / 38.3 / 42.9   16.6 / 18.0 / 22.0 / 24.9
//            H = 1024, 1 token of one slot (64; 128)                       14.9                        16.6
bool few_gates(const FewArgs& a)
{
    const int places = a.R < a.E ? a.R : a.E, T = a.T;
    const int groups = places * (a.I / 16) + (a.sw2 ? a.S / 16 : 0);
    if (T < 1 || T > kFewGateTokens || T * (a.H + 16) > 24 * 1024 || a.E > 256 || a.R > 64 || groups > 576) return false;
    const int rankers = T == 1 ? 8 : T == 2 ? 4 : 2, held = a.E <= 64 ? 1 : a.E <= 128 ? 2 : 4;  // few_gate, few_forward
    const int quantisers = (kFewWaves - T) / T;                                                  // of the row that has fewest
    const int rounds = (a.H + 512 * quantisers - 1) / (512 * quantisers);
    return ((a.E + rankers - 1) / rankers * held + 30 * (rounds - 1)) * (groups > 256 ? 2 : 1) <= 128;
}

int few_forward(const FewArgs& args, const GateCall* gate, hipStream_t st)
{
    if (!few_supported(args)) return MOE355_E_SHAPE;
    FewArgs a = args;
    a.by_k = SmallDivisor(a.k);
    a.by_i4 = SmallDivisor(a.I / 4);
    a.by_i16 = SmallDivisor(a.I / 16);
    a.by_s4 = SmallDivisor(a.S / 4);
    a.by_s16 = SmallDivisor(a.S / 16);
    a.by_parts = SmallDivisor((a.I / 64 + kFewItem - 1) / kFewItem);
    if (gate) {
        const int rc = check_gate(*gate);
        if (rc != MOE355_OK) return rc;
    }
    // the scales are read one by one here, but the operators take none that are not aligned
    for (const void* p : {(const void*)a.xq, (const void*)a.y, (const void*)a.q1, (const void*)a.w13, (const void*)a.w2,
                          (const void*)a.sw13, (const void*)a.sw2, (const void*)a.s13, (const void*)a.s2,
                          (const void*)a.ss13, (const void*)a.ss2})
        if ((uintptr_t)p & 15) return MOE355_E_SHAPE;
    const int places = a.R < a.E ? a.R : a.E;
    const dim3 up((unsigned)(places * (a.I / 16) + (a.sw2 ? a.S / 16 : 0)));
    hipEvent_t ev0, ev1;
    take_profile_events(ev0, ev1);
    const GateCall g = gate ? *gate : GateCall{};
    const size_t up_lds = gate ? (size_t)a.T * (a.H + 16) + (size_t)3 * a.T * ((a.E + 3) & ~3) * 4 : 0;
#define MOE355_FEW_UP(P_, L_, X_)                                                                                     \
    do {                                                                                                             \
        auto kernel = few_up_kernel<4, P_, L_, X_>;                                                                  \
        if (ev0) hipExtLaunchKernelGGL(kernel, up, dim3(kFewThreads), up_lds, st, ev0, ev1, 0, a, g);                 \
        else hipLaunchKernelGGL(kernel, up, dim3(kFewThreads), up_lds, st, a, g);                                     \
    } while (0)
#define MOE355_FEW_UP_PER(L_, X_)                      \
    do {                                                \
        if (a.E <= 64) MOE355_FEW_UP(1, L_, X_);        \
        else if (a.E <= 128) MOE355_FEW_UP(2, L_, X_);  \
        else MOE355_FEW_UP(4, L_, X_);                  \
    } while (0)
#define MOE355_FEW_UP_X(L_)                                \
    do {                                                    \
        if (a.f16) MOE355_FEW_UP_PER(L_, MOE355_DT_F16);    \
        else MOE355_FEW_UP_PER(L_, MOE355_DT_BF16);         \
    } while (0)
    if (!gate) MOE355_FEW_UP(0, MOE355_DT_F32, MOE355_DT_BF16);
    else if (g.logits_dtype == MOE355_DT_F32) MOE355_FEW_UP_X(MOE355_DT_F32);
    else if (g.logits_dtype == MOE355_DT_BF16) MOE355_FEW_UP_X(MOE355_DT_BF16);
    else MOE355_FEW_UP_X(MOE355_DT_F16);
#undef MOE355_FEW_UP_X
#undef MOE355_FEW_UP_PER
#undef MOE355_FEW_UP
    const size_t lds = few_lds_bytes(a);
    const bool inside = few_quant_inside(a);
    if (!inside) hipLaunchKernelGGL(few_quant_kernel, dim3((unsigned)(a.R + (a.sw2 ? a.T : 0))), dim3(256), 0, st, a);
    // 16 channels a workgroup; with fewer of those than half the compute units 8 channels, if the tokens allow it (two tokens
    // of the Qwen3 shape 27.4 -> 25.9 us, 8 of the small layer 21.7 -> 20.9); with fewer than compute units 16 wavefronts in
    // each of them
    const bool narrow = a.T <= 8 && a.H / 16 <= 128;
    const dim3 down((unsigned)(a.H / (narrow ? 8 : 16)));
    const bool wide = a.H / 16 <= 256;
#define MOE355_FEW_DOWN(Q_, N_, C_)                                                                               \
    do {                                                                                                            \
        static OncePerDevice once;                                                                                  \
        if (!allow_dynamic_lds(once, (const void*)few_down_kernel<Q_, N_, C_>, 80 * 1024)) {                        \
            (void)hipGetLastError();                                                                                \
            return MOE355_E_LAUNCH;                                                                                 \
        }                                                                                                           \
        hipLaunchKernelGGL((few_down_kernel<Q_, N_, C_>), down, dim3(N_), lds, st, a);                              \
    } while (0)
    if (narrow && inside) MOE355_FEW_DOWN(true, 1024, 8);
    else if (narrow) MOE355_FEW_DOWN(false, 1024, 8);
    else if (inside && wide) MOE355_FEW_DOWN(true, 1024, 16);
    else if (inside) MOE355_FEW_DOWN(true, 512, 16);
    else if (wide) MOE355_FEW_DOWN(false, 1024, 16);
    else MOE355_FEW_DOWN(false, 512, 16);
#undef MOE355_FEW_DOWN
    return launch_status();
}

}  // namespace moe355
