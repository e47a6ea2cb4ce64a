// The expert MLPs of a few tokens (at most 64 (token, slot) pairs): what the first tokens of a decode
// batch cost is not the weight stream (38 MB of the Qwen3 shape are 5.5 us) but launches, each of them 3 to 6 us with
// its dispatch, its first look at the ids and its last store.  Behind the gating launch there are two here:
//
//   few_up_kernel    gate_up GEMM + SwiGLU of the routed experts AND of the shared expert, and the maxima of every row
//                    piece (atomics on one maximum per row meet at the memory side: 1536 of them cost 12 us);
//   few_down_kernel  re-quantisation, down GEMM and the weighted combine: a workgroup owns 16 output channels of ALL
//                    pairs, so the k rows of a token meet in its LDS and leave as one finished row.
//
// From about 12 K SwiGLU values on every workgroup re-quantising all rows costs more than a launch (few_quant_kernel).
// The ids of at most 64 pairs are one load of one wavefront: every wavefront knows the distinct experts, its expert's
// rows and its share of the work from ballots, without LDS tables or barriers.  Tokens are the 16-column operand of
// v_mfma_i32_16x16x64_i8, so an accumulator is four registers and 8 wavefronts cutting K meet in 2 KB of LDS.
#include <hip/hip_ext.h>

#include "gmm_common.h"
#include "layer_parts.h"

namespace moe355 {

constexpr int kFewThreads = 512;
constexpr int kFewWaves = kFewThreads / 64;

struct FewExperts {
    int id;                     // this lane's pair's expert, or -1
    unsigned long long lead;    // lanes that are the first pair of their expert
};

__device__ __forceinline__ FewExperts few_experts(const FewArgs& a, int lane)
{
    FewExperts f;
    f.id = lane < a.R ? a.ids[lane] : -1;
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
// Workgroup = (expert, 16 gate channels and their 16 up channels), K cut over 8 wavefronts.  UN K steps of 64 are
// requested together (K = 2048: the whole share of a wavefront).
template <int UN>
__global__ __launch_bounds__(kFewThreads, 4) void few_up_kernel(FewArgs a)
{
    __shared__ int32_t acc[16 * 33];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int units = a.I >> 4, places = a.R < a.E ? a.R : a.E;
    const int b = blockIdx.x;
    const bool shared = b >= places * units;
    const int K = a.H, KB = K >> 6;
    int e = 0, rows = a.T, list = lane, p, width;
    const int8_t* w;
    const float* sc;
    if (!shared) {
        const int slot = b / units;
        p = b - slot * units;
        width = a.I;
        const FewExperts f = few_experts(a, lane);
        if (slot >= __popcll(f.lead)) return;
        e = __builtin_amdgcn_readlane(f.id, nth_lane(f.lead, slot, lane));
        const unsigned long long m = __ballot(f.id == e);
        rows = __popcll(m) < 16 ? __popcll(m) : 16;  // the slots of a token are different experts: at most T
        list = compacted(m, lane);
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

    // token rows: lane l holds row l % 16 of the expert, pair `pair`, token pair / k (shared expert: the token)
    const int tok = lane & 15;
    const int pair = __shfl(list, tok, 64);
    const bool valid = tok < rows;
    const int8_t* xr = a.xq + (int64_t)(valid ? (shared ? pair : pair / a.k) : 0) * K + (lane >> 4) * 16;

    v4i g[UN], u[UN], t[UN];
    auto request = [&](int kb) {
#pragma unroll
        for (int i = 0; i < UN; ++i) {
            const bool in = kb + i < kb1;
            g[i] = in ? gload16_nt(wg + (int64_t)(kb + i) * 2048) : (v4i){0, 0, 0, 0};
            u[i] = in ? gload16_nt(wu + (int64_t)(kb + i) * 2048) : (v4i){0, 0, 0, 0};
        }
#pragma unroll
        for (int i = 0; i < UN; ++i)
            t[i] = (valid && kb + i < kb1) ? *(const v4i*)(xr + (kb + i) * 64) : (v4i){0, 0, 0, 0};
    };
    request(kb0);
    // epilogue operands, requested behind the first weights: thread (row, channel)
    const int row = tid >> 4, ch = tid & 15;
    const int epair = __shfl(list, row & 63, 64);
    const bool mine = row < rows;
    float rs = 0.0f, s0 = 0.0f, s1 = 0.0f;
    if (mine) {
        rs = a.x_scale[shared ? epair : epair / a.k];
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
        if (kb + UN < kb1) request(kb + UN);
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

// the maximum of row `row` (routed pairs, then the shared expert's tokens), in every lane of the wavefront
__device__ __forceinline__ float few_row_max(const FewArgs& a, int row, int lane)
{
    const bool shared = row >= a.R;
    const int n = (shared ? a.S : a.I) >> 4;
    const float* m = a.ymax + (shared ? a.R * (a.I >> 4) + (row - a.R) * n : row * n);
    float v = 0.0f;
    for (int i = lane; i < n; i += 64) v = m[i] > v ? m[i] : v;
    return wave_max(v);
}

__device__ __forceinline__ uint32_t few_pack(const FewQuant& q, v4f v)
{
    uint32_t pk = 0u;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int8_t b = (q.amax == 0.0f) ? (int8_t)0 : sat_rint_i8(q.shared ? v[j] / q.s : v[j] * q.inv);
        pk |= (uint32_t)(uint8_t)b << (8 * j);
    }
    return pk;
}

// rows of y -> int8 and scale, one workgroup per row
__global__ __launch_bounds__(256) void few_quant_kernel(FewArgs a)
{
    const int row = blockIdx.x;
    const FewQuant q = few_quant(a, row, few_row_max(a, row, threadIdx.x & 63));
    const int width = q.shared ? a.S : a.I;
    const int64_t at = q.shared ? (int64_t)a.R * a.I + (int64_t)(row - a.R) * a.S : (int64_t)row * a.I;
    if (threadIdx.x == 0) a.q1_scale[row] = q.amax == 0.0f ? 0.0f : q.s;
    for (int i = threadIdx.x; i < width >> 2; i += 256)
        ((uint32_t*)(a.q1 + at))[i] = few_pack(q, ((const v4f*)(a.y + at))[i]);
}

// ------------------------------------------------------------------ down GEMM + combine
// Workgroup = 16 output channels of every pair.  The int8 rows lie in LDS (quantised here, or copied when
// few_quant_kernel ran); the K ranges of all touched experts (and of the shared expert) are one list of items of up to
// 8 K steps of 64, cut evenly over the wavefronts; a wavefront always has the next item's weights in flight.
template <bool QUANT, int NT>
__global__ __launch_bounds__(NT, 4) void few_down_kernel(FewArgs a)
{
    extern __shared__ __attribute__((aligned(16))) int8_t few_lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nrows = a.R + (a.sw2 ? a.T : 0);
    const int pitch = a.I + 16, pitch_s = a.S + 16;  // rows 16 bytes apart in the banks
    int8_t* q = few_lds;
    int8_t* q_s = q + (int64_t)a.R * pitch;
    int32_t* acc = (int32_t*)(q_s + (a.sw2 ? a.T * pitch_s : 0));  // [nrows][17]
    float* chs = (float*)(acc + nrows * 17);                       // [R + 1][16] channel scales of every pair's expert
    float* qsc = chs + (a.R + 1) * 16;                             // [nrows] scales of the quantised rows
    float* wts = qsc + nrows;                                      // [R] routing weights
    int32_t* idl = (int32_t*)(wts + a.R);                          // [R] ids
    const int p = blockIdx.x;                                      // 16-channel group
    const FewExperts f = few_experts(a, lane);
    const int distinct = __popcll(f.lead);
    constexpr int UN = 8;
    const int KB = a.I >> 6, parts = (KB + UN - 1) / UN;
    const int KBs = a.S >> 6, parts_s = a.sw2 ? (KBs + UN - 1) / UN : 0;
    const int items = distinct * parts + parts_s;
    const int first = items * wave / (NT / 64), last = items * (wave + 1) / (NT / 64);
    const int64_t lane_off = operand_offset(p & 1, lane);

    // item -> weights and K range
    auto request = [&](int it, v4i* w) {
        if (it >= last) return;
        const int8_t* base;
        int kb, end;
        if (it < distinct * parts) {
            const int j = it / parts;
            kb = (it - j * parts) * UN;
            end = KB;
            const int e = __builtin_amdgcn_readlane(f.id, nth_lane(f.lead, j, lane));
            base = a.w2_list ? a.w2_list[e] : a.w2 + (int64_t)e * a.H * a.I;
            base += (int64_t)(p >> 1) * (a.I >> 5) * 1024;
        } else {
            kb = (it - distinct * parts) * UN;
            end = KBs;
            base = a.sw2 + (int64_t)(p >> 1) * (a.S >> 5) * 1024;
        }
        base += lane_off;
#pragma unroll
        for (int i = 0; i < UN; ++i)
            w[i] = kb + i < end ? gload16_nt(base + (int64_t)(kb + i) * 2048) : (v4i){0, 0, 0, 0};
    };
    v4i wa[UN], wb[UN];
    request(first, wa);

    // scales and routing weights of the epilogue, the zeroed sums, the int8 rows
    for (int i = tid; i < nrows * 17; i += NT) acc[i] = 0;
    for (int i = tid; i < a.R * 16; i += NT) {
        int e = a.ids[i >> 4];
        if (e < 0 || e >= a.E) e = 0;
        const float* s = a.s2_list ? a.s2_list[e] : a.s2 + (int64_t)e * a.H;
        chs[i] = s[p * 16 + (i & 15)];
    }
    if (a.sw2 && tid < 16) chs[a.R * 16 + tid] = a.ss2[p * 16 + tid];
    if constexpr (QUANT) {
        for (int r = wave; r < nrows; r += (NT / 64)) {
            const float m = few_row_max(a, r, lane);
            if (lane == 0) qsc[r] = m;  // the maximum for now
        }
        __syncthreads();
    } else {
        if (tid < nrows) qsc[tid] = a.q1_scale[tid];
    }
    if (tid < a.R) idl[tid] = f.id;  // tid < 64: the first wavefront's lanes
    if (tid < a.R) wts[tid] = a.f16 ? f16_to_f32(a.tw[tid]) : bf16_to_f32(a.tw[tid]);
    if constexpr (QUANT) {
        const int per = a.I >> 2, per_s = a.S >> 2, n = a.R * per, n_s = a.sw2 ? a.T * per_s : 0;
        for (int i = tid; i < n + n_s; i += NT) {
            const bool sh = i >= n;
            const int ii = sh ? i - n : i;
            const int r = ii / (sh ? per_s : per), c = ii - r * (sh ? per_s : per);
            const FewQuant fq = few_quant(a, sh ? a.R + r : r, qsc[sh ? a.R + r : r]);
            *(uint32_t*)((sh ? q_s + r * pitch_s : q + r * pitch) + c * 4) = few_pack(fq, ((const v4f*)a.y)[i]);
        }
    } else {
        const int per = a.I >> 4, per_s = a.S >> 4, n = a.R * per, n_s = a.sw2 ? a.T * per_s : 0;
        for (int i = tid; i < n + n_s; i += NT) {
            const bool sh = i >= n;
            const int ii = sh ? i - n : i;
            const int r = ii / (sh ? per_s : per), c = ii - r * (sh ? per_s : per);
            *(v4i*)((sh ? q_s + r * pitch_s : q + r * pitch) + c * 16) = ((const v4i*)a.q1)[i];
        }
    }
    __syncthreads();
    if constexpr (QUANT) {  // read again behind the next barrier only
        if (tid < nrows) qsc[tid] = qsc[tid] == 0.0f ? 0.0f : few_quant(a, tid, qsc[tid]).s;
    }

    const int tok = lane & 15, slice = (lane >> 4) * 16;
    v4i c = {0, 0, 0, 0};
    int held = -1, held_row = 0;  // expert slot whose sums c holds; this lane's row of it
    bool held_valid = false;
    auto flush = [&]() {
        if (held >= 0 && held_valid) {
#pragma unroll
            for (int j = 0; j < 4; ++j) atomicAdd(&acc[held_row * 17 + 4 * (lane >> 4) + j], c[j]);
        }
        c = (v4i){0, 0, 0, 0};
    };
    auto compute = [&](int it, const v4i* w) {
        const bool sh = it >= distinct * parts;
        const int j = sh ? distinct : it / parts;
        const int kb = (sh ? it - distinct * parts : it - j * parts) * UN;
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
            const v4i t = i < n ? *(const v4i*)(rowp + i * 64) : (v4i){0, 0, 0, 0};
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

    // combine: thread (token, channel); slots in order, the shared expert last, one rounding at the end
    for (int i = tid; i < a.T * 16; i += NT) {
        const int t = i >> 4, ch = i & 15;
        float sum = 0.0f;
        for (int s = 0; s < a.k; ++s) {
            const int r = t * a.k + s;
            if (idl[r] < 0) continue;  // a dropped pair
            const float v = ((float)acc[r * 17 + ch] * qsc[r]) * chs[r * 16 + ch];
            const float o = a.f16 ? f16_to_f32(f32_to_f16(v)) : bf16_to_f32(f32_to_bf16(v));
            const float pr = wts[r] * o;
            sum = sum + pr;
        }
        if (a.sw2) {
            const int r = a.R + t;
            const float v = ((float)acc[r * 17 + ch] * qsc[r]) * chs[a.R * 16 + ch];
            sum = sum + (a.f16 ? f16_to_f32(f32_to_f16(v)) : bf16_to_f32(f32_to_bf16(v)));
        }
        a.out[(int64_t)t * a.H + p * 16 + ch] = a.f16 ? f32_to_f16(sum) : f32_to_bf16(sum);
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
           rows * 4 + (size_t)a.R * 8;
}

// At most 64 pairs (a lane each) of at most 16 tokens (the columns of the MFMA), whole 64-wide K steps, and int8 rows
// that leave room for two workgroups in a compute unit's LDS.  Measured against pair order (us a layer call, 2 GEMM
// launches of its own, and 4 more for a shared expert): Qwen3 shape, 1 / 2 / 4 / 8 tokens 20.6 / 27.5 / 42 / 74 against
// 27.0 / 32.2 / 39 / 60 (128 workgroups of the down GEMM have to read all touched experts by themselves); small layer
// of 8 experts, 1 / 4 / 8 / 16 tokens of two slots 17 / 20 / 23 / 26 against 24 / 25 / 27 / 25; DeepSeek-V3 shape with a
// shared expert on its side stream, 1 / 2 / 3 / 4 tokens 78 / 132 / 186 / 229 against 97 / 150 / 204 / 240, without one
// 3 tokens 179 against 180.  So: up to 16 pairs, and with a shared expert as many as fit.
bool few_supported(const FewArgs& a)
{
    return a.T > 0 && a.T <= 16 && a.R <= (a.sw2 ? 64 : 16) && a.H % 64 == 0 && a.I % 64 == 0 && (!a.sw2 || a.S % 64 == 0) &&
           few_lds_bytes(a) <= 80 * 1024 - 512;
}

// up to here every workgroup of the down GEMM re-quantises all rows itself, beyond it a launch of 4.7 us does (one
// token of the DeepSeek-V3 shape, 18 K values: 82 us inside, 78 us with the launch)
static bool few_quant_inside(const FewArgs& a) { return (int64_t)a.R * a.I + (a.sw2 ? a.T * a.S : 0) <= 12 * 1024; }

int few_forward(const FewArgs& a, hipStream_t st)
{
    if (!few_supported(a)) return MOE355_E_SHAPE;
    // the scales are read one by one here, but the operators take none that are not aligned
    for (const void* p : {(const void*)a.xq, (const void*)a.y, (const void*)a.q1, (const void*)a.w13, (const void*)a.w2,
                          (const void*)a.sw13, (const void*)a.sw2, (const void*)a.s13, (const void*)a.s2,
                          (const void*)a.ss13, (const void*)a.ss2})
        if ((uintptr_t)p & 15) return MOE355_E_SHAPE;
    const int places = a.R < a.E ? a.R : a.E;
    const dim3 up((unsigned)(places * (a.I / 16) + (a.sw2 ? a.S / 16 : 0)));
    hipEvent_t ev0, ev1;
    take_profile_events(ev0, ev1);
    if (ev0) hipExtLaunchKernelGGL(few_up_kernel<4>, up, dim3(kFewThreads), 0, st, ev0, ev1, 0, a);
    else hipLaunchKernelGGL(few_up_kernel<4>, up, dim3(kFewThreads), 0, st, a);
    const size_t lds = few_lds_bytes(a);
    const bool inside = few_quant_inside(a);
    if (!inside) hipLaunchKernelGGL(few_quant_kernel, dim3((unsigned)(a.R + (a.sw2 ? a.T : 0))), dim3(256), 0, st, a);
    const dim3 down((unsigned)(a.H / 16));
    // fewer workgroups than compute units: 16 wavefronts in each of them
    const bool wide = a.H / 16 <= 256;
#define MOE355_FEW_DOWN(Q_, N_)                                                                                   \
    do {                                                                                                            \
        static OncePerDevice once;                                                                                  \
        if (!allow_dynamic_lds(once, (const void*)few_down_kernel<Q_, N_>, 80 * 1024)) {                            \
            (void)hipGetLastError();                                                                                \
            return MOE355_E_LAUNCH;                                                                                 \
        }                                                                                                           \
        hipLaunchKernelGGL((few_down_kernel<Q_, N_>), down, dim3(N_), lds, st, a);                                  \
    } while (0)
    if (inside && wide) MOE355_FEW_DOWN(true, 1024);
    else if (inside) MOE355_FEW_DOWN(true, 512);
    else if (wide) MOE355_FEW_DOWN(false, 1024);
    else MOE355_FEW_DOWN(false, 512);
#undef MOE355_FEW_DOWN
    return launch_status();
}

}  // namespace moe355
