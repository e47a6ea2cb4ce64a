// W4A8 grouped GEMM: int4 weights (two per byte), int8 activations, fp32 scales per K group.
//
// Weight-streaming kernel (the W4A8 shapes are HBM-bound: half the weight bytes of W8A8).
// Storage tile = 32 channels x 64 K in 1 KiB: lane l (channel l%32, K half l/32) holds 16 bytes;
// byte j carries, in its low nibble, w[k = 64*kb + 16*(l/32) + j] (first 32-wide K step) and in its
// high nibble w[k + 32] (second K step).  One 16-byte load therefore feeds two MFMAs.  A nibble is
// moved into the top half of its byte ((v << 4) & 0xF0..., v & 0xF0...), which is the signed int8
// value 16*w: the int32 accumulator is exactly 16x the true sum and is shifted back before use.
// Every `group` K values the accumulator is folded into fp32, f += float(acc) * scale[e, g, n], in
// ascending group order (one wavefront owns the whole K range of its channels, so the order is the
// sequential one), then f (+ bias) * token_scale goes through the shared epilogues.
#include <hip/hip_ext.h>

#include <type_traits>

#include "gmm_common.h"
#include "gmm_tiled.h"
#include "layer_parts.h"

namespace moe355 {

// ------------------------------------------------------------------ format cast
// SRC 0: int8 [E, N, K] holding one int4 value (-8..7) each (checkpoint order).
// SRC 1: packed [E, K, N/2] bytes, low nibble = even channel (the reference's packing,
//        vllm_ascend/quantization/methods/w4a8.py:327-336).
template <int SRC>
__global__ __launch_bounds__(256) void format_cast_nz_int4_kernel(const uint8_t* __restrict__ w, int64_t E, int64_t N,
                                                                  int64_t K, uint8_t* __restrict__ out)
{
    const int64_t total = E * N * K / 32;  // 16-byte chunks (32 nibbles each)
    const int64_t KB = K / 64, NB = N / 32;
    for (int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x; id < total; id += (int64_t)gridDim.x * 256) {
        const int lane = (int)(id & 63);
        const int64_t tile = id >> 6;
        const int64_t kb = tile % KB;
        const int64_t nb = (tile / KB) % NB;
        const int64_t e = tile / (KB * NB);
        const int64_t n = nb * 32 + (lane & 31);
        const int64_t k0 = kb * 64 + (lane >> 5) * 16;
        uint32_t p[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            uint32_t lo, hi;
            if constexpr (SRC == 0) {
                lo = w[(e * N + n) * K + k0 + j] & 0xFu;
                hi = w[(e * N + n) * K + k0 + 32 + j] & 0xFu;
            } else {
                const uint8_t b0 = w[(e * K + k0 + j) * (N / 2) + (n >> 1)];
                const uint8_t b1 = w[(e * K + k0 + 32 + j) * (N / 2) + (n >> 1)];
                lo = (n & 1) ? (b0 >> 4) : (b0 & 0xFu);
                hi = (n & 1) ? (b1 >> 4) : (b1 & 0xFu);
            }
            p[j >> 2] |= (lo | (hi << 4)) << (8 * (j & 3));
        }
        *(v4i*)(out + id * 16) = (v4i){(int)p[0], (int)p[1], (int)p[2], (int)p[3]};
    }
}

// corr[e, n] = 8 * sum_g float(sum_{k in g} w[e, n, k]) * scale[e, g, n]  (g ascending, fp32):
// the term the Ascend kernel's unsigned-nibble trick adds (x = (x - 8) + 8), which callers of the
// int4 op pass in as `bias` / `weight_assist_matrix`.  One wavefront per (expert, 32-channel tile).
__global__ __launch_bounds__(256) void w4_offset_correction_kernel(const uint8_t* __restrict__ w4,
                                                                   const float* __restrict__ gscale, int E, int N,
                                                                   int K, int group, float* __restrict__ corr)
{
    const int lane = threadIdx.x & 63;
    const int64_t tile_row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int NB = N >> 5, KB64 = K >> 6;
    if (tile_row >= (int64_t)E * NB) return;
    const int e = (int)(tile_row / NB), nb = (int)(tile_row % NB);
    const uint8_t* wp = w4 + (tile_row * KB64) * 1024 + lane * 16;
    const int steps_per_group = group >> 6;
    const int n_groups = K / group;
    const int ch = nb * 32 + (lane & 31);
    float total = 0.0f;
    for (int g = 0; g < n_groups; ++g) {
        int sum = 0;
        for (int t = 0; t < steps_per_group; ++t) {
            const v4i v = *(const v4i*)(wp + (int64_t)(g * steps_per_group + t) * 1024);
#pragma unroll
            for (int d = 0; d < 4; ++d) {
#pragma unroll
                for (int b = 0; b < 8; ++b) sum += ((int)((unsigned)v[d] << (28 - 4 * b))) >> 28;  // signed nibble b
            }
        }
        sum += __shfl_xor(sum, 32, 64);  // the two K halves of the tile
        total = total + (float)sum * gscale[((int64_t)e * n_groups + g) * N + ch];
    }
    if (lane < 32) corr[(int64_t)e * N + ch] = 8.0f * total;
}

struct W4Args {
    GmmArgs g;            // x, gl, R, K, N, E, row_scale, limit, outputs; g.w unused
    const uint8_t* w4;    // tiled int4 storage
    const float* gscale;  // [E, K/group, N]
    const float* bias;    // [E, N] or null, added before the token scale
    int group;            // K values per scale group (multiple of 64)
    TileMap tm;           // sorted rows: the list of chunks, built by the routing launch, or null (found from the group list)
};

__device__ __forceinline__ v4i nib_lo(v4i v)
{
    return (v4i){(int)(((unsigned)v[0] << 4) & 0xF0F0F0F0u), (int)(((unsigned)v[1] << 4) & 0xF0F0F0F0u),
                 (int)(((unsigned)v[2] << 4) & 0xF0F0F0F0u), (int)(((unsigned)v[3] << 4) & 0xF0F0F0F0u)};
}
__device__ __forceinline__ v4i nib_hi(v4i v)
{
    return (v4i){(int)((unsigned)v[0] & 0xF0F0F0F0u), (int)((unsigned)v[1] & 0xF0F0F0F0u),
                 (int)((unsigned)v[2] & 0xF0F0F0F0u), (int)((unsigned)v[3] & 0xF0F0F0F0u)};
}

// Float twin of epilogue_run: g/u already hold sum_g float(acc_g)*scale_g (+ bias); the token scale is
// applied here, last.
__device__ __forceinline__ void dequant_run_w4(const GmmArgs& a, const float* g, const float* u, float rs, v4u16& o0, v4u16& o1)
{
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        o0[j] = a.out_f16 ? f32_to_f16(g[j] * rs) : f32_to_bf16(g[j] * rs);
        o1[j] = a.out_f16 ? f32_to_f16(u[j] * rs) : f32_to_bf16(u[j] * rs);
    }
}
__device__ __forceinline__ v4f swiglu_run_w4(const GmmArgs& a, const float* g, const float* u, float rs)
{
    v4f y;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        float gg = g[j] * rs;
        float uu = u[j] * rs;
        if (a.limit > 0.0f) {
            gg = gg > a.limit ? a.limit : gg;
            uu = uu > a.limit ? a.limit : uu;
            uu = uu < -a.limit ? -a.limit : uu;
        }
        y[j] = m_silu(gg) * uu;
    }
    return y;
}
template <int EPI>
__device__ __forceinline__ void epilogue_run_w4(const GmmArgs& a, int64_t row, bool valid, int c0, int c1,
                                                const float* g, const float* u, float rs)
{
    if (!valid) return;
    if constexpr (EPI == EPI_DEQUANT) {
        v4u16 o0, o1;
        dequant_run_w4(a, g, u, rs, o0, o1);
        *(v4u16*)(a.out + row * a.N + c0) = o0;
        *(v4u16*)(a.out + row * a.N + c1) = o1;
    } else {
        *(v4f*)(a.y + row * (a.N >> 1) + c0) = swiglu_run_w4(a, g, u, rs);
    }
}

// Chunk c of the list "rows of expert 0 in pieces of CHUNK rows, then expert 1, ...": which expert, which
// rows, and whether it is the expert's only chunk.  Every lane returns the same answer; false past the last chunk.  Lane l owns experts
// [l*seg, (l+1)*seg): local counts, a wavefront scan, then a short walk inside the owning lane's segment.
__device__ __forceinline__ bool find_chunk(const int64_t* gl, int gl_type, int E, int c, int CHUNK, int lane, int& e,
                                           int64_t& row0, int64_t& row1, bool& only_chunk)
{
    auto rows_of = [&](int i) -> int {
        const int64_t m = (gl_type == MOE355_GL_COUNT) ? gl[i] : gl[i] - (i > 0 ? gl[i - 1] : 0);
        return m < 0 ? 0 : (int)m;
    };
    const int seg = (E + 63) >> 6;
    const int e0 = lane * seg;
    int rows = 0, chunks = 0;
    for (int j = 0; j < seg; ++j) {
        if (e0 + j < E) {
            const int m = rows_of(e0 + j);
            rows += m;
            chunks += (m + CHUNK - 1) / CHUNK;
        }
    }
    int inc_rows = rows, inc_chunks = chunks;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int r = __shfl_up(inc_rows, off, 64), k = __shfl_up(inc_chunks, off, 64);
        if (lane >= off) {
            inc_rows += r;
            inc_chunks += k;
        }
    }
    if (c >= __shfl(inc_chunks, 63, 64)) return false;
    const uint64_t owns = __ballot(c < inc_chunks);  // lanes at or after the owner
    const int owner = __builtin_ctzll(owns);
    int cc = __shfl(inc_chunks - chunks, owner, 64);
    int64_t rr = __shfl(inc_rows - rows, owner, 64);
    const int oe0 = owner * seg;
    for (int j = 0; j < seg; ++j) {
        const int i = oe0 + j;
        if (i >= E) break;
        const int m = rows_of(i);
        const int nc = (m + CHUNK - 1) / CHUNK;
        if (c - cc < nc) {
            e = i;
            row0 = rr + (int64_t)(c - cc) * CHUNK;
            row1 = rr + m;
            only_chunk = nc == 1;
            return true;
        }
        cc += nc;
        rr += m;
    }
    return false;
}

// One wavefront per unit (chunk of up to 64 rows of one expert, 32 channels), whole K range in ascending order (the fp32
// sum over scale groups has one fixed order).  An expert with many rows becomes many units that run side by side on
// different CUs and find the expert's weights in L2 / Infinity Cache, instead of one wavefront streaming the same weights
// once per 32 rows.
// 32 channels instead of a pair of 32-channel tiles: accumulators and fp32 sums are 64 registers, four wavefronts fit a SIMD
// (with up to 32 scale groups, see w4_scales_in_lds).
// The vector instructions of the fold and of the unpacking, the MFMAs, the LDS reads and the wait for memory follow each
// other in a wavefront, so what runs beside them is other wavefronts.  For the gate_up product the 32 channels are 16 of the
// gate and the 16 of the up projection that belong to them, out of half a storage tile each: they meet in one lane.
// The four wavefronts of a workgroup share the chunk's tokens: stages of 8 KiB (two K blocks of 64 rows, or four of 32 for a
// chunk of at most 32 rows) in a ring of three, copied by LDS-direct loads (no registers) two stages ahead, and one barrier
// per stage.  A wavefront requests its weights two stages ahead as well, between the tokens of the same stages: the memory
// counter retires loads in order, so that the wait for a stage is a count.
// The fold is conversion, product and sum alone: no shift (the scales in LDS are a sixteenth) and no clearing (the first
// product of a group starts from the instruction's own zero).
// What bounds it: the weight stream where the experts have one chunk each (6.1 to 6.4 TB/s), the vector unit and the MFMAs,
// which share its issue, where a hot expert's chunks find their weights in L2.  DeepSeek-V3 shape, groups of 256, us a layer
// call on 64 channels per wavefront with two of them on a SIMD, tokens through registers and a barrier every two K blocks
// of 64 / on this: uniform 100 / 600 / 1024 tokens 928 / 1047 / 1164 -> 876 / 983 / 1085, Zipf(1.1) 256 / 512 / 1024 tokens
// 428 / 606 / 890 -> 391 / 563 / 838.  More loads in flight (three or four stages of weights, three of tokens, then three
// wavefronts on a SIMD) 2 to 4 % slower; the chunks of hot experts first, or spread among the others, 0 to 2 % slower than in
// the order of the experts; all weights through the caches 1037 -> 1126 at 600 tokens.
constexpr int kW4Chunk = 64;
constexpr int kW4LdsGroups = 32;     // K groups whose scales the pair-order kernel keeps in LDS (8 KiB per wavefront)
constexpr int kW4StageBytes = 8192;  // LDS bytes of the tokens of one stage
constexpr int kW4Ring = 3 * kW4StageBytes;

// LDS: the ring of token stages, the group scales of four times 32 channels
static int64_t w4_lds_bytes(int64_t n_groups) { return kW4Ring + n_groups * 512; }
constexpr int kW4LdsMax = 163840;
// With the scales in LDS four workgroups fit a compute unit up to 32 groups, three up to 58, two up to 112 and one up to 272;
// with the scales read from memory in every fold four always do.  Two or more of them win at any size; a single one wins as long
// as the launch is about two rounds of the chip (`blocks`, an upper bound of the workgroups that have rows, below two and a
// half).  Layers, us a call with the scales in LDS / from memory, uniform (Zipf(1.1)):
//   48 groups: 128 experts of 3072 / 1024, 64 / 400 / 1200 tokens 154 / 178 / 335 against 174 / 203 / 383 (89 / 165 / 317 against
//     103 / 187 / 360); 56: 256 of 7168 / 2048, 50 / 600 / 1024 tokens 758 / 1086 / 1237 against 848 / 1195 / 1365 (512 tokens 674
//     against 733)
//   80 groups: 64 of 5120 / 1536, 50 / 200 / 800 tokens 192 / 206 / 416 against 223 / 234 / 449 (123 / 203 / 408 against 146 / 247
//     / 435); 112: 256 of 7168 / 2048, 50 / 600 / 1024 tokens 1010 / 1385 / 1555 against 1107 / 1484 / 1694 (512 tokens 889
//     against 951)
//   128 groups, by blocks: 8 of 8192 / 1024, 224 / 320 / 416 95 / 104 / 175 against 129 / 129 / 160 (99 / 105 / 177 against 131 /
//     138 / 163); 16 of 2048 / 8192, 352 / 448 / 544 / 656 / 848 153 / 204 / 286 / 300 / 419 against 205 / 243 / 314 / 291 / 370
//     (202 / 237 / 276 / 334 at 352 / 448 / 544 / 656 against 232 / 279 / 305 / 334); 16 of 8192 / 2048, 576 / 640 / 704 144 / 145 /
//     155 against 147 / 148 / 167 (150 / 163 / 205 against 175 / 180 / 195); 32 of 8192 / 1024, 544 / 608 143 / 145 against 147 / 149
//     (136 / 158 against 138 / 174); 18 of 8192 / 2048, 640 195 against 162 (196 against 188); 32 of them, 1184 / 1408 258 / 330
//     against 213 / 275 (264 / 407 against 227 / 349)
//   224 groups, 8 of 4096 / 14336, 320 / 512 / 576 / 640 / 704 / 896 235 / 449 / 510 / 525 / 579 / 755 against 306 / 508 / 467 / 510 /
//     538 / 679 (268 / 440 / 496 / 526 / 635 against 360 / 487 / 536 / 583 / 627, 899 against 808 at 1024); 272 groups, 8 of 2048 /
//     17408, 224 / 320 / 416 / 528 262 / 342 / 526 / 583 against 373 / 427 / 490 / 553 (276 / 331 / 522 / 573 against 395 / 450 / 533 / 608)
static bool w4_scales_in_lds(int64_t n_groups, int64_t blocks)
{
    return w4_lds_bytes(n_groups) <= (2 * blocks < 5 * 256 ? kW4LdsMax : kW4LdsMax / 2);
}

#define MOE355_LPTR(p) ((__attribute__((address_space(3))) void*)(p))

// what the bodies of a chunk share: everything but the lane's own offsets is the same in all lanes of a wavefront
struct W4Unit {
    int8_t* lds;
    const float* scales;   // LDS: scale / 16 (shift: scale) of the unit's channels, [group][32]
    const float* gscale;   // scales of the expert, [group][N]
    const uint8_t* w;      // the lane's 16 bytes of the unit's first K block
    int e, u, first, row0, row1;  // first: unit of the workgroup's first wavefront; row1: the end of the expert's rows
    bool have, shift;
};

// NB: blocks of 32 rows.  STREAM: the expert has a single chunk, nobody else reads these weights: non-temporal loads (the
// faster pure stream).  That goes for the number of chunks, not of rows: with the last 32 rows and fewer of a hot expert past
// the caches too, Zipf(1.1), 128 / 256 / 512 / 1024 tokens took 322 / 413 / 623 / 896 us a layer call and take 314 / 406 / 615 /
// 884 (512 tokens: 1766 and 802 MB read from HBM by the two products, 1708 and 770 so).  Otherwise the sibling chunks of the expert run
// at the same time and ordinary loads let them share a fetch: in L2 where a chunk has a multiple of eight workgroups (N of about
// a multiple of 1024), so that the same channels of all chunks are on one XCD, else in the last-level cache.
template <int EPI, bool LDS_SCALES, int NB, bool STREAM, bool FAR>
__device__ __forceinline__ void w4_chunk_body(const W4Args& p, const W4Unit& t, const __amdgpu_buffer_rsrc_t xr, const int8_t* xb,
                                              const int64_t* xo)
{
    constexpr int BLOCKS = 4 / NB;            // K blocks of a stage
    constexpr int BLOCK_BYTES = NB * 2048;
    const GmmArgs& a = p.g;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int c32 = lane & 31, hi = lane >> 5;
    const int KB64 = a.K >> 6;
    const int steps_per_group = p.group >> 6;  // K blocks per scale group
    // channel of the lane's run q (0..3) of four results: 8 q + 4 hi + 0..3 of the unit
    auto run_channel = [&](int q) {
        return EPI == EPI_SWIGLU ? (q >= 2 ? a.N >> 1 : 0) + t.u * 16 + 8 * (q & 1) + 4 * hi : t.u * 32 + 8 * q + 4 * hi;
    };
    int frag[2];  // where this lane's operand bytes of K 0..31 and 32..63 of a block lie; rows 32.. are 2048 bytes further
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) frag[kk] = c32 * 64 + (((2 * kk + hi) ^ ((c32 >> 2) & 3)) * 16);

    v16i c[NB];
    float f[NB][16];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        c[b] = (v16i){0};
#pragma unroll
        for (int v = 0; v < 16; ++v) f[b][v] = 0.0f;
    }
    int in_group = 0, grp = 0;
    // f += float(acc / 16) * scale[e, grp, channel]
    auto fold = [&]() {
        if (t.shift) {
#pragma unroll
            for (int b = 0; b < NB; ++b) c[b] = c[b] >> 4;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            v4f s;
            if constexpr (LDS_SCALES) s = *(const v4f*)(t.scales + grp * 32 + 8 * q + 4 * hi);
            else s = *(const v4f*)(t.gscale + (int64_t)grp * a.N + run_channel(q));
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int j = 0; j < 4; ++j) f[b][4 * q + j] = f[b][4 * q + j] + (float)c[b][4 * q + j] * s[j];
        }
        in_group = 0;
        ++grp;
    };

    // A wavefront copies 16 rows x 64 values by one load.  NB == 2: rows 16 w .. of both blocks of a stage, else both halves of
    // the rows of block w.
    auto load_tokens = [&](int8_t* stage, int kb) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int kw = kb + (NB == 2 ? i : wave);
            const int k = kw < KB64 ? kw : KB64 - 1;  // past the end: the last block again, never used
            int8_t* to = stage + (NB == 2 ? i * BLOCK_BYTES + wave * 1024 : wave * BLOCK_BYTES + i * 1024);
            const int64_t from = xo[NB == 2 ? 0 : i];
            if constexpr (FAR) *(v4i*)(to + lane * 16) = *(const v4i*)(xb + from + (int64_t)k * 64);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, MOE355_LPTR(to), 16, (int)from, k * 64, 0, 0);
        }
    };
    v4i w[2 * BLOCKS];  // weights of the two stages in flight
    auto load_weights = [&](int slot, int kb) {
        const int k = kb < KB64 ? kb : KB64 - 1;
        if constexpr (STREAM) w[slot] = __builtin_nontemporal_load((const v4i*)(t.w + (int64_t)k * 1024));
        else w[slot] = *(const v4i*)(t.w + (int64_t)k * 1024);
    };
    // one K block of a stage
    auto block = [&](const int8_t* st, v4i wv) {
        v4i x[2][NB];  // [K half][rows]
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int b = 0; b < NB; ++b) x[kk][b] = *(const v4i*)(st + b * 2048 + frag[kk]);
        const v4i lo = nib_lo(wv), up = nib_hi(wv);
        const bool first = in_group == 0;  // of its scale group: the accumulators start from the instruction's own zero
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if (first) c[b] = mfma_i8(lo, x[0][b], (v16i){0});
            else c[b] = mfma_i8(lo, x[0][b], c[b]);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) c[b] = mfma_i8(up, x[1][b], c[b]);
        if (++in_group == steps_per_group) fold();
    };
    const int n_stages = (KB64 + 2 * BLOCKS - 1) / (2 * BLOCKS) * 2;  // the registers go by pairs of stages: the last ones may hold nothing
    int8_t* st_now = t.lds;  // stage s, and where stage s + 2 goes
    int8_t* st_load = t.lds + 2 * kW4StageBytes;
    auto next_stage = [&](int8_t* st) { return st == t.lds + 2 * kW4StageBytes ? t.lds : st + kW4StageBytes; };
    // Stage s.  PAR: which half of the weight registers; LOAD: stage s + 2 is requested; LAST: the last stage.
    // Behind the tokens of a stage there are its weights, the tokens and the weights of the next stage when its turn comes;
    // in front of the last one the next stage's are missing.
    auto run_stage = [&](auto par, auto load, auto last, int s) {
        constexpr int PAR = decltype(par)::value;
        constexpr bool LOAD = decltype(load)::value, LAST = decltype(last)::value;
        constexpr int BEHIND = LAST ? 0 : 2 * BLOCKS + 2;
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(BEHIND) : "memory");
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (LOAD) load_tokens(st_load, (s + 2) * BLOCKS);
#pragma unroll
        for (int i = 0; i < BLOCKS; ++i) {
            if (!LOAD && s * BLOCKS + i >= KB64) break;
            block(st_now + i * BLOCK_BYTES, w[PAR * BLOCKS + i]);
            if constexpr (LOAD) load_weights(PAR * BLOCKS + i, (s + 2) * BLOCKS + i);
        }
        __builtin_amdgcn_sched_barrier(0);
        st_now = next_stage(st_now);
        st_load = next_stage(st_load);
    };
    {
        const std::integral_constant<int, 0> p0;
        const std::integral_constant<int, 1> p1;
        const std::true_type yes;
        const std::false_type no;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            load_tokens(t.lds + s * kW4StageBytes, s * BLOCKS);
#pragma unroll
            for (int i = 0; i < BLOCKS; ++i) load_weights(s * BLOCKS + i, s * BLOCKS + i);
            __builtin_amdgcn_sched_barrier(0);
        }
        int s = 0;
        for (; s + 2 < n_stages; s += 2) {
            run_stage(p0, yes, no, s);
            run_stage(p1, yes, no, s + 1);
        }
        run_stage(p0, no, no, s);
        run_stage(p1, no, yes, s + 1);
    }
    // A wavefront has 64 bytes of every row of the result.  The workgroup's 256 meet in LDS (where the tokens were), so that whole
    // lines are written, and through the L2 (store16_through).  Stored by each wavefront in pieces of 16 and 8 bytes a lane, the
    // layer of 256 experts of 7168 / 2048 took, uniform routing (Zipf(1.1)), 400 / 1000 tokens 938 / 1158 us (at 300 / 512 / 1000
    // tokens 470 / 616 / 856) and takes 919 / 1081 (456 / 595 / 844).
    constexpr int PITCH = 256 + 16;
    static_assert(64 * PITCH <= kW4Ring, "the rows fit the place of the tokens");
    __syncthreads();
    if (t.have) {
        float rs[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int r = t.row0 + 32 * b + c32 < t.row1 ? t.row0 + 32 * b + c32 : t.row0;
            rs[b] = a.row_scale[a.row_src ? a.row_src[r] : r];
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            int8_t* const to = t.lds + (32 * b + c32) * PITCH + wave * 64;
#pragma unroll
            for (int q = 0; q < 2; ++q) {  // runs q and q + 2: a gate run and its up run, or any two
                float g[4], up[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    g[j] = f[b][4 * q + j];
                    up[j] = f[b][8 + 4 * q + j];
                }
                if (p.bias) {
                    const v4f bg = *(const v4f*)(p.bias + (int64_t)t.e * a.N + run_channel(q));
                    const v4f bu = *(const v4f*)(p.bias + (int64_t)t.e * a.N + run_channel(q + 2));
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        g[j] = g[j] + bg[j];
                        up[j] = up[j] + bu[j];
                    }
                }
                if constexpr (EPI == EPI_DEQUANT) {
                    v4u16 o0, o1;
                    dequant_run_w4(a, g, up, rs[b], o0, o1);
                    *(v4u16*)(to + (8 * q + 4 * hi) * 2) = o0;
                    *(v4u16*)(to + (8 * (q + 2) + 4 * hi) * 2) = o1;
                } else {
                    *(v4f*)(to + (8 * q + 4 * hi) * 4) = swiglu_run_w4(a, g, up, rs[b]);
                }
            }
        }
    }
    __syncthreads();
    // piece i of 16 bytes: row i / 16, wavefront (i / 4) % 4
    const int units = (a.N >> 5) - t.first < 4 ? (a.N >> 5) - t.first : 4;
    int8_t* const result = EPI == EPI_DEQUANT ? (int8_t*)(a.out + t.first * 32) : (int8_t*)(a.y + t.first * 16);
    const int64_t pitch = (int64_t)a.N * 2;  // of a row of N 16-bit or N / 2 fp32 values
    const int rows = t.row1 - t.row0 < 32 * NB ? t.row1 - t.row0 : 32 * NB;
    for (int i = threadIdx.x; i < rows * 16; i += 256) {
        const int r = i >> 4, c = i & 15;
        if ((c >> 2) < units) store16_through(result + (t.row0 + r) * pitch + c * 16, *(const v4i*)(t.lds + r * PITCH + c * 16));
    }
}

// LDS_SCALES: the group scales of the wavefront's channels are in LDS
template <int EPI, bool LDS_SCALES>
__global__ __launch_bounds__(256, LDS_SCALES ? 4 : 3) void gmm_w4_stream_kernel(W4Args p)
{
    const GmmArgs& a = p.g;
    extern __shared__ __attribute__((aligned(16))) int8_t w4_lds[];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int NB = a.N >> 5, KB64 = a.K >> 6;
    // workgroup = (chunk, four neighbouring units of 32 channels); a wavefront past the last unit still stages tokens
    const int quads = (NB + 3) >> 2;
    const int chunk = (int)(blockIdx.x / quads);
    const int u_raw = (int)(blockIdx.x % quads) * 4 + wave;
    W4Unit t;
    t.lds = w4_lds;
    t.have = u_raw < NB;
    t.u = t.have ? u_raw : 0;
    t.first = u_raw - wave;
    int e, row0, row1;  // (rows are fewer than 2^31)
    bool single;
    if (p.tm.count) {
        if (chunk >= p.tm.count[0]) return;
        e = p.tm.expert[chunk];
        row0 = p.tm.row_begin[chunk];
        row1 = p.tm.row_end[chunk];
        single = (e & kOnlyTile) != 0;
        e &= ~kOnlyTile;
    } else {
        int64_t first_row, end_row;
        if (!find_chunk(a.gl, a.gl_type, a.E, chunk, kW4Chunk, lane, e, first_row, end_row, single)) return;
        row0 = (int)first_row;
        row1 = (int)(end_row < a.R ? end_row : a.R);
    }
    t.e = __builtin_amdgcn_readfirstlane(e);
    t.row0 = __builtin_amdgcn_readfirstlane(row0);
    row1 = __builtin_amdgcn_readfirstlane(row1);
    single = __builtin_amdgcn_readfirstlane((int)single);
    t.row1 = row1 < a.R ? row1 : (int)a.R;
    if (t.row1 <= t.row0) return;

    // lane l of an MFMA operand: channel l % 32 of the unit, K half l / 32
    const int c32 = lane & 31, hi = lane >> 5;
    const int tile = EPI == EPI_SWIGLU ? (t.u >> 1) + (c32 >= 16 ? NB >> 1 : 0) : t.u;
    const int chunk16 = EPI == EPI_SWIGLU ? hi * 32 + (t.u & 1) * 16 + (c32 & 15) : lane;
    t.w = p.w4 + (((int64_t)t.e * NB + tile) * KB64) * 1024 + chunk16 * 16;

    // The scales sit in LDS, loaded once up front: the K loop then has no load whose result is needed at once.
    // Kept there as scale / 16: the sixteen of the accumulators then cancels in the product, bit for bit as long as the
    // quotient is exact; a wavefront with a scale so small that it is not shifts its accumulators instead.
    const int n_groups = a.K / p.group;
    t.gscale = p.gscale + (int64_t)t.e * n_groups * a.N;
    float* ss = (float*)(w4_lds + kW4Ring) + wave * n_groups * 32;
    t.scales = ss;
    t.shift = !LDS_SCALES;
    if constexpr (LDS_SCALES) {
        const float* gs = t.gscale + (EPI == EPI_SWIGLU ? (c32 >= 16 ? a.N >> 1 : 0) + t.u * 16 + (c32 & 15) : t.u * 32 + c32);
        bool inexact = false;
        for (int g0 = 0; g0 < n_groups; g0 += 16) {  // eight loads in flight at a time
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int g = g0 + 2 * j + hi;
                v[j] = gs[(int64_t)(g < n_groups ? g : n_groups - 1) * a.N];
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int g = g0 + 2 * j + hi;
                if (g < n_groups) ss[g * 32 + c32] = v[j] * 0.0625f;
                inexact |= (v[j] * 0.0625f) * 16.0f != v[j];
            }
        }
        t.shift = __ballot(inexact) != 0;
        if (t.shift)
            for (int g = hi; g < n_groups; g += 2) ss[g * 32 + c32] = gs[(int64_t)g * a.N];
    }

    // Tokens: a load copies 16 rows x 64 values of a K block, the 16-byte piece c of row r to place c ^ (r / 4) % 4 of the
    // row's 64 bytes: sixteen rows at one piece fall into sixteen different bank groups.
    const bool two = t.row0 + 32 < t.row1;  // the second block of 32 rows holds some
    const int rows = t.row1 - t.row0;
    int64_t xo[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = (two ? wave : i) * 16 + (lane >> 2);
        const int lrow = r < rows ? r : rows - 1;  // rows past the chunk's end repeat its last row (never stored)
        // the row's values lie in its token's row, or in the row itself
        xo[i] = (int64_t)(a.row_src ? a.row_src[t.row0 + lrow] : lrow) * a.K + (((lane & 3) ^ ((r >> 2) & 3)) * 16);
    }
    const int8_t* xb = a.row_src ? a.x : a.x + (int64_t)t.row0 * a.K;
    // Buffer loads, whose offsets have 32 bits: a global load to LDS counts as a flat access, behind which the compiler waits
    // for every load in flight.  A chunk with rows further away than that copies them through registers.
    const bool far = __ballot((xo[0] > xo[1] ? xo[0] : xo[1]) + a.K > 0xffffffffll) != 0;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)xb, 0, -1, 0x00027000);
    if (two) {
        if (far) w4_chunk_body<EPI, LDS_SCALES, 2, false, true>(p, t, xr, xb, xo);
        else if (single) w4_chunk_body<EPI, LDS_SCALES, 2, true, false>(p, t, xr, xb, xo);
        else w4_chunk_body<EPI, LDS_SCALES, 2, false, false>(p, t, xr, xb, xo);
    } else {
        if (far) w4_chunk_body<EPI, LDS_SCALES, 1, false, true>(p, t, xr, xb, xo);
        else if (single) w4_chunk_body<EPI, LDS_SCALES, 1, true, false>(p, t, xr, xb, xo);
        else w4_chunk_body<EPI, LDS_SCALES, 1, false, false>(p, t, xr, xb, xo);
    }
}

// ------------------------------------------------------------------ decode batches, pair order
// The same product for at most 40 tokens (see w4_pairs_supported) whose ids come straight from the gate: an expert has
// one to a few rows, so nothing is sorted (a row belongs to its pair throughout, as in gmm_stream_kernel's pair order),
// nothing is staged and no wavefront waits for another one inside the K loop.  One wavefront per 32 channels (SwiGLU: 16 of the gate
// and the 16 of the up projection that belong to them) over the whole K range (the fp32 sum over the scale groups has one
// fixed order); tokens are the 16 columns of v_mfma_i32_16x16x64_i8, one or two times.  HBM-bound.
// DeepSeek-V3 shape, us a layer call with 64 channels per wavefront, two wavefronts per SIMD / with 32, four: uniform
// routing, 1 / 4 / 8 / 16 / 24 tokens 57 / 136 / 230 / 385 / 501 against 50 / 127 / 217 / 362 / 468 (16 tokens: 2.2 GB at
// 6.1 TB/s); Zipf(1.1), 16 / 20 / 24 tokens 148 / 171 / 178 against 137 / 155 / 169.  A ring of 3 (six wavefronts), 4 (five),
// 5, 6, 7, 8, 10 or 14 (two) blocks, 1 and 16 tokens: 56 and 366, 53 and 362, 50 and 359, 50 and 360, 50 and 367, 51 and
// 367, 50 and 371, 54 and 391.  More than 16 rows under Zipf(1.1), 24 / 32 tokens: two blocks at a time 169 / 194, one
// after the other 183 / 213, the second block in workgroups of its own 185 / 207.
// An int4 tile (lane = channel l % 32, K half l / 32; low nibbles K 0..31, high nibbles K 32..63) becomes the operands of
// its two groups of 16 channels by one exchange: rows of 16 lanes 1 and 3 of the low-nibble register against rows 0 and 2
// of the high-nibble register (v_permlane16_swap) leave channels 0..15 in one register and 16..31 in the other, row r of
// either holding the K slice 0, 32, 16 or 48 + 0..15 for r = 0, 1, 2, 3.  The tokens are read in that order.
constexpr int kW4PairMax = 1024;
constexpr int kW4PairExperts = 2048;
constexpr int kW4PairRing = 6;     // K blocks of weights and tokens in flight per wavefront,
constexpr int kW4PairRing2 = 4;    // with two blocks of 16 rows: what 128 registers hold

__device__ __forceinline__ void w4_operands(v4i v, v4i& first, v4i& second)
{
    const v4i lo = nib_lo(v), hi = nib_hi(v);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const auto r = __builtin_amdgcn_permlane16_swap((unsigned)lo[d], (unsigned)hi[d], false, false);
        first[d] = (int)r[0];
        second[d] = (int)r[1];
    }
}

// The expert of a slot (the slot-th one that has pairs) and, in plist, its pairs in ascending order; every thread of the
// workgroup calls it and gets the same answer, -1 where there are fewer such experts.  See gmm_stream_kernel.
__device__ __forceinline__ int w4_slot_pairs(const GmmArgs& a, int slot, int wave, int lane, uint32_t* pmap,
                                             int32_t* pcount, uint16_t* plist, int& rows)
{
    const int Q = (((int)a.R + 255) >> 8) << 6;
    int pid[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int f = wave * Q + c * 64 + lane;
        pid[c] = (c * 64 < Q && f < (int)a.R) ? a.pair_ids[f] : -1;
    }
    if (threadIdx.x < kW4PairExperts / 32) pmap[threadIdx.x] = 0u;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (pid[c] >= 0 && pid[c] < a.E) atomicOr(&pmap[pid[c] >> 5], 1u << (pid[c] & 31));
    __syncthreads();
    const uint32_t bits = pmap[lane];
    const int cnt = __popc(bits);
    const int incl = wave_scan_inclusive_i32(cnt);
    const bool has = slot >= incl - cnt && slot < incl;
    const unsigned long long holder = __ballot(has);
    if (holder == 0ull) return -1;
    uint32_t t = bits;
    for (int i = has ? slot - (incl - cnt) : 0; i > 0; --i) t &= t - 1;
    const int e = __builtin_amdgcn_readlane(lane * 32 + (t ? __builtin_ctz(t) : 0), __builtin_ctzll(holder));
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    bool mine[4];
    int n = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        mine[c] = pid[c] == e;
        n += __popcll(__ballot(mine[c]));
    }
    if (lane == 0) pcount[wave] = n;
    __syncthreads();
    int base = 0;
    rows = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        if (w < wave) base += pcount[w];
        rows += pcount[w];
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const unsigned long long m = __ballot(mine[c]);
        if (mine[c]) plist[base + __popcll(m & below)] = (uint16_t)(wave * Q + c * 64 + lane);
        base += __popcll(m);
    }
    __syncthreads();
    return e;
}

// Workgroup = (slot, four groups of 32 channels).
template <int EPI>
__global__ __launch_bounds__(256, 4) void gmm_w4_pairs_kernel(W4Args p)
{
    const GmmArgs& a = p.g;
    __shared__ uint16_t plist[kW4PairMax];       // the expert's pairs, ascending
    __shared__ int32_t pcount[4];
    __shared__ uint32_t pmap[kW4PairExperts / 32];  // one bit per expert that has pairs
    __shared__ float Ss[4][kW4LdsGroups * 32];      // group scales of every wavefront's channels
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int NB = a.N >> 5, KB64 = a.K >> 6;
    const int quads = (NB + 3) >> 2;
    const int u_raw = (int)(blockIdx.x % quads) * 4 + wave;
    const bool have = u_raw < NB;
    const int u = have ? u_raw : 0;
    int rows;
    const int e = w4_slot_pairs(a, (int)(blockIdx.x / quads), wave, lane, pmap, pcount, plist, rows);
    if (e < 0 || !have) return;  // no barrier behind this one

    const int c32 = lane & 31, hi = lane >> 5;
    const int tile = EPI == EPI_SWIGLU ? (u >> 1) + (c32 >= 16 ? NB >> 1 : 0) : u;
    const int chunk16 = EPI == EPI_SWIGLU ? hi * 32 + (u & 1) * 16 + (c32 & 15) : lane;
    const uint8_t* wp = p.w4 + (((int64_t)e * NB + tile) * KB64) * 1024 + chunk16 * 16;
    const int n_groups = a.K / p.group, steps_per_group = p.group >> 6;
    const int tok = lane & 15, r16 = lane >> 4;
    const int slice = 16 * ((r16 >> 1) + 2 * (r16 & 1));  // K 0, 32, 16, 48 for rows 0..3
    // one pass over the weights for NT blocks of 16 rows, D blocks of K in flight
    auto pass = [&](auto blocks, auto depth, int first) {
        constexpr int NT = decltype(blocks)::value, D = decltype(depth)::value;
        v4i w[D], x[D][NT];
        bool valid[NT];
        int row[NT];  // where the row's result goes
        const int8_t* xp[NT];
        float rs[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            valid[n] = first + 16 * n + tok < rows;
            row[n] = plist[valid[n] ? first + 16 * n + tok : 0];
            const int src = a.pair_gather ? row[n] / a.pair_k : row[n];
            xp[n] = a.x + (int64_t)src * a.K + slice;
            rs[n] = a.row_scale[src];
        }
        auto request = [&](int s, int kb) {
            const int k = kb < KB64 ? kb : KB64 - 1;  // past the end: a valid block that is never used
            w[s] = gload16_nt(wp + (int64_t)k * 1024);
#pragma unroll
            for (int n = 0; n < NT; ++n) x[s][n] = *(const v4i*)(xp[n] + k * 64);
        };
#pragma unroll
        for (int i = 0; i < D; ++i) request(i, i);
        if (first == 0) {
            const float* gs = p.gscale + (int64_t)e * n_groups * a.N +
                              (EPI == EPI_SWIGLU ? (c32 >= 16 ? a.N >> 1 : 0) + u * 16 + (c32 & 15) : u * 32 + c32);
            for (int g0 = 0; g0 < n_groups; g0 += 16) {  // eight loads in flight at a time
                float v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int g = g0 + 2 * j + hi;
                    v[j] = gs[(int64_t)(g < n_groups ? g : n_groups - 1) * a.N];
                }
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (g0 + 2 * j + hi < n_groups) Ss[wave][(g0 + 2 * j + hi) * 32 + c32] = v[j];
            }
            wave_lds_order();
        }
        v4i c[NT][2];  // 16 channels each
        float f[NT][2][4];
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                c[n][h] = (v4i){0, 0, 0, 0};
#pragma unroll
                for (int j = 0; j < 4; ++j) f[n][h][j] = 0.0f;
            }
        int in_group = 0, grp = 0;
        auto step = [&](int s, int kb) {  // s = kb % D, compile time
            v4i lo, up;
            w4_operands(w[s], lo, up);
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                c[n][0] = mfma_i8_16(lo, x[s][n], c[n][0]);
                c[n][1] = mfma_i8_16(up, x[s][n], c[n][1]);
            }
            request(s, kb + D);
            if (++in_group == steps_per_group) {  // f += float(acc / 16) * scale[e, grp, channel]
                const float* sl = &Ss[wave][grp * 32 + 4 * r16];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const v4f sc = *(const v4f*)(sl + 16 * h);
#pragma unroll
                    for (int n = 0; n < NT; ++n) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) f[n][h][j] = f[n][h][j] + (float)(c[n][h][j] >> 4) * sc[j];
                        c[n][h] = (v4i){0, 0, 0, 0};
                    }
                }
                in_group = 0;
                ++grp;
            }
        };
        const int kb_full = (KB64 / D) * D;
        for (int kb = 0; kb < kb_full; kb += D) {
#pragma unroll
            for (int i = 0; i < D; ++i) step(i, kb + i);
        }
#pragma unroll
        for (int i = 0; i < D - 1; ++i)
            if (kb_full + i < KB64) step(i, kb_full + i);
        const int c0 = EPI == EPI_SWIGLU ? u * 16 + 4 * r16 : u * 32 + 4 * r16;
#pragma unroll
        for (int n = 0; n < NT; ++n)
            epilogue_run_w4<EPI>(a, row[n], valid[n], c0, EPI == EPI_SWIGLU ? c0 + (a.N >> 1) : c0 + 16, f[n][0], f[n][1],
                                 rs[n]);
    };
    int first = 0;
    for (; rows - first > 16; first += 32)
        pass(std::integral_constant<int, 2>{}, std::integral_constant<int, kW4PairRing2>{}, first);
    if (first < rows) pass(std::integral_constant<int, 1>{}, std::integral_constant<int, kW4PairRing>{}, first);
}

// workgroups: an upper bound of the number of 64-row chunks (known on the host without reading the group
// list) times the groups of four units of 32 channels
static int64_t w4_blocks(int64_t rows, int num_experts, int64_t n)
{
    // a chunk has at least one row: a decode batch of a few rows has a few chunks, not one per expert (a workgroup
    // that only finds its chunk missing still costs its dispatch)
    const int64_t by_experts = rows / kW4Chunk + num_experts;
    return (rows < by_experts ? rows : by_experts) * ((n / 32 + 3) / 4);
}

template <int EPI>
static bool launch_w4(const W4Args& p, int64_t blocks, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1)
{
    const int64_t n_groups = p.g.K / p.group;
    const bool lds_scales = w4_scales_in_lds(n_groups, blocks);
    const int lds = lds_scales ? (int)w4_lds_bytes(n_groups) : kW4Ring;
    auto kernel = lds_scales ? gmm_w4_stream_kernel<EPI, true> : gmm_w4_stream_kernel<EPI, false>;
    static OncePerDevice once;
    if (lds_scales && !allow_dynamic_lds(once, (const void*)gmm_w4_stream_kernel<EPI, true>, kW4LdsMax)) return false;
    if (ev0 && ev1)
        hipExtLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), lds, st, ev0, ev1, 0, p);
    else
        hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), lds, st, p);
    return true;
}

static int check_w4(const void* x, const void* w, const float* scale, const int64_t* gl, int gl_type, int64_t rows,
                    int64_t k, int64_t n, int E, int64_t group)
{
    if (rows < 0 || k <= 0 || n <= 0 || E <= 0 || group <= 0) return MOE355_E_ARG;
    if (gl_type != MOE355_GL_CUMSUM && gl_type != MOE355_GL_COUNT) return MOE355_E_ARG;
    if (n % 64 != 0 || k % 64 != 0 || group % 64 != 0 || k % group != 0) return MOE355_E_SHAPE;
    if (rows >= 0x7fffffffLL || n >= 0x7fffffffLL || k >= 0x7fffffffLL) return MOE355_E_SHAPE;
    if (rows > 0 && (!x || !w || !scale || !gl)) return MOE355_E_ARG;
    if (((uintptr_t)x & 15) || ((uintptr_t)w & 15) || ((uintptr_t)scale & 15)) return MOE355_E_SHAPE;
    return MOE355_OK;
}

}  // namespace moe355

using namespace moe355;

extern "C" int moe355_format_cast_nz_int4(const uint8_t* w, int source, int64_t num_experts, int64_t n, int64_t k,
                                          uint8_t* out, void* stream)
{
    if (num_experts <= 0 || n <= 0 || k <= 0 || !w || !out) return MOE355_E_ARG;
    if (source != 0 && source != 1) return MOE355_E_ARG;
    if (n % 32 != 0 || k % 64 != 0) return MOE355_E_SHAPE;
    if ((uintptr_t)out & 15) return MOE355_E_SHAPE;
    const int64_t total = num_experts * n * k / 32;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipStream_t st = (hipStream_t)stream;
    if (source == 0)
        hipLaunchKernelGGL(format_cast_nz_int4_kernel<0>, dim3((unsigned)blocks), dim3(256), 0, st, w, num_experts, n, k,
                           out);
    else
        hipLaunchKernelGGL(format_cast_nz_int4_kernel<1>, dim3((unsigned)blocks), dim3(256), 0, st, w, num_experts, n, k,
                           out);
    return launch_status();
}

extern "C" int moe355_w4_offset_correction(const uint8_t* weight_nz4, const float* weight_scale, int64_t group_size,
                                           int num_experts, int64_t n, int64_t k, float* corr, void* stream)
{
    if (num_experts <= 0 || n <= 0 || k <= 0 || group_size <= 0 || !weight_nz4 || !weight_scale || !corr)
        return MOE355_E_ARG;
    if (n % 32 != 0 || k % 64 != 0 || group_size % 64 != 0 || k % group_size != 0) return MOE355_E_SHAPE;
    if ((uintptr_t)weight_nz4 & 15) return MOE355_E_SHAPE;
    const int64_t tiles = (int64_t)num_experts * (n / 32);
    hipLaunchKernelGGL(w4_offset_correction_kernel, dim3((unsigned)((tiles + 3) / 4)), dim3(256), 0,
                       (hipStream_t)stream, weight_nz4, weight_scale, num_experts, (int)n, (int)k, (int)group_size,
                       corr);
    return launch_status();
}

TileSpec moe355::w4_chunk_spec(int64_t rows, int num_experts, void* workspace)
{
    TileSpec t = tile_spec(rows, num_experts, kW4Chunk, workspace);
    t.flag_only = 1;
    return t;
}

int moe355::gmm1_w4_impl(const int8_t* x, const uint8_t* weight_nz4, const float* weight_scale, int64_t group_size,
                         const float* bias, const float* x_scale, const int64_t* group_list, int group_list_type,
                         int64_t rows, int64_t k, int64_t n, int num_experts, float swiglu_limit, int8_t* out,
                         float* out_scale, void* workspace, size_t workspace_bytes, void* stream,
                         const int32_t* row_src, const TileMap* chunks)
{
    int rc = check_w4(x, weight_nz4, weight_scale, group_list, group_list_type, rows, k, n, num_experts, group_size);
    if (rc != MOE355_OK) return rc;
    if (rows == 0) return MOE355_OK;
    if (!x_scale || !out || !out_scale) return MOE355_E_ARG;
    if (((uintptr_t)bias & 15) || ((uintptr_t)out & 3)) return MOE355_E_SHAPE;
    const size_t ybytes = ((size_t)rows * (size_t)(n / 2) * 4 + 255) & ~(size_t)255;
    if (!workspace || ((uintptr_t)workspace & 255) || workspace_bytes < ybytes) return MOE355_E_WORKSPACE;
    hipStream_t st = (hipStream_t)stream;
    W4Args p = {};
    p.g.x = x;
    p.g.gl = group_list;
    p.g.gl_type = group_list_type;
    p.g.R = rows;
    p.g.K = (int)k;
    p.g.N = (int)n;
    p.g.E = num_experts;
    p.g.row_scale = x_scale;
    p.g.row_src = row_src;
    p.g.limit = swiglu_limit;
    p.g.y = (float*)workspace;
    p.w4 = weight_nz4;
    p.gscale = weight_scale;
    p.bias = bias;
    p.group = (int)group_size;
    if (chunks) p.tm = *chunks;
    const int64_t blocks = w4_blocks(rows, num_experts, n);
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    take_profile_events(ev0, ev1);
    if (!launch_w4<EPI_SWIGLU>(p, blocks, st, ev0, ev1)) return MOE355_E_LAUNCH;
    launch_swiglu_requant(p.g.y, group_list, group_list_type, num_experts, rows, (int)(n / 2), out, out_scale, st);
    return launch_status();
}

extern "C" int moe355_gmm1_swiglu_quant_w4(const int8_t* x, const uint8_t* weight_nz4, const float* weight_scale,
                                           int64_t group_size, const float* bias, const float* x_scale,
                                           const int64_t* group_list, int group_list_type, int64_t rows, int64_t k,
                                           int64_t n, int num_experts, float swiglu_limit, int8_t* out,
                                           float* out_scale, void* workspace, size_t workspace_bytes, void* stream)
{
    return gmm1_w4_impl(x, weight_nz4, weight_scale, group_size, bias, x_scale, group_list, group_list_type, rows, k,
                        n, num_experts, swiglu_limit, out, out_scale, workspace, workspace_bytes, stream, nullptr, nullptr);
}

extern "C" int moe355_gmm1_swiglu_quant_w4_gather(const int8_t* x, const float* x_scale, const int32_t* row_token,
                                                  const uint8_t* weight_nz4, const float* weight_scale,
                                                  int64_t group_size, const float* bias, const int64_t* group_list,
                                                  int group_list_type, int64_t rows, int64_t k, int64_t n,
                                                  int num_experts, float swiglu_limit, int8_t* out, float* out_scale,
                                                  void* workspace, size_t workspace_bytes, void* stream)
{
    if (rows > 0 && !row_token) return MOE355_E_ARG;
    return gmm1_w4_impl(x, weight_nz4, weight_scale, group_size, bias, x_scale, group_list, group_list_type, rows, k,
                        n, num_experts, swiglu_limit, out, out_scale, workspace, workspace_bytes, stream, row_token, nullptr);
}

// Up to 24 tokens; 32, two blocks of 16 rows, with experts under 16 MiB, where the launches of a sorted layer cost as much
// as a few more bytes; 40 under 5 MiB, where they cost more than a second reading of the experts with more than 32 rows.  Beyond,
// a skewed batch waits for its hot experts; the host cannot know.  Pair order / sorted, us a call.  DeepSeek-V3 shape (22 MB),
// 20 / 24 / 32 / 48 tokens: uniform routing 423 / 468 / 548 / 685 against 442 / 493 / 571 / 709, Zipf(0.8) 205 / 219 / 244 / 308
// against 216 / 231 / 248 / 291, Zipf(1.1) 155 / 169 / 194 / 241 against 162 / 172 / 190 / 207, Zipf(1.4) 127 / 140 / 159 / 225
// against 134 / 141 / 148 / 171.  28 / 32 tokens: 128 experts of 2.4 MB uniform 63 / 65 against 70 / 72, Zipf(1.1) 41 / 43
// against 43 / 44; of 9.4 MB 173 / 182 against 183 / 195, 91 / 100 against 93 / 98.  33 / 36 / 40 tokens, uniform (Zipf(1.1)):
//   0.8 MB (256 of 1024 / 512)   45 / 46 / 47    (30 / 34 / 36) against    53 / 55 / 56    (35 / 37 / 37)
//   2.2 MB (8 of 1024 / 1408)    25 / 26 / 27    (30 / 31 / 35) against    34 / 33 / 33    (33 / 34 / 36)
//   2.4 MB (128 of 2048 / 768)   65 / 66 / 66    (46 / 51 / 52) against    73 / 74 / 75    (46 / 48 / 49)
//   4.3 MB (64 of 2048 / 1408)   62 / 63 / 63    (48 / 59 / 60) against    73 / 73 / 73    (51 / 56 / 56)
//   4.7 MB (64 of 2048 / 1536)   65 / 66 / 67    (58 / 65 / 68) against    74 / 75 / 75    (57 / 60 / 60)
//   6.3 MB (128 of 4096 / 1024) 134 / 136 / 138  (80 / 92 / 93) against   144 / 146 / 147  (75 / 78 / 79)
//   7.9 MB (64 of 5120 / 1024)   96 / 97 / 98    (73 / 92 / 94) against   103 / 105 / 105  (65 / 73 / 75)
bool moe355::w4_pairs_supported(int64_t num_tokens, int top_k, int num_experts, int64_t hidden, int64_t intermediate,
                                int64_t group13, int64_t group2)
{
    const int64_t expert = hidden * intermediate * 3 / 2;
    const int64_t most = expert < (5 << 20) ? 40 : expert < (16 << 20) ? 32 : 24;
    return num_tokens > 0 && num_tokens <= most && num_tokens * top_k <= kW4PairMax && num_experts <= kW4PairExperts &&
           group13 > 0 && group2 > 0 && hidden / group13 <= kW4LdsGroups && intermediate / group2 <= kW4LdsGroups;
}

// one GEMM in pair order: the gate_up one (y set: fp32 SwiGLU values, rows re-quantised into out) or the down one
static W4Args w4_pair_args(const int8_t* x, const float* x_scale, const int32_t* topk_ids, int64_t num_tokens, int top_k,
                           const uint8_t* w, const float* scale, int64_t group, int64_t k, int64_t n, int num_experts)
{
    W4Args p = {};
    p.g.x = x;
    p.g.R = num_tokens * top_k;
    p.g.K = (int)k;
    p.g.N = (int)n;
    p.g.E = num_experts;
    p.g.row_scale = x_scale;
    p.g.pair_ids = topk_ids;
    p.g.pair_k = top_k;
    p.w4 = w;
    p.gscale = scale;
    p.group = (int)group;
    return p;
}

template <int EPI>
static void launch_w4_pairs(const W4Args& p, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1)
{
    const int64_t slots = p.g.R < (int64_t)p.g.E ? p.g.R : (int64_t)p.g.E;
    auto kernel = gmm_w4_pairs_kernel<EPI>;
    const dim3 grid((unsigned)(slots * ((p.g.N / 32 + 3) / 4)));
    if (ev0 || ev1)
        hipExtLaunchKernelGGL(kernel, grid, dim3(256), 0, st, ev0, ev1, 0, p);
    else
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, p);
}

int moe355::gmm1_w4_pairs(const int8_t* x, const float* x_scale, const int32_t* topk_ids, int64_t num_tokens, int top_k,
                          const uint8_t* w, const float* scale, int64_t group, int64_t k, int64_t n, int num_experts,
                          float swiglu_limit, float* y, int8_t* out, float* out_scale, hipStream_t st)
{
    if (!x || !x_scale || !topk_ids || !w || !scale || !y || !out || !out_scale) return MOE355_E_ARG;
    if (n % 64 != 0 || k % 64 != 0 || group % 64 != 0 || k % group != 0) return MOE355_E_SHAPE;
    if (((uintptr_t)x & 15) || ((uintptr_t)w & 15) || ((uintptr_t)scale & 15) || ((uintptr_t)y & 15)) return MOE355_E_SHAPE;
    W4Args p = w4_pair_args(x, x_scale, topk_ids, num_tokens, top_k, w, scale, group, k, n, num_experts);
    p.g.pair_gather = 1;
    p.g.limit = swiglu_limit;
    p.g.y = y;
    hipEvent_t ev0, ev1;
    take_profile_events(ev0, ev1);
    launch_w4_pairs<EPI_SWIGLU>(p, st, ev0, ev1);
    launch_swiglu_requant(y, nullptr, 0, num_experts, p.g.R, (int)(n / 2), out, out_scale, st);
    return launch_status();
}

int moe355::gmm2_w4_pairs(const int8_t* x, const float* x_scale, const int32_t* topk_ids, int64_t num_tokens, int top_k,
                          const uint8_t* w, const float* scale, int64_t group, int64_t k, int64_t n, int num_experts,
                          void* out, int out_dtype, hipStream_t st)
{
    if (!x || !x_scale || !topk_ids || !w || !scale || !out) return MOE355_E_ARG;
    if (n % 64 != 0 || k % 64 != 0 || group % 64 != 0 || k % group != 0) return MOE355_E_SHAPE;
    if (((uintptr_t)x & 15) || ((uintptr_t)w & 15) || ((uintptr_t)scale & 15) || ((uintptr_t)out & 7)) return MOE355_E_SHAPE;
    W4Args p = w4_pair_args(x, x_scale, topk_ids, num_tokens, top_k, w, scale, group, k, n, num_experts);
    p.g.out = (uint16_t*)out;
    p.g.out_f16 = out_dtype == MOE355_DT_F16;
    launch_w4_pairs<EPI_DEQUANT>(p, st, nullptr, nullptr);
    return launch_status();
}

int moe355::gmm2_w4_impl(const int8_t* x, const uint8_t* weight_nz4, const float* scale, int64_t group_size,
                         const float* bias, const float* per_token_scale, const int64_t* group_list, int group_list_type,
                         int64_t rows, int64_t k, int64_t n, int num_experts, void* out, int out_dtype, void* stream,
                         const TileMap* chunks)
{
    int rc = check_w4(x, weight_nz4, scale, group_list, group_list_type, rows, k, n, num_experts, group_size);
    if (rc != MOE355_OK) return rc;
    if (out_dtype != MOE355_DT_BF16 && out_dtype != MOE355_DT_F16) return MOE355_E_UNSUPPORTED;
    if (rows == 0) return MOE355_OK;
    if (!per_token_scale || !out) return MOE355_E_ARG;
    if (((uintptr_t)bias & 15) || ((uintptr_t)out & 7)) return MOE355_E_SHAPE;
    W4Args p = {};
    p.g.x = x;
    p.g.gl = group_list;
    p.g.gl_type = group_list_type;
    p.g.R = rows;
    p.g.K = (int)k;
    p.g.N = (int)n;
    p.g.E = num_experts;
    p.g.row_scale = per_token_scale;
    p.g.out = (uint16_t*)out;
    p.g.out_f16 = out_dtype == MOE355_DT_F16;
    p.w4 = weight_nz4;
    p.gscale = scale;
    p.bias = bias;
    p.group = (int)group_size;
    if (chunks) p.tm = *chunks;
    const int64_t blocks = w4_blocks(rows, num_experts, n);
    if (!launch_w4<EPI_DEQUANT>(p, blocks, (hipStream_t)stream, nullptr, nullptr)) return MOE355_E_LAUNCH;
    return launch_status();
}

extern "C" int moe355_gmm2_dequant_w4(const int8_t* x, const uint8_t* weight_nz4, const float* scale,
                                      int64_t group_size, const float* bias, const float* per_token_scale,
                                      const int64_t* group_list, int group_list_type, int64_t rows, int64_t k,
                                      int64_t n, int num_experts, void* out, int out_dtype, void* stream)
{
    return gmm2_w4_impl(x, weight_nz4, scale, group_size, bias, per_token_scale, group_list, group_list_type, rows, k, n,
                        num_experts, out, out_dtype, stream, nullptr);
}
