// Grouped int8 down product for many rows per expert and a short K (the width of an expert): the tokens of a 128-row tile
// stay in LDS for the whole of K.
//
// A workgroup of eight wavefronts, one per compute unit, takes 128 rows x 1024 channels.  It copies the rows' K values to LDS
// once (LDS-direct loads, K <= 896) and meets at one barrier; from there on every wavefront walks alone: 64 channels at a
// time, their weights straight into registers two K blocks ahead, refilled in place and across the seam to its next 64
// channels, so that they are on their way while the first ones' results go out.  The 128-row tiles of gmm_tiled.hip load the
// tokens again for every 256 channels and meet twice in every K block of 64; with 12 K blocks their start and their
// epilogue took half of the time.  128 experts of 512 rows, 768 / 2048: 117 us alone and 148 to 151 back to back against 176
// and 174 (268 MB of results leave behind either: 520 MB that have to come and go in all).  Ordinary / non-temporal
// stores 158 / 148 us back to back; written through the L2, as now, a layer of 8192 tokens takes 0.993 of the time with the latter.
// Four K blocks in flight: spills, 180 us.
#include <hip/hip_ext.h>

#include <type_traits>

#include "gmm_common.h"
#include "gmm_tiled.h"
#include "tile_map.h"

namespace moe355 {

constexpr int kResWaves = 8;
constexpr int kResRowB = 128 + 16;                      // epilogue patch: bytes per token row (padded)
constexpr int kResPatch = 32 * kResRowB;                // one wavefront's patch
constexpr int kResLdsBytes = 163840;

// LDS: tokens, patches, 128 token scales, the channel scales of the workgroup's channels
static int resident_lds(int64_t K, int group_span) { return (int)(128 * K) + kResWaves * kResPatch + 128 * 4 + group_span * 64 * 4; }

#define MOE355_GPTR(p) ((const __attribute__((address_space(1))) void*)(p))
#define MOE355_LPTR(p) ((__attribute__((address_space(3))) void*)(p))

// Rows [row0, row_end) of expert e (at most 32 * NBLK) x the channel groups (64 channels) g0 .. g0 + span - 1: wavefront w
// takes groups g0 + w, g0 + w + 8 (at most two).  The rows of a down product lie in x one after the other.  S: K blocks of
// 64 values whose weights are in flight per wavefront; K is a multiple of 64 * S and holds at least two such pieces.
// EVEN: every wavefront has two groups.
template <int NBLK, int S, bool F16, bool EVEN>
__device__ __forceinline__ void resident_body(const GmmArgs& a, int e, int64_t row0, int64_t row_end, int g0, int span,
                                              int8_t* lds)
{
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int tok = lane & 15, quarter = lane >> 4;
    const int K = a.K, KB = K >> 5;
    const int groups = a.N >> 6;
    int8_t* patch = lds + 128 * K + wave * kResPatch;
    float* rs_l = (float*)(lds + 128 * K + kResWaves * kResPatch);
    float* cs_l = rs_l + 128;

    const int8_t* we = expert_weights(a, e);
    const float* cs = expert_scales(a, e);
    // uniform pointers throughout: base in scalar registers, the lane's part is one register for all of them
    auto tile_of = [&](int g) { return we + (int64_t)g * KB * 2048; };  // its two storage tiles follow each other

    // ---- tokens: a load covers 8 rows x 128 K bytes; piece u = (K / 128, row / 8), wavefront u % 8.  The 16-byte chunk c of
    // row r lies in slot c ^ (r / 2) % 8 of its 128 bytes: sixteen rows at one chunk fall into sixteen different bank groups.
    {
        const int r8 = lane >> 3;
        const int pieces = (K >> 7) * (NBLK * 4);
        for (int u = wave; u < pieces; u += kResWaves) {
            const int seg = u / (NBLK * 4), rp = u % (NBLK * 4);
            const int c = (lane & 7) ^ ((r8 >> 1) | ((rp & 1) << 2));
            int64_t r = row0 + rp * 8 + r8;
            if (r > row_end - 1) r = row_end - 1;  // rows past the expert's end repeat its last row (never stored)
            __builtin_amdgcn_global_load_lds(MOE355_GPTR(a.x + r * K + seg * 128 + c * 16), MOE355_LPTR(lds + u * 1024), 16, 0, 0);
        }
    }
    const int first_group = g0 + wave;
    const bool have0 = wave < span && first_group < groups;
    const bool have1 = wave + 8 < span && first_group + 8 < groups;
    const unsigned wl = weight_lane(lane);
    v4i A[S][4];
    const int8_t* p = tile_of(have0 ? first_group : 0);
    const int8_t* p_next = tile_of(have1 ? first_group + 8 : 0);
    auto load_step = [&](int s, const int8_t* w) {
#pragma unroll
        for (int t = 0; t < 4; ++t) A[s][t] = gload16(w + (t >> 1) * KB * 1024 + s * 2048 + (t & 1) * 256 + wl);
    };
#pragma unroll
    for (int s = 0; s < S; ++s) load_step(s, p);
    if (threadIdx.x < 128) {
        int64_t r = row0 + threadIdx.x;
        if (r > row_end - 1) r = row_end - 1;
        rs_l[threadIdx.x] = a.row_scale[r];
    }
    for (int i = threadIdx.x; i < span * 64; i += 64 * kResWaves)
        cs_l[i] = g0 * 64 + i < a.N ? cs[g0 * 64 + i] : 0.0f;
    // the compiler does not count LDS-direct loads against the LDS reads that consume them
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (!have0) return;  // no barrier behind this one

    int frag[2];  // of the two K blocks of 128 K bytes
#pragma unroll
    for (int q = 0; q < 2; ++q)
        frag[q] = (tok >> 3) * 1024 + (tok & 7) * 128 + (((q * 4 + quarter) ^ ((tok >> 1) & 7)) * 16);
    constexpr int SEG = NBLK * 4096;  // LDS bytes of 128 K values
    v4i fb[2][NBLK];                  // half of the tokens: fragments of 16 tokens x 64 K
    v4i acc[4][2 * NBLK];
    auto read_frag = [&](int half, int b, const int8_t* xb, int s) {
        fb[half][b] = *(const v4i*)(xb + frag[s & 1] + (s >> 1) * SEG + (half * NBLK + b) * 2048);
    };
    // S K blocks: the MFMAs of half the tokens, under them the operands of the other half; then the block's weight registers
    // are requested again, S blocks ahead (q: where those lie)
    auto steps = [&](auto first, auto load, const int8_t* xb, const int8_t* xb_next, const int8_t* q) {
        constexpr bool FIRST = decltype(first)::value, LOAD = decltype(load)::value;
#pragma unroll
        for (int s = 0; s < S; ++s) {
#pragma unroll
            for (int half = 0; half < 2; ++half) {
#pragma unroll
                for (int b = 0; b < NBLK; ++b) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        v4i& c = acc[t][half * NBLK + b];
                        c = mfma_i8_16(A[s][t], fb[half][b], FIRST && s == 0 ? (v4i){0} : c);
                    }
                    if (half == 0) read_frag(1, b, xb, s);
                    else if (s + 1 < S) read_frag(0, b, xb, s + 1);
                    else read_frag(0, b, xb_next, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if constexpr (LOAD) {
                load_step(s, q);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    const int64_t n_rows = row_end - row0 < 32 * NBLK ? row_end - row0 : 32 * NBLK;
    const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc((void*)(a.out + row0 * a.N), 0, (int)(n_rows * a.N * 2), 0x00027000);
    // Whole 128-byte row segments through the wavefront's own LDS patch (see tiled_epilogue_body).  The buffer's length cuts
    // the rows past the expert's end: every store is issued, so that the waits for the next group's weights, which are in
    // flight already, are exact.  Row and column are in the vector offset alone.  That is what the length is
    // compared with, where the scalar offset need not be; and behind a 16-byte store with a scalar offset the compiler lets the
    // next vector instruction write over the store's data, which gfx950 then stores (every other row's first four bytes were
    // the next store's address), while without one it waits for as long as the store takes its data.
    auto epilogue = [&](int g) {
        const float* sg = cs_l + (g - g0) * 64 + 4 * quarter;
        const int c16 = lane & 7, r8 = lane >> 3;
#pragma unroll
        for (int b = 0; b < NBLK; ++b) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float rs = rs_l[b * 32 + h * 16 + tok];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const v4f sc = *(const v4f*)(sg + 16 * t);
                    v4u16 o;
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        o[j] = f32_to_half<F16 ? MOE355_DT_F16 : MOE355_DT_BF16>(((float)acc[t][2 * b + h][j] * rs) * sc[j]);
                    *(v4u16*)(patch + (16 * h + tok) * kResRowB + (16 * t + 4 * quarter) * 2) = o;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            wave_lds_order();
            v4i t[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) t[i] = *(const v4i*)(patch + (r8 + 8 * i) * kResRowB + c16 * 16);
            wave_lds_order();
            int at = r8 * a.N * 2 + g * 128 + c16 * 16;
            asm volatile("" : "+v"(at));  // the sums below are made here: kept over the K loop they would cost 16 registers
#pragma unroll
            for (int i = 0; i < 4; ++i)
                __builtin_amdgcn_raw_buffer_store_b128(t[i], out, at + (b * 32 + 8 * i) * a.N * 2, 0, 16 /* sc1: see store16_through */);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
#pragma unroll
    for (int b = 0; b < NBLK; ++b) read_frag(0, b, lds, 0);
    const int n_pieces = KB / (2 * S);
    constexpr int XPIECE = S / 2 * SEG;
    const int8_t* xb;
    auto all_but_last = [&]() {
        steps(std::true_type{}, std::true_type{}, lds, lds + XPIECE, p + S * 2048);
        xb = lds + XPIECE;
        p += 2 * S * 2048;
        for (int i = 1; i + 1 < n_pieces; ++i) {
            steps(std::false_type{}, std::true_type{}, xb, xb + XPIECE, p);
            xb += XPIECE;
            p += S * 2048;
        }
    };
    if constexpr (EVEN) {
        all_but_last();
        steps(std::false_type{}, std::true_type{}, xb, lds, p_next);
        p = p_next;
        epilogue(first_group);
        all_but_last();
        steps(std::false_type{}, std::false_type{}, xb, lds, p);
        epilogue(first_group + 8);
    } else {
        for (int g = first_group; g < g0 + span && g < groups; g += kResWaves) {
            all_but_last();
            steps(std::false_type{}, std::true_type{}, xb, lds, p_next);  // (past the last group: weights that are never used)
            p = p_next;
            epilogue(g);
        }
    }
}

template <int S, bool F16, bool EVEN>
__global__ __launch_bounds__(512, 1) void gmm_resident_kernel(GmmArgs a, TileMap tm, int parts, int span)
{
    extern __shared__ __attribute__((aligned(16))) int8_t res_lds[];
    const int total = tm.count[0] * parts;
    const int per_xcd = (total + 7) / 8;
    const int slot = (int)(blockIdx.x / 8);
    const int item = (int)(blockIdx.x % 8) * per_xcd + slot;
    if (slot >= per_xcd || item >= total) return;
    const int mt = item / parts, part = item % parts;
    const int e = __builtin_amdgcn_readfirstlane(tm.expert[mt]);
    const int64_t row0 = tm.row_begin[mt];
    int64_t row_end = tm.row_end[mt];
    if (row_end > a.R) row_end = a.R;
    if (row0 >= row_end) return;
    const int64_t rows = row_end - row0;
    if (rows <= 64) resident_body<2, S, F16, EVEN>(a, e, row0, row_end, part * span, span, res_lds);
    else resident_body<4, S, F16, EVEN>(a, e, row0, row_end, part * span, span, res_lds);
}

// From 288 rows per expert on.  The layer on 128-row tiles / on these, us, 128 experts of 2048 / 768, eight slots, uniform
// routing (Zipf(1.1)): 192 rows 267.0 / 264.7, 200 (275.7 / 281.1), 256 330.0 / 331.7, 312 369.8 / 363.6, 344 (398.6 /
// 399.2), 500 544.7 / 527.9.  One workgroup per compute unit and 32 KiB of weights for 64 channels: an expert's last, short
// tile costs more than on the smaller tiles.
//
// The other lines, by the product alone, back to back, time of 128-row tiles = 1, uniform routing (Zipf(1.1)):
// - Places: a workgroup's wavefronts take one or two whole groups of 64 channels each, so 1280 channels fill 20 of 32 places.
//   K = 768, 128 experts of 512 rows, 1088 / 1152 / 1280 channels (0.53 to 0.63 of the places) 1.06 / 1.06 / 1.03 (1.05 / 1.05
//   / 1.04); 1408 / 1536 / 1792 / 2112 / 2304 / 2560 / 2880 (0.69 to 0.94) 0.93 / 0.94 / 0.94 / 0.90 / 0.90 / 0.92 / 0.87 (0.94
//   / 0.94 / 0.96 / 0.92 / 0.92 / 0.92 / 0.88); 2048 and 4096 (all) 0.85 and 0.90 (0.89 and 0.87).  K = 896 the same, K = 640
//   from 1408 on.
// - Below 1024 channels, one workgroup for a tile either way, nothing is won: 448 / 576 / 768 0.96 / 1.00 / 1.00 (1.05 / 1.04 /
//   1.02).
// - A short K has less to keep.  128 experts of 300 rows, 1536 / 2304 / 2560 channels at K = 512 0.95 / 0.98 / 0.96 (1.05 / 1.07
//   / 1.05), at K = 384 0.94 / 0.95 / 0.97 (1.02 / 1.05 / 1.05), 1024 at K = 512 and 512 rows 0.96 (1.08); 2880 at K = 512 / 384 /
//   256 0.93 / 0.91 / 0.90 (0.97 / 1.00 / 1.01; K = 256 at 512 rows 1.05); 2048 at K = 512 / 384 / 256 0.88 / 0.89 / 0.88 (1.02 / 1.01 / 0.84) and at 512
//   rows 0.89 / 0.88 / 0.89 (0.90 / 0.94 / 0.88).  And thousands of rows share an expert's weights in L2 as it is: K = 384, 2048
//   channels, 65536 rows of 4 / 8 / 16 / 32 experts 1.04 / 1.04 / 1.02 / 0.99 (1.05 / 1.05 / 1.04 / 1.01).
// - Rounds: workgroups for half a round more than the chip holds leave the rest of it idle.  2048 channels, 34000 rows of 4 / 8 /
//   16 experts (2.1 rounds) 1.09 / 1.06 / 1.05 at K = 896 and 1.01 / 1.04 / 1.04 at 640, 45000 rows (2.8) 0.89 / 0.88 / 0.90 and
//   0.88 / 0.86 / 0.87, 65536 (4.0 to 4.1) 0.98 / 0.98 / 0.94 and 0.95 / 0.96 / 0.95, 131072 0.79 / 0.81 / 0.82 and 0.92 / 0.83 /
//   0.82; 60 experts of 600 rows (2.4) 0.93 and 0.94.  With 1024 channels half as many workgroups do the same: 512 (two rounds
//   and the experts' short tiles), K = 640 / 768 / 896, 64 experts 0.89 / 0.93 / 0.93, 128 0.92 / 0.94 / 0.95.
bool resident_supported(const GmmArgs& a)
{
    if (a.K % 128 || a.K < 256 || a.N < 1024 || a.N > (1 << 20) || resident_lds(a.K, 16) > kResLdsBytes) return false;
    if (a.E < 2 || a.R / a.E < 288) return false;
    const int64_t groups = a.N / 64;
    const int64_t parts = (groups + 15) / 16;
    const int64_t places = ((groups + parts - 1) / parts + 7) / 8 * 8 * parts;
    if (a.K >= 640 ? 16 * groups < 11 * places
                   : a.N < 2048 || 16 * groups < (a.K >= 384 ? 15 : 16) * places || a.R / a.E >= 4096) return false;
    if (a.R / 128 * parts < 512) return false;
    const int64_t workgroups = (a.R / 128 + a.E / 2) * parts;  // half of the experts end in a tile that is hardly begun
    return parts == 1 || workgroups >= 200 * ((workgroups + 255) / 256);
}

// (the tile map is in the workspace)
bool launch_resident(const GmmArgs& a, void* workspace, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1)
{
    const TileSpec spec = tile_spec(a.R, a.E, 128, workspace);
    const int groups = a.N / 64;
    const int parts = (groups + 15) / 16;
    const int span = (groups + parts - 1) / parts;
    const int lds = resident_lds(a.K, 16);
    const int grid = (spec.max_tiles * parts + 7) / 8 * 8;
    auto launch = [&](auto kernel, OncePerDevice& once) {
        if (!allow_dynamic_lds(once, (const void*)kernel, kResLdsBytes)) return false;
        if (ev0 || ev1)
            hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(512), lds, st, ev0, ev1, 0, a, spec.tm, parts, span);
        else
            hipLaunchKernelGGL(kernel, dim3(grid), dim3(512), lds, st, a, spec.tm, parts, span);
        return true;
    };
    static OncePerDevice once[4];
    if (groups % 16 == 0) {
        if (a.out_f16) return launch(gmm_resident_kernel<2, true, true>, once[0]);
        return launch(gmm_resident_kernel<2, false, true>, once[1]);
    }
    if (a.out_f16) return launch(gmm_resident_kernel<2, true, false>, once[2]);
    return launch(gmm_resident_kernel<2, false, false>, once[3]);
}

}  // namespace moe355
