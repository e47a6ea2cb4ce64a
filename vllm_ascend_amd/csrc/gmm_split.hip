// Dense int8 GEMM for some dozens to some hundreds of rows (one expert owns them all: the shared expert of a mixed batch).
// Neither the weight stream nor the matrix units bound such a product but its depth: 256 rows x 4096 channels are 32 tiles
// of 128 x 256 for 256 compute units, each walking K = 7168 alone (100 us; the 29 MB of weights are 4 us).
//
// Workgroup = 64 rows of one expert x 64 channels (a gate tile and its up tile, or two neighbouring tiles), K cut over
// the four wavefronts: eight times as many workgroups as 128 x 256 tiles, each a quarter as long, and no operand is read
// by two wavefronts.  A wavefront owns the whole 64 x 64 accumulator of its quarter of K (64 registers).  Weights go
// straight into registers (a storage tile is an MFMA operand); tokens are loaded as whole 64-byte pieces of rows and turned
// into operands through a patch of LDS that belongs to the wavefront alone, so the K loop has no barrier.  In the end
// the wavefronts exchange quarters of the channels through LDS (int32: exact in any order) and each finishes one.
// DeepSeek-V3 layer with its shared expert in line, 128 / 256 tokens: 1767 / 1882 -> 1660 / 1738 us.  For grouped products of
// a small layer (K = 1024: four stages for a wavefront) the start and the end of a workgroup weigh more than what is in
// between; 64-row tiles were faster there (1024 tokens 59 against 49 us a layer).
#include <hip/hip_ext.h>

#include "gmm_tiled.h"

namespace moe355 {

constexpr int kSplitRing = 3;                        // stages of 64 K in registers: one in use, two in flight
constexpr int TB = 2;                                // blocks of 32 rows of a workgroup
constexpr int kSplitPatch = TB * 32 * 64;            // LDS: tokens of a stage, one wavefront
constexpr int kSplitSums = TB * 4 * 3 * 2 * 1024;    // ... what the wavefronts hand each other
constexpr int kSplitLds = 4 * kSplitPatch > kSplitSums ? 4 * kSplitPatch : kSplitSums;

template <int EPI>
__global__ __launch_bounds__(256, 2) void gmm_split_kernel(GmmArgs a, int units)
{
    __shared__ __attribute__((aligned(16))) int8_t lds[kSplitLds];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    // an XCD (workgroup number modulo 8) works on every eighth unit of all tiles: the rows of one expert that share a
    // unit's weights find them in its L2, where the tokens of all tiles have room as well
    const int upx = (units + 7) >> 3, in_xcd = (int)blockIdx.x >> 3;
    const int p = (in_xcd % upx) * 8 + ((int)blockIdx.x & 7), tile = in_xcd / upx;
    if (p >= units) return;
    const int64_t row0 = (int64_t)tile * 32 * TB, row_end = a.gl[0] < a.R ? a.gl[0] : a.R;
    if (row0 >= row_end) return;
    const int NB = a.N >> 5, KB = a.K >> 5;
    const int nb0 = EPI == EPI_SWIGLU ? p : 2 * p, nb1 = EPI == EPI_SWIGLU ? p + (NB >> 1) : 2 * p + 1;
    const int8_t* we = expert_weights(a, 0);
    const int8_t* w0 = we + (int64_t)nb0 * KB * 1024;
    const int8_t* w1 = we + (int64_t)nb1 * KB * 1024;
    const int K64 = a.K >> 6, k0 = K64 * wave / 4, n = K64 * (wave + 1) / 4 - k0;

    // token pieces of this lane: 16 bytes of row 16 i + lane / 4 (rows past the end repeat the last one).  Whole pointers:
    // row_src may name any token of an x larger than 4 GiB, however few rows there are, and 64-bit offsets that the loop adds to
    // x and clears past the last stage cost it 3 to 5 %.
    const int8_t* xr[2 * TB];
#pragma unroll
    for (int i = 0; i < 2 * TB; ++i) {
        int64_t r = row0 + 16 * i + (lane >> 2);
        if (r >= row_end) r = row_end - 1;
        xr[i] = a.x + (a.row_src ? (int64_t)a.row_src[r] : r) * a.K + (lane & 3) * 16;
    }
    // operands of the epilogue, in front of everything else in the queue of answers: this wavefront finishes the channels
    // of quarter `wave`
    const int tok = lane & 31, ch = quad_channel(wave, lane);
    float rs[TB];
    v4f cs0 = {0.0f, 0.0f, 0.0f, 0.0f}, cs1 = cs0;
#pragma unroll
    for (int b = 0; b < TB; ++b) {
        rs[b] = 0.0f;
        if constexpr (EPI != EPI_I32) {
            int64_t r = row0 + 32 * b + tok;
            if (r >= row_end) r = row_end - 1;
            rs[b] = a.row_scale[a.row_src ? (int64_t)a.row_src[r] : r];
        }
    }
    if constexpr (EPI != EPI_I32) {
        const float* cs = expert_scales(a, 0);
        cs0 = gload4f(cs + nb0 * 32 + ch);
        cs1 = gload4f(cs + nb1 * 32 + ch);
    }

    v4i w[kSplitRing][2][2], x[kSplitRing][2 * TB];
    // Requests past the wavefront's last stage go to the first bytes of the weights (all lanes to the same ones) and of the
    // rows: the loop stays free of conditional loads, so that every wait is for a stage and not for all that is in flight.
    auto request = [&](int it, int slot) {
        const bool in = it < n;
        const int64_t kw = in ? (int64_t)(k0 + it) * 2048 : 0;
        const uint32_t lo = in ? (uint32_t)lane * 16 : 0u;
        const int kx = in ? (k0 + it) * 64 : 0;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            w[slot][0][s] = gload16(w0 + kw + s * 1024 + lo);
            w[slot][1][s] = gload16(w1 + kw + s * 1024 + lo);
        }
#pragma unroll
        for (int i = 0; i < 2 * TB; ++i) x[slot][i] = gload16(xr[i] + kx);
    };
    // a row's four pieces of a stage lie rotated by half its number: neither the writes (two whole rows at a time) nor the
    // reads (one piece of eight rows) meet in a bank
    int8_t* patch = lds + wave * kSplitPatch;
    const int wr = (lane >> 2) * 64 + (((lane & 3) + (lane >> 3)) & 3) * 16;
    int rd[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) rd[s] = tok * 64 + ((2 * s + (lane >> 5) + (tok >> 1)) & 3) * 16;

    v16i c0[TB], c1[TB];
#pragma unroll
    for (int b = 0; b < TB; ++b) c0[b] = c1[b] = (v16i){0};
    auto step = [&](int it, int slot) {
        request(it + 2, (slot + 2) % kSplitRing);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2 * TB; ++i) *(v4i*)(patch + i * 1024 + wr) = x[slot][i];
        wave_lds_order();
        v4i t[2][TB];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int b = 0; b < TB; ++b) t[s][b] = *(const v4i*)(patch + b * 2048 + rd[s]);
        wave_lds_order();
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                c0[b] = mfma_i8(w[slot][0][s], t[s][b], c0[b]);
                c1[b] = mfma_i8(w[slot][1][s], t[s][b], c1[b]);
            }
        __builtin_amdgcn_sched_barrier(0);
    };
    request(0, 0);
    request(1, 1);
    __builtin_amdgcn_sched_barrier(0);
    const int whole = n / kSplitRing * kSplitRing;
    for (int it = 0; it < whole; it += kSplitRing) {
        step(it, 0);
        step(it + 1, 1);
        step(it + 2, 2);
    }
    if (n - whole >= 1) step(whole, 0);
    if (n - whole >= 2) step(whole + 1, 1);
    __syncthreads();  // the patches are no longer needed
    v4i* sums = (v4i*)lds;
    auto sum_at = [&](int b, int from, int q, int t) { return (((b * 4 + from) * 3 + (q < from ? q : q - 1)) * 2 + t) * 64 + lane; };
#pragma unroll
    for (int b = 0; b < TB; ++b)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (q == wave) continue;
            sums[sum_at(b, wave, q, 0)] = (v4i){c0[b][4 * q], c0[b][4 * q + 1], c0[b][4 * q + 2], c0[b][4 * q + 3]};
            sums[sum_at(b, wave, q, 1)] = (v4i){c1[b][4 * q], c1[b][4 * q + 1], c1[b][4 * q + 2], c1[b][4 * q + 3]};
        }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < TB; ++b) {
        int g[4], u[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (q == wave)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    g[j] = c0[b][4 * q + j];
                    u[j] = c1[b][4 * q + j];
                }
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            if (f == wave) continue;
            const v4i v0 = sums[sum_at(b, f, wave, 0)], v1 = sums[sum_at(b, f, wave, 1)];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                g[j] += v0[j];
                u[j] += v1[j];
            }
        }
        const int64_t row = row0 + 32 * b + tok;
        epilogue_run<EPI>(a, row, row < row_end, nb0 * 32 + ch, nb1 * 32 + ch, g, u, rs[b], cs0, cs1);
    }
}

template <int EPI>
static void launch_split_t(const GmmArgs& a, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1)
{
    const int units = a.N / 64;
    const int64_t tiles = (a.R + 32 * TB - 1) / (32 * TB);
    const dim3 grid((unsigned)(tiles * ((units + 7) / 8) * 8));
    auto kernel = gmm_split_kernel<EPI>;
    if (ev0 || ev1) hipExtLaunchKernelGGL(kernel, grid, dim3(256), 0, st, ev0, ev1, 0, a, units);
    else hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, a, units);
}

void launch_split(int epi, const GmmArgs& a, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1)
{
    if (epi == EPI_I32) launch_split_t<EPI_I32>(a, st, ev0, ev1);
    else if (epi == EPI_SWIGLU) launch_split_t<EPI_SWIGLU>(a, st, ev0, ev1);
    else launch_split_t<EPI_DEQUANT>(a, st, ev0, ev1);
}

}  // namespace moe355
