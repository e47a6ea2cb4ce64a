// Grouped int8 x int8 -> int32 GEMM for the expert MLPs, with the three
// epilogues (raw int32, dequant+SwiGLU, dequant to bf16), the weight format
// cast, and the per-row re-quantisation that finishes the SwiGLU op.
//
// Weight-streaming kernel: few rows per expert (decode), where the time is the
// HBM stream of the weights.  Work unit = (expert, pair of 32-channel tiles).
// The weights of a unit are contiguous 1 KiB tiles along K and go straight from
// HBM into MFMA operand registers with one 16-byte load per lane (no LDS: each
// weight byte is used by exactly one wavefront).  The expert's tokens are
// processed 32 at a time as the MFMA's second operand.  With KSPLIT = 4 the
// four wavefronts of a workgroup split K and add their int32 partials through
// LDS (integer addition: exact, order free).
#include <hip/hip_ext.h>
#include <stdlib.h>
#include <type_traits>

#include "gmm_common.h"
#include "gmm_tiled.h"
#include "layer_parts.h"

namespace moe355 {

// ------------------------------------------------------------------ format cast
template <int LAYOUT>
__global__ __launch_bounds__(256) void format_cast_nz_kernel(const int8_t* __restrict__ w, int64_t E, int64_t N,
                                                             int64_t K, int8_t* __restrict__ out)
{
    const int64_t total = E * N * K / 16;
    const int64_t KB = K / 32, NB = N / 32;
    for (int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x; id < total; id += (int64_t)gridDim.x * 256) {
        const int lane = (int)(id & 63);
        const int64_t tile = id >> 6;
        const int64_t kb = tile % KB;
        const int64_t nb = (tile / KB) % NB;
        const int64_t e = tile / (KB * NB);
        const int64_t n = nb * 32 + (lane & 31);
        const int64_t k0 = kb * 32 + (lane >> 5) * 16;
        v4i v;
        if constexpr (LAYOUT == MOE355_W_ENK) {
            v = *(const v4i*)(w + (e * N + n) * K + k0);
        } else {
            uint32_t p[4] = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int b = 0; b < 16; ++b)
                p[b >> 2] |= (uint32_t)(uint8_t)w[(e * K + k0 + b) * N + n] << (8 * (b & 3));
            v = {(int)p[0], (int)p[1], (int)p[2], (int)p[3]};
        }
        *(v4i*)(out + id * 16) = v;
    }
}

// ------------------------------------------------------------------ streaming GEMM
// SLABS: K is cut into gridDim.y slabs (the dense few-row int32 product only; reading gridDim costs every
// wavefront a scalar load in front of its first weight request, 4 us per launch of the decode down GEMM)
// EARLY: the first weight tiles are requested before the group list is read (decode batches: nearly every expert
// has rows, and the lookup hides behind the HBM latency).  A launch that covers only some of the experts of a
// large batch reads the group list first: a unit whose expert is empty or belongs to the other kernel of the call
// would otherwise fetch 32 KiB for nothing, times thousands of units.
// PAIRS: the rows of an expert are not a range of a sorted activation but the (token, slot) pairs that chose it,
// found here from the ids of all pairs (at most 1024: a decode batch).  The four wavefronts of a workgroup work on
// one expert (KSPLIT == 1: four units of it; the host picks that form only when the units of an expert come in
// fours), scan a quarter of the ids each and leave the expert's pairs, in ascending order, in LDS.  The routing
// launch in front of the GEMM then is gating and quantisation only: no sort, no hand-off between workgroups.
// the n-th expert (counting from 0) whose group has rows, or -1: every lane of the wavefront calls it and gets the
// same answer (64 experts per step: one load per lane, a ballot, a count of bits)
__device__ __forceinline__ int nth_expert_with_rows(const int64_t* gl, int gl_type, int E, int n, int lane)
{
    int seen = 0;
    for (int base = 0; base < E; base += 64) {
        const int e = base + lane;
        int64_t c = 0;
        if (e < E) c = (gl_type == 1) ? gl[e] : gl[e] - (e ? gl[e - 1] : 0);
        const unsigned long long m = __ballot(c > 0);
        const int pc = __popcll(m);
        if (n < seen + pc) {
            unsigned long long t = m;
            for (int i = n - seen; i > 0; --i) t &= t - 1;
            return base + __builtin_ctzll(t);
        }
        seen += pc;
    }
    return -1;
}

constexpr int kPairMax = 1024;
constexpr int kPairExperts = 2048;  // that the lookups of the slots can hold

// REQ (pair order, down GEMM): the activation is still the fp32 SwiGLU output; the workgroup re-quantises the rows
// of its expert itself, 32 at a time, into LDS (a wavefront holds whole rows in registers: their maximum by a butterfly, then
// rint(v * (1 / (max / 127))), the arithmetic of swiglu_requant_kernel) and the MFMA operands come from there: the
// re-quantisation launch and its int8 round trip disappear.  The workgroups of an expert (one for every 256 channels) each
// do it again for the expert's rows.
// REQ_ROWS: rows that a wavefront re-quantises at a time, REQ_VEC: 256 values of each are held (K <= 256 REQ_VEC).
template <int EPI, int KSPLIT, int UN, int OCC, bool SLABS = false, bool EARLY = true, bool PAIRS = false,
          int REQ_ROWS = 0, int REQ_VEC = 8>
__global__ __launch_bounds__(256, OCC) void gmm_stream_kernel(GmmArgs a)
{
    static_assert(KSPLIT == 1 || KSPLIT == 4, "workgroup barriers need all four wavefronts on one unit");
    static_assert(!PAIRS || (!SLABS && EARLY && EPI != EPI_I32), "pair order: the two GEMMs of a decode layer");
    constexpr bool REQ = REQ_ROWS > 0;
    static_assert(!REQ || (PAIRS && EPI == EPI_DEQUANT), "the re-quantisation sits in the pair-order down GEMM");
    extern __shared__ __attribute__((aligned(16))) int8_t qtile[];  // REQ: 32 rows of K + 16 bytes
    __shared__ float qscale[REQ ? 32 : 1];
    constexpr int kRed = (KSPLIT > 1) ? 32 * 64 : 1;
    __shared__ int32_t red[PAIRS && kRed < kPairExperts ? kPairExperts : kRed];
    __shared__ uint16_t plist[PAIRS ? kPairMax : 1];
    __shared__ int32_t pcount[4];
    __shared__ uint32_t pmap[PAIRS ? 64 : 1];  // one bit per expert (at most 2048) that has pairs
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // tell the compiler: addresses go to SGPRs
    const int lane = threadIdx.x & 63;
    const int NB = a.N >> 5, KB = a.K >> 5;
    const int upe = NB >> 1;  // units per expert
    const int64_t unit = (KSPLIT == 1) ? (int64_t)blockIdx.x * 4 + wave : (int64_t)blockIdx.x;
    // pair order: the grid has slots instead of a place per expert (an idle expert's workgroup only finds that out, but
    // it still costs its dispatch -- 28,000 of them are 150 us -- and the weights it has requested by then), and slot s
    // belongs to the s-th expert that has pairs; the workgroups that start first have places (pair_places below)
    const int places = PAIRS ? a.sh_blocks + a.pair_first + a.pair_slots + a.pair_extra : (!EARLY && a.gl_slots > 0) ? a.gl_slots : a.E;
    if (unit >= (int64_t)places * upe) return;  // KSPLIT == 1: no barriers below; KSPLIT == 4: whole workgroup leaves
    int e = (int)(unit / upe);
    const int p = (int)(unit % upe);
    int block = 0;        // pair order: which 32 rows of the expert
    bool shared = false;  // ... and whether it is the shared one (the same answer in all four wavefronts)
    if constexpr (PAIRS) {
        shared = e < a.sh_blocks;
        if (shared) block = e;
        e = shared ? 0 : e - a.sh_blocks;
        // further blocks are numbered behind the slots, the first pair_early of them run in front of the slots
        if (e >= a.pair_first && e < a.pair_first + a.pair_early + a.pair_slots)
            e = e < a.pair_first + a.pair_early ? e + a.pair_slots : e - a.pair_early;
    }
    const int nb0 = (EPI == EPI_SWIGLU) ? p : 2 * p;
    const int nb1 = (EPI == EPI_SWIGLU) ? p + upe : 2 * p + 1;

    // K is cut into gridDim.y slabs (SLABS: the dense few-row product, whose workgroups store their int32 partial
    // sums to a plane per slab, or without scratch add them into a zeroed result with atomics: integer addition,
    // exact and order free), and a slab into KSPLIT pieces, one per wavefront
    const int ks = (KSPLIT == 1) ? 0 : wave;
    int slab_begin = 0, slab_end = KB;
    if constexpr (SLABS) {
        slab_begin = (int)(((int64_t)KB * blockIdx.y) / gridDim.y);
        slab_end = (int)(((int64_t)KB * (blockIdx.y + 1)) / gridDim.y);
    }
    const int kb_begin = slab_begin + ((slab_end - slab_begin) * ks) / KSPLIT;
    const int kb_end = slab_begin + ((slab_end - slab_begin) * (ks + 1)) / KSPLIT;

    // pair order: wavefront w scans pairs [w Q, (w + 1) Q), Q a multiple of 64 and at most 256.  The ids are
    // requested in front of the weights: answers come back in the order of the requests, and the list of the
    // expert's pairs (which the token loads wait for) should not queue behind the first weight tiles from HBM.
    const int Q = PAIRS ? (((int)a.R + 255) >> 8) << 6 : 0;
    int pid[PAIRS ? 4 : 1];
    if constexpr (PAIRS) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int f = wave * Q + c * 64 + lane;
            pid[c] = (c * 64 < Q && f < (int)a.R) ? a.pair_ids[f] : -1;
        }
    }
    if constexpr (PAIRS) {
        if (shared) {
            // nothing to look up
        } else if (e >= a.pair_first + a.pair_slots) {
            // further blocks of experts with more than 32 rows, in the order of the experts: the pairs of every expert
            // are counted in LDS and every wavefront walks the counts, 64 experts at a time
            for (int i = threadIdx.x; i < a.E; i += 256) red[i] = 0;
            __syncthreads();
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (pid[c] >= 0 && pid[c] < a.E) atomicAdd(&red[pid[c]], 1);
            __syncthreads();
            int left = e - a.pair_first - a.pair_slots;
            e = -1;
            for (int base = 0; base < a.E && e < 0; base += 64) {
                const int n = base + lane < a.E ? red[base + lane] : 0;
                const int more = n > 32 ? (n - 1) >> 5 : 0;
                const int incl = wave_scan_inclusive_i32(more);
                const bool has = left >= incl - more && left < incl;
                const unsigned long long holder = __ballot(has);
                if (holder) {
                    const int h = __builtin_ctzll(holder);
                    e = base + h;
                    block = 1 + __builtin_amdgcn_readlane(left - (incl - more), h);
                } else {
                    left -= __builtin_amdgcn_readlane(incl, 63);
                }
            }
            if (e < 0) return;  // not so many blocks (the same answer in all four wavefronts)
            __syncthreads();    // the counts are read before the sums take their place
        } else if (e >= a.pair_first) {  // the same answer in all four wavefronts (KSPLIT == 1: units come in fours)
            // the experts that have pairs, as a bit map in LDS; every wavefront then finds the expert of the
            // workgroup's slot by itself: a count of the bits in front of each word, and the word's bit
            if (threadIdx.x < 64) pmap[threadIdx.x] = 0u;
            __syncthreads();
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (pid[c] >= 0 && pid[c] < a.E) atomicOr(&pmap[pid[c] >> 5], 1u << (pid[c] & 31));
            __syncthreads();
            const int mine0 = lane * 32;
            const uint32_t bits = a.pair_first <= mine0 ? pmap[lane]
                                  : a.pair_first >= mine0 + 32 ? 0u : pmap[lane] & (~0u << (a.pair_first - mine0));
            const int cnt = __popc(bits);
            int incl = cnt;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int t = __shfl_up(incl, off, 64);
                if (lane >= off) incl += t;
            }
            const int excl = incl - cnt;
            const int slot = e - a.pair_first;
            const bool has = slot >= excl && slot < incl;
            const unsigned long long holder = __ballot(has);
            if (holder == 0ull) return;  // fewer experts with pairs than slots (the same answer in all four wavefronts)
            uint32_t t = bits;
            for (int i = has ? slot - excl : 0; i > 0; --i) t &= t - 1;
            const int mine = mine0 + (t ? __builtin_ctz(t) : 0);
            e = __builtin_amdgcn_readlane(mine, __builtin_ctzll(holder));
        }
    }
    if constexpr (!PAIRS && !EARLY) {
        if (a.gl_slots > 0) {  // few rows over many experts: the workgroup's place is a slot, not an expert
            e = __builtin_amdgcn_readfirstlane(nth_expert_with_rows(a.gl, a.gl_type, a.E, e, lane));
            if (e < 0) return;
        }
    }
    const int8_t* we = (PAIRS && shared) ? a.sh_w : expert_weights(a, e);
    const int8_t* w0 = we + ((int64_t)nb0 * KB) * 1024 + lane * 16;
    const int8_t* w1 = we + ((int64_t)nb1 * KB) * 1024 + lane * 16;

    // The weight addresses depend only on the unit, so the first batch of weight tiles is requested
    // before the expert's row range is known: the group-list lookup hides behind the HBM latency.
    v4i a0[UN], a1[UN];
    auto load_weights = [&](int kb) {
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const int k = kb + u;
            if (k < kb_end) {
                a0[u] = gload16_nt(w0 + (int64_t)k * 1024);
                a1[u] = gload16_nt(w1 + (int64_t)k * 1024);
            } else {
                a0[u] = (v4i){0, 0, 0, 0};
                a1[u] = (v4i){0, 0, 0, 0};
            }
        }
    };
    if constexpr (EARLY) load_weights(kb_begin);

    int64_t row0 = 0, row1 = 0;
    if (PAIRS && shared) {
        row0 = 32 * block;
        row1 = row0 + 32 < a.sh_rows ? row0 + 32 : a.sh_rows;
    } else if constexpr (PAIRS) {
        const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
        bool mine[4];
        int cnt = 0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            mine[c] = pid[c] == e;
            cnt += __popcll(__ballot(mine[c]));
        }
        if (lane == 0) pcount[wave] = cnt;
        __syncthreads();
        int base = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            if (w < wave) base += pcount[w];
            row1 += pcount[w];
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const unsigned long long m = __ballot(mine[c]);
            if (mine[c]) plist[base + __popcll(m & below)] = (uint16_t)(wave * Q + c * 64 + lane);
            base += __popcll(m);
        }
        __syncthreads();
        if (row1 == 0) return;  // the whole workgroup: nobody chose this expert
        if (a.pair_extra > 0) {
            row0 = 32 * block;
            if (row1 > row0 + 32) row1 = row0 + 32;
        }
    } else {
        expert_rows(a.gl, a.gl_type, e, lane, row0, row1);
        if (row1 > a.R) row1 = a.R;
        if (row1 <= row0) return;
    }
    if constexpr (!EARLY) load_weights(kb_begin);

    const int tok = lane & 31;
    const int kh = lane >> 5;

    // The channel scales of the runs this wavefront finishes (all four quarters, or quarter `wave` when K is
    // split) are requested together and before the first store of the epilogue: a load placed behind a store
    // waits for it (the memory counter retires in order), one round trip per run.  With K split they are two
    // registers and are requested in front of the K loop; the unsplit form requests them when the K loop has
    // ended, two quarters at a time (all eight together cost a wavefront of occupancy).
    constexpr int NQ = (KSPLIT == 1) ? 2 : 1;  // quarters whose scales are held at a time
    v4f cs0[NQ], cs1[NQ];
    auto load_channel_scales = [&](int q_first) {
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            cs0[i] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
            cs1[i] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (EPI != EPI_I32) {
                const float* cs = (PAIRS && shared) ? a.sh_scale : expert_scales(a, e);
                const int ch = quad_channel(KSPLIT == 1 ? q_first + i : wave, lane);
                cs0[i] = gload4f(cs + nb0 * 32 + ch);
                cs1[i] = gload4f(cs + nb1 * 32 + ch);
            }
        }
    };
    if constexpr (KSPLIT > 1) load_channel_scales(0);

    for (int64_t r0 = row0; r0 < row1; r0 += 32) {
        const bool valid = r0 + tok < row1;
        using Index = std::conditional_t<PAIRS, int32_t, int64_t>;  // at most 1024 rows in pair order
        Index row, src;  // where the row's result goes, where its values lie
        if constexpr (PAIRS) {
            if (shared) {
                const int t = valid ? (int)r0 + tok : (int)row0;
                row = (int)a.R + t;
                src = a.pair_gather ? t : row;
            } else {
                row = plist[valid ? r0 + tok : 0];
                src = a.pair_gather ? row / a.pair_k : row;
            }
        } else {
            row = r0 + tok;
            src = a.row_src ? (int64_t)a.row_src[valid ? row : row0] : row;
        }
        const int8_t* xb = REQ ? qtile : a.x;
        std::conditional_t<PAIRS, uint32_t, int64_t> xo;  // this lane's operand bytes of the row, behind xb
        float rs = 0.0f;
        if constexpr (!REQ) xo = src * a.K + kh * 16;
        if constexpr (REQ) {
            // rows r0 .. r0 + 31 of the expert -> int8 in LDS: a wavefront takes every fourth row and holds REQ_ROWS of them in
            // registers between their maxima and their quantisation
            const int pitch = a.K + 16;  // rows 16 bytes apart in the banks
            const int rows_now = (int)(row1 - r0 < 32 ? row1 - r0 : 32);
            if (r0 != row0) __syncthreads();  // nobody still reads the rows of the pass before
            for (int rr = wave; rr < rows_now; rr += 4 * REQ_ROWS) {
                v4f v[REQ_ROWS][REQ_VEC];
                float amax[REQ_ROWS];
#pragma unroll
                for (int t = 0; t < REQ_ROWS; ++t) {
                    const bool on = rr + 4 * t < rows_now;
                    const float* y = a.y_in + (int64_t)plist[r0 + (on ? rr + 4 * t : rr)] * a.K + lane * 4;
#pragma unroll
                    for (int i = 0; i < REQ_VEC; ++i)
                        v[t][i] = on && i * 256 + lane * 4 < a.K ? *(const v4f*)(y + i * 256) : (v4f){0.0f, 0.0f, 0.0f, 0.0f};
                }
#pragma unroll
                for (int t = 0; t < REQ_ROWS; ++t) {
                    bool nan = false;
                    amax[t] = 0.0f;
#pragma unroll
                    for (int i = 0; i < REQ_VEC; ++i) amax[t] = max_abs(amax[t], v[t][i], nan);
                    if (nan) {
                        amax[t] = 0.0f;
#pragma unroll
                        for (int i = 0; i < REQ_VEC; ++i) amax[t] = max_abs_any(amax[t], v[t][i]);
                    }
                }
#pragma unroll
                for (int off = 32; off > 0; off >>= 1)
#pragma unroll
                    for (int t = 0; t < REQ_ROWS; ++t) {
                        const float o = __shfl_xor(amax[t], off, 64);
                        amax[t] = o > amax[t] ? o : amax[t];
                    }
#pragma unroll
                for (int t = 0; t < REQ_ROWS; ++t) {
                    const int at = rr + 4 * t;
                    if (at >= rows_now) break;
                    const float inv = 1.0f / (amax[t] / 127.0f);
#pragma unroll
                    for (int i = 0; i < REQ_VEC; ++i) {
                        if (i * 256 + lane * 4 >= a.K) break;
                        *(uint32_t*)(qtile + at * pitch + i * 256 + lane * 4) = quantise_times(v[t][i], inv);
                    }
                    if (lane == 0) qscale[at] = (amax[t] == 0.0f) ? 0.0f : amax[t] / 127.0f;
                }
            }
            __syncthreads();
            xo = (valid ? tok : 0) * pitch + kh * 16;
            rs = qscale[valid ? tok : 0];
        } else if constexpr (EPI != EPI_I32) {
            rs = a.row_scale[(PAIRS || a.row_src) ? src : (valid ? row : row0)];
        }
        v16i c0 = {0}, c1 = {0};
        if (r0 != row0) load_weights(kb_begin);
        for (int kb = kb_begin; kb < kb_end; kb += UN) {
            v4i b[UN];
#pragma unroll
            for (int u = 0; u < UN; ++u)
                b[u] = (valid && kb + u < kb_end) ? *(const v4i*)(xb + (xo + (kb + u) * 32)) : (v4i){0, 0, 0, 0};
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                c0 = mfma_i8(a0[u], b[u], c0);
                c1 = mfma_i8(a1[u], b[u], c1);
            }
            if (kb + UN < kb_end) load_weights(kb + UN);
        }
        if constexpr (KSPLIT > 1) {
            // int32 partial sums of the four K slices meet in LDS (integer adds: exact, order free),
            // then every wavefront finishes one quarter of the channels
            if (wave == 0) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    red[v * 64 + lane] = c0[v];
                    red[(16 + v) * 64 + lane] = c1[v];
                }
            }
            __syncthreads();
            if (wave > 0) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    atomicAdd(&red[v * 64 + lane], c0[v]);
                    atomicAdd(&red[(16 + v) * 64 + lane], c1[v]);
                }
            }
            __syncthreads();
            int g[4], u[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                g[j] = red[(4 * wave + j) * 64 + lane];
                u[j] = red[(16 + 4 * wave + j) * 64 + lane];
            }
            const int ch = quad_channel(wave, lane);
            if constexpr (EPI == EPI_I32 && SLABS) {
                if (valid && a.acc_part) {
                    // the slab's partial sums to its own plane of the scratch; slab_sum_kernel adds the planes
                    int32_t* plane = a.acc_part + ((int64_t)blockIdx.y * a.R + (int64_t)row) * a.N;
                    *(v4i*)(plane + nb0 * 32 + ch) = (v4i){g[0], g[1], g[2], g[3]};
                    *(v4i*)(plane + nb1 * 32 + ch) = (v4i){u[0], u[1], u[2], u[3]};
                } else if (valid) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        atomicAdd(a.acc + (int64_t)row * a.N + nb0 * 32 + ch + j, g[j]);
                        atomicAdd(a.acc + (int64_t)row * a.N + nb1 * 32 + ch + j, u[j]);
                    }
                }
            } else {
                epilogue_run<EPI>(a, row, valid, nb0 * 32 + ch, nb1 * 32 + ch, g, u, rs, cs0[0], cs1[0],
                                  PAIRS && shared);
            }
            __syncthreads();
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (q % NQ == 0) load_channel_scales(q);  // two quarters per round trip
                int g[4] = {c0[4 * q], c0[4 * q + 1], c0[4 * q + 2], c0[4 * q + 3]};
                int u[4] = {c1[4 * q], c1[4 * q + 1], c1[4 * q + 2], c1[4 * q + 3]};
                const int ch = quad_channel(q, lane);
                epilogue_run<EPI>(a, row, valid, nb0 * 32 + ch, nb1 * 32 + ch, g, u, rs, cs0[q % NQ], cs1[q % NQ],
                                  PAIRS && shared);
            }
        }
    }
}

// ------------------------------------------------------------------ SwiGLU re-quantisation
// One wavefront per row: SwiGLU values y fp32 [R, I] -> row absmax -> int8 + scale.
// Rows at or beyond the last group are left untouched.
// NV > 0: the row (at most NV x 256 values) stays in registers between the two passes, so y is read once;
// NV == 0: any length, second pass re-reads the row.
// Bound by memory: 251 MB of 65,536 rows of 768 values in 44 us, 335 MB of 32,768 rows of 2048 in 57 (47 and 60 with a
// comparison and a selection per bound and value, shifts and masks for the bytes and ordinary loads; two, four and eight
// rows per wavefront 44 / 49 / 61 and - / 61 / 69).
template <int NV>
__global__ __launch_bounds__(256) void swiglu_requant_kernel(const float* __restrict__ y,
                                                             const int64_t* __restrict__ gl, int gl_type, int E,
                                                             int64_t R, int I, int8_t* __restrict__ q,
                                                             float* __restrict__ qs, int64_t shared_from)
{
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= R) return;
    const v4f* yr = (const v4f*)(y + row * I);
    const int nvec = I >> 2;
    v4f held[NV > 0 ? NV : 1];
    if constexpr (NV > 0) {  // requested before the group list is looked at, and past the caches: nobody reads them again
#pragma unroll
        for (int n = 0; n < NV; ++n) {
            const int i = lane + 64 * n;
            held[n] = i < nvec ? __builtin_nontemporal_load(yr + i) : (v4f){0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    if (gl) {  // without a group list (pair order) every row is a row of some expert
        int64_t r0, total;
        expert_rows(gl, gl_type, E - 1, lane, r0, total);
        if (row >= total) return;
    }
    float amax = 0.0f;
    if constexpr (NV > 0) {
        bool nan = false;
#pragma unroll
        for (int n = 0; n < NV; ++n) amax = max_abs(amax, held[n], nan);
        if (nan) {
            amax = 0.0f;
#pragma unroll
            for (int n = 0; n < NV; ++n) amax = max_abs_any(amax, held[n]);
        }
    } else {
        for (int i = lane; i < nvec; i += 64) amax = max_abs_any(amax, yr[i]);
    }
    amax = wave_max(amax);
    const bool shared = row >= shared_from;
    const float s = shared ? amax * (float)(1.0 / 127.0) : amax / 127.0f;
    const float inv = 1.0f / s;
    if (lane == 0) qs[row] = (amax == 0.0f) ? 0.0f : s;
    uint32_t* qr = (uint32_t*)(q + row * I);
    auto pack = [&](v4f v) {
        if (shared) return quantise_over(v, s);
        return quantise_times(v, inv);
    };
    if constexpr (NV > 0) {
#pragma unroll
        for (int n = 0; n < NV; ++n) {
            const int i = lane + 64 * n;
            if (i < nvec) qr[i] = pack(held[n]);
        }
    } else {
        for (int i = lane; i < nvec; i += 64) qr[i] = pack(yr[i]);
    }
}

void launch_swiglu_requant(const float* y, const int64_t* gl, int gl_type, int E, int64_t R, int I, int8_t* q,
                           float* qs, hipStream_t st, int64_t shared_from)
{
    const dim3 grid((unsigned)((R + 3) / 4));
#define MOE355_REQUANT(NV_) \
    hipLaunchKernelGGL(swiglu_requant_kernel<NV_>, grid, dim3(256), 0, st, y, gl, gl_type, E, R, I, q, qs, shared_from)
    if (I <= 4 * 256) MOE355_REQUANT(4);
    else if (I <= 8 * 256) MOE355_REQUANT(8);
    else if (I <= 16 * 256) MOE355_REQUANT(16);
    else MOE355_REQUANT(0);
#undef MOE355_REQUANT
}

static int check_gmm(const void* x, const void* w, const int64_t* gl, int gl_type, int64_t rows, int64_t k, int64_t n,
                     int E)
{
    if (rows < 0 || k <= 0 || n <= 0 || E <= 0) return MOE355_E_ARG;
    if (gl_type != MOE355_GL_CUMSUM && gl_type != MOE355_GL_COUNT) return MOE355_E_ARG;
    if (n % 64 != 0 || k % 32 != 0) return MOE355_E_SHAPE;
    if (rows >= 0x7fffffffLL || n >= 0x7fffffffLL || k >= 0x7fffffffLL) return MOE355_E_SHAPE;
    if ((int64_t)E * (n / 64) >= 0x7fffffffLL) return MOE355_E_SHAPE;
    if (rows > 0 && (!x || !w || !gl)) return MOE355_E_ARG;
    if (((uintptr_t)x & 15) || ((uintptr_t)w & 15)) return MOE355_E_SHAPE;
    return MOE355_OK;
}

// Measurement hook: events that bracket exactly the next grouped-GEMM kernel launched from
// this thread (set by moe355_profile_next_gemm, consumed by one launch).
static thread_local hipEvent_t t_ev_start = nullptr;
static thread_local hipEvent_t t_ev_stop = nullptr;

void take_profile_events(hipEvent_t& start, hipEvent_t& stop)
{
    start = t_ev_start;
    stop = t_ev_stop;
    t_ev_start = nullptr;
    t_ev_stop = nullptr;
}

__global__ __launch_bounds__(256) void zero_i32_kernel(int32_t* __restrict__ p, int64_t n4)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n4) ((v4i*)p)[i] = (v4i){0, 0, 0, 0};
}

// acc = sum of the slabs' planes, for the rows of the one expert (gl[0] of them: count and running sum are the
// same number for one expert); the other rows become zero.  Integer sums: exact in any order.
__global__ __launch_bounds__(256) void slab_sum_kernel(const int32_t* __restrict__ part, int slabs, int64_t R, int N,
                                                       const int64_t* __restrict__ gl, int32_t* __restrict__ acc)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // 16-byte piece of acc
    const int64_t n4 = R * (int64_t)N / 4;
    if (i >= n4) return;
    int64_t rows = gl[0];
    if (rows > R) rows = R;
    v4i s = {0, 0, 0, 0};
    if (i * 4 / N < rows) {
        for (int p = 0; p < slabs; ++p) {
            const v4i v = ((const v4i*)(part + (int64_t)p * R * N))[i];
            s = (v4i){s[0] + v[0], s[1] + v[1], s[2] + v[2], s[3] + v[3]};
        }
    }
    ((v4i*)acc)[i] = s;
}

template <typename KernelT>
static void launch_gemm(KernelT kernel, dim3 grid, hipStream_t st, const GmmArgs& a, hipEvent_t ev0, hipEvent_t ev1)
{
    if (ev0 || ev1) hipExtLaunchKernelGGL(kernel, grid, dim3(256), 0, st, ev0, ev1, 0, a);
    else hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, a);
}

// Rows per expert decide the kernel: a handful -> weight streaming over single wavefronts; more -> LDS-tiled MFMA
// kernel with 128-row tiles; many, when K is long enough to amortise a tile's fill and epilogue, the weight-streaming
// tiles (up to 256 rows) that fetch an expert's weights once.  The host only knows the mean, and the histogram may be
// skewed (real routers are): the 128-row tiles cost a cold expert little more than streaming does (a short tile that
// is its expert's only one reads its weights once, past the caches) and a hot one a fraction of it, so they start early.
constexpr int64_t kComputeUnits = 256;

static int tiled_bm(const GmmArgs& a)
{
    if (a.K % 64 != 0) return 0;
#ifdef MOE355_DEV_KNOBS  // experiments only (never defined for the shipped library): force one kernel family
    static const char* force = getenv("MOE355_GEMM");
    if (force && force[0] == 's') return 0;
    if (force && force[0] == 't') return 128;
    if (force && force[0] == 'T') return 256;
    if (force && force[0] == 'u') return 64;
#endif
    const int64_t avg = a.R / a.E;
    const int64_t weights = (int64_t)a.E * a.N * a.K;
    // Streaming or 128-row tiles, the whole layer through the sorted path in us, uniform routing and Zipf(1.1):
    //   256 experts, K = 7168 / 2048 (7 and 3.5 GiB): 16 tokens (half a row per expert) 685 against 703 and 253
    //     against 281; 32 tokens 1097 against 1100 and 351 against 328; 64 tokens 1455 against 1449 and 442 against
    //     406; 96 tokens 1584 against 1592 and 508 against 423.  So from one row per expert on: tiles.
    //   Products of one GiB, 256 experts of 2048 x 2048 (the down product alone), 1 / 2 / 4 / 8 / 14 / 23 rows per
    //     expert: 123 / 144 / 160 / 167 / 174 / 191 streaming, 116 / 142 / 162 / 166 / 172 / 175 on tiles; Zipf 91 / 117 /
    //     148 / 202 / 230 / 309 against 74 / 100 / 122 / 154 / 166 / 176; K from 512 to 8192 and 128 experts alike.
    //     Sending the experts of up to 32 rows to streaming and the others to tiles, in two launches: uniform 115 / 143 /
    //     164 / 171 / 178 / 207, Zipf 72 / 114 / 137 / 162 / 171 / 184 (never more than 3 % ahead of the tiles, up to
    //     35 % behind them at K = 8192).
    //   128 experts, K = 2048 / 768 (0.4 and 0.2 GB): 48 / 100 tokens 107 / 112 against 117 / 131 and 81 / 86 against
    //     73 / 81, so decode batches (fewer than 1024 rows) stream; 130 / 190 tokens 120 / 123 against 123 / 126 and
    //     153 / 183 against 80 / 88: tiles.
    //   From 32 rows per expert on an expert streams its weights more than once, and few rows go on tiles as well: 16
    //     experts, K = 2048 / 1408, 24 / 32 / 40 rows per expert 57.9 / 68.2 / 73.7 against 54.8 / 56.7 / 58.2 (Zipf 92 / 110
    //     / 131 against 56 / 57 / 58); 24 experts, K = 4096 / 2048, 27 / 40: 154 / 232 against 133 / 138; 8 experts of that
    //     shape, 24 / 32: 59.6 / 83.0 against 72.8 / 74.9, so no earlier.
    //     That is so because streaming fills the chip.  With workgroups for half of it the second reading costs nothing, and a
    //     tile's walk along K alone does: one product, 32 to 47 rows per expert, tiles / streaming at up to 128 workgroups 1.37
    //     to 1.61 for K from 2048, 1.25 to 1.29 for K = 1024; at 192 and 256 1.04 to 1.38, at 288 to 512 0.69 to 1.21.  Skewed
    //     routing pays for the passes of its hot experts, the more the more experts there are: up to 128 workgroups, mean of
    //     uniform routing and of Zipf(1.1), 4 experts 1.39 and 1.07, 8 experts 1.38 and 0.78, 16 experts 1.40 and 0.57, 24
    //     experts 1.38 and 0.43.  So up to eight experts.  With K below 1024 it is little: layers of 8 to 24 experts of 256 to
    //     768, 26 to 29 us streaming and 28 to 32 on tiles (Zipf 30 to 59 against 28 to 38).
    if (a.R < a.E) return 0;
    const bool few_streams = a.E <= 8 && (int64_t)a.E * (a.N / 64) <= kComputeUnits / 2 && a.K >= 1024;
    if (avg < (few_streams ? 48 : 32) && a.R < 1024 && (a.R < 128 || weights < (1ll << 30))) return 0;
    // Few experts and few rows: as long as tiles of half the height do not outnumber the compute units they are twice as
    // many and half as long (rows / 64 and half a tile per expert for its last one).  8 experts of 2816 x 1024 and 1024 x
    // 1408, the layer at 512 / 768 / 1024 / 1536 tokens of two slots 50.8 / 51.5 / 52.5 / 62.6 us on 128-row tiles, 41.7 /
    // 46.5 / 49.1 / 59.9 with this rule (2048 tokens, where it would be one tile too many for the down product: 65.8
    // against 67.2).  Half a tile per expert is what a uniform batch needs; under skewed routing nearly every expert has a last
    // tile of its own, and where that makes one more than the chip holds the launch takes twice as long.  With up to 16
    // experts it makes few (small layer under Zipf(1.1), 576 / 639 / 1900 tokens 48.4 / 50.9 / 62.4 us with this rule, 51.4 /
    // 51.6 / 65.0 on 128-row tiles); beyond, three quarters are taken: 24 experts of 7168 x 2048, 48 rows each under Zipf(1.1)
    // 68 us on 128-row tiles, 111 on 64-row tiles, 64 of 4096 x 768, 40 rows each 42 against 64, while uniform batches lose 3 %
    // there.  Not for products of up to 512 channels (below).
    const int64_t last_tiles = a.E <= 16 ? a.E / 2 : 3 * (int64_t)a.E / 4;
    if (a.E > 1 && a.N > 512 && (a.R / 64 + last_tiles) * ((a.N + 255) / 256) <= kComputeUnits) return 64;
    // the list of 256-row tiles is built from 16-bit counters (tile_map_kernel, by_length)
    const bool wide_ok = a.R / 256 + a.E < 32768;
    // K = 7168 / 2048, uniform routing, 28 / 40 / 48 / 56 / 64 / 94 rows per expert: the layer takes 1968 / 2028 / 2055 /
    // 2091 / 2126 / 2280 us with the weight-streaming tiles in the first product, 1867 / 1975 / 2031 / 2088 / 2162 / 2512
    // us on 128-row tiles; Zipf(1.1) at 28 / 40 / 64 / 94 / 128 1115 / 1361 / 1703 / 2164 / 2616 against 1069 / 1339 /
    // 1667 / 2155 / 2648.  128 experts at K = 4096, 56 / 69 / 81 rows: 526 / 547 / 567 against 511 / 552 / 576.
    // Since then tiles that are their expert's only one read its weights past the caches, and the wide tiles, bound by that
    // stream, win a little earlier in uniform routing, not under Zipf(1.1): the same layer, 44 / 50 / 56 rows 1896 / 2020 /
    // 2032 us on 128-row tiles, 1869 / 1951 / 1895 on wide ones, Zipf 1435 / 1545 / 1654 against 1464 / 1600 / 1633; 128
    // experts at K = 4096, 40 to 64 rows, 0.96 to 0.99 of the time and 1.04 to 1.10.  So the line stays at 64.
    // A handful of wide tiles leaves most of the chip idle: 8 experts, K = 4096 / 2048 (64 columns of tiles), 500 / 800 / 1000
    // tokens of two slots 123 / 159 / 169 us with them, 99 / 102 / 126 on 128-row tiles (Zipf(1.1) 154 / 159 / 172 against 97 /
    // 104 / 136); 16 experts (128 columns), 600 / 1000 / 1500 tokens 136 / 160 / 193 against 120 / 168 / 160; 32 experts 196 /
    // 215 / 272 against 196 / 262 / 276.  (One expert: a dense product on a side stream, which should leave the chip idle.)
    const bool narrow = a.N <= 512;
    const int64_t columns = (int64_t)a.E * ((a.N + 511) / 512);
    // Since their tall tiles are spread among the others they win earlier under Zipf(1.1) too where there are columns for four
    // rounds of the chip and more.  One product, wide / 128-row tiles, uniform (Zipf(1.1)), at 24 / 40 / 60 rows: 1024 columns, 128
    // experts of 7168 / 4096 0.98 / 0.95 / 0.94 (1.01 / 0.94 / 0.92); 1280 and 1536 columns of them 0.98 / 0.96 / 0.91 (0.99 to 1.01 /
    // 0.92 to 0.95 / 0.94 to 0.96); 256 of 5120 / 4096 0.96 / 0.94 / 0.90 (1.00 / 0.92 / 0.92), of 4096 / 4096 0.99 / 0.98 / 0.97
    // (1.03 / 0.98 / 0.96), of 7168 / 3072 0.97 / 0.96 / 0.90 (1.02 / 0.93 / 0.91); 160 of 6144 / 6144 0.99 / 0.97 / 0.92 (0.99 /
    // 0.95 / 0.92): from 40 rows on.  Below 1024 columns uniform routing wins and Zipf does not: 512 and 256 columns of 7168 / 4096
    // at 48 rows 0.98 and 0.99 (1.03 and 1.18), 768 of 128 experts of 4096 / 3072 0.94 (1.03).
    // From 2048 columns on earlier still, and with many experts and a long K, where more of the time is the weight stream, before
    // that.  Layers, the mean over uniform routing, Zipf(0.8) and Zipf(1.1), ten draws each, wide / 128-row tiles at 12 / 16 / 18 /
    // 20 / 24 / 28 / 36 rows:
    //   256 experts of 7168 / 2048 1.02 / 0.99 / 0.98 / 0.98 / 0.99 / 0.96 / 0.96, of 5120 / 2048 1.04 / 0.99 / 0.98 / 0.98 / 0.98 /
    //     0.96 / 0.95: from 17 on, though mildly skewed batches lose until 24 (at 18 rows uniform 0.98 and 0.97, Zipf(0.8) 1.02 and
    //     1.02, Zipf(1.1) 0.95 and 0.94)
    //   256 of 4096 / 2048 1.05 / 1.01 / 1.00 / 1.00 / 1.00 / 0.98 / 0.97 (Zipf(0.8) 1.04 at 18 and 20, 0.99 at 28), 512 of 4096 / 1024
    //     1.03 / 1.01 / 0.99 / 0.99 / 1.00 / 0.99 / 0.99, 192 of 7168 / 2816 1.03 / 1.02 / 1.01 / 1.00 / 0.99 / 0.98 / 0.97, 128 of 7168 /
    //     4096 0.99 / 1.01 / 1.00 / 1.00 / 1.00 / 0.98 / 0.96, of 8192 / 4096 0.98 / 1.02 / 1.01 / 1.02 / 1.02 / 0.98 / 0.95, of 5120 / 4096
    //     0.98 / 1.01 / 0.99 / 1.01 / 1.00 / 0.97 / 0.96, 64 of 6144 / 8192 1.00 / 0.99 / 0.99 / 0.98 / 0.98 / 0.96 / 0.95: from 28 on
    const int64_t early = a.E >= 256 && a.K >= 5120 ? 17 : 28;
    const int64_t from = columns < 4 * kComputeUnits || narrow ? 64 : columns < 8 * kComputeUnits ? 40 : early;
    if (avg >= from && avg <= 256 && a.K >= 4096 && wide_ok && (narrow || a.E == 1 || columns >= kComputeUnits / 2)) return 256;
    // Above 256 rows an expert has two tall tiles and more, and they fetch its weights half as often as the 128-row tiles.  That
    // is what counts where an expert's weights are several times the 4 MiB of an XCD's L2.  One product, wide / 128-row tiles:
    //   32 MiB and more per expert at K >= 4096: 16 experts of 14336 x 4096, 264 / 352 / 512 / 1024 rows 0.79 / 0.78 / 0.69 /
    //     0.65 (991 against 681 us at 512), Zipf(1.1) 1.00 / 0.83 / 0.80 / 0.78; 64 of 8192 x 5120 0.77 / 0.81 / 0.71 / 0.69, Zipf
    //     0.91 / 0.87 / 0.82 / 0.75; 32 of 8192 x 4096 0.85 / 0.91 / 0.86 / 0.84, Zipf 0.93 / 0.91 / 0.89 / 0.87.
    //   14 MiB and more, from 384 rows on (two tiles of 256 are mostly padding before): 256 experts of 7168 x 2048, 352 / 384 /
    //     512 / 1024 rows 1.05 / 0.95 / 0.93 / 0.89, Zipf 0.94 / 0.90 at 384 / 512; 64 of them 1.05 / 0.96 / 0.93 / 0.89, Zipf
    //     0.92 / 0.97 / 0.95 / 0.89; 128 of 5120 x 3072 0.97 / 0.95 / 0.93 at 384 / 512 / 1024, Zipf 0.97 / 0.93 / 0.92.  With
    //     fewer columns of tiles the last tall ones weigh more: 384 / 512 / 1024 rows, 266 columns (19 experts of 7168 x 2048)
    //     1.06 / 1.01 / 0.92, Zipf 1.07 / 0.90 / 0.89, 260 (26 of 5120 x 3072) 1.14 / 1.00 / 0.94, Zipf 1.09 / 0.95 / 0.98, 520 (52
    //     of them) 1.05 / 1.01 / 0.95, Zipf 0.98 / 0.97 / 0.93; so from 512 rows on below 768 columns.  Ten MiB (5120 x 2048)
    //     1.05, Zipf 1.00 to 1.04.
    //   Fewer channels than 5120 from 3072 on, for 20 MiB, K >= 5120 and 768 columns: 384 / 512 / 1024 rows, 256 experts of 4096 x
    //     7168 0.91 / 0.92 / 0.90 (512 rows 4961 against 4565 us), Zipf 0.94 / 0.94 / 0.91; 128 of them 0.89 / 0.91 / 0.89, Zipf
    //     0.97 / 0.95 / 0.91; 160 of 4608 x 7168 0.90 / 0.90 / 0.89, Zipf 0.94 / 0.93 / 0.87; 128 of 4096 x 6144 0.94 / 0.95 /
    //     0.92, Zipf 0.98 / 0.98 / 0.93; 256 of 4096 x 5120 0.98 / 0.98 / 0.96, Zipf 0.96 / 0.97 / 0.94; 160 of 3072 x 7168 0.98 /
    //     0.99 / 0.96, Zipf 0.97 / 0.97 / 0.93.  300 rows 0.97 to 1.12.  256 columns (32 of 4096 x 7168) 0.89 / 0.91 / 0.92, Zipf
    //     1.12 / 0.99 / 0.95, 258 (43 of 3072 x 7168) 1.11 / 1.03 / 0.98, Zipf 1.13 / 0.97 / 0.96.  2048 x 7168 0.97 to 1.01; 4096 x
    //     4096 0.97 to 1.01, Zipf 0.99 to 1.08.
    const int64_t own = (int64_t)a.N * a.K;
    const bool many_columns = columns >= 3 * kComputeUnits;
    const bool tall = a.N >= 5120 ? own >= (14 << 20) : many_columns && a.N >= 3072 && a.K >= 5120 && own >= (20 << 20);
    if (avg > 256 && a.K >= 2048 && wide_ok && columns >= kComputeUnits
        && ((a.K >= 4096 && own >= (32 << 20)) || (avg >= (many_columns ? 384 : 512) && tall))) return 256;
    // Around 128 rows per expert most experts fit one wide tile of 128 or 160 rows and fetch their weights once, which
    // pays from K = 1024 on if the experts are about equally popular and there are enough of them to fill the chip.  128
    // experts, K = 2048 / 768, the layer at 100 / 112 / 128 / 144 / 160 / 192 rows per expert: 201 / 210 / 224 / 241 / 260 /
    // 280 us with the wide tiles in the first product, 193 / 212 / 232 / 250 / 253 / 264 us on 128-row tiles; Zipf(1.1) at
    // 96 / 128 / 192 219 / 254 / 322 against 187 / 213 / 268, so no further than they win.  With 128 to 255 columns they win on
    // uniform routing (128-row tiles take 0.97 to 1.14 of their time at 128 columns, 1.04 to 1.43 at 192) and lose more under
    // Zipf(1.1) (0.63 to 0.73, 0.65 to 0.90): 32 experts of 2880 / 2880, 1000 tokens of four slots, a layer with the wide tiles
    // in both products / in the first 245 / 267, Zipf 312 / 300; 60 of 2048 / 1408, 2100 tokens 193 / 203, Zipf 252 / 231.
    // (From 256 columns on they win less than they lose as well.  That is left as it is.)
    // Products of up to 512 channels are on the wide tiles from 96 to 192 rows (from 64 to 256 if K is long) at any number of
    // columns, and behind the others there: K / N = 1024 / 512, 128 rows, 8 and 128 experts 25 and 29 us against 13 and 31 on
    // 64-row tiles and 14 and 31 on 128-row tiles (Zipf 34 and 48 against 14 and 34, 14 and 30).  Left as it is as well.
    // From 144 rows on nearly every expert has a second tile, which comes out of the last-level cache.  Uniform routing still
    // wins there, at any shape; under Zipf(1.1) the hot expert's tall tiles are the end of the launch unless an expert's weights
    // are several times an XCD's L2 and there are many columns of tiles.  One product, wide / 128-row tiles: K = 2048, N = 7168
    // (14 MiB and 14 columns per expert), 256 experts, 144 / 160 / 192 / 224 / 250 rows 0.78 / 0.80 / 0.84 / 0.88 / 0.94 (160 rows
    // 826 against 1035 us), Zipf 1.02 / 1.00 / 0.97 / 0.97 / 0.97; 128 experts, 160 / 192 / 224 rows 0.79 / 0.84 / 0.87, Zipf 1.00
    // / 0.94 / 0.92; 64 experts, 160 / 208 rows 0.84 / 0.91, Zipf 1.00 / 1.01.  K = 3072, N = 5120 (15 MiB), 150 / 200 / 250 rows,
    // 128 experts 0.71 / 0.82 / 0.90, Zipf 1.04 / 0.97 / 1.00, 90 experts 0.73 / 0.85 / 0.95, Zipf 1.01 / 1.00 / 0.98.  70 experts
    // of K = 3072, N = 6144 (840 columns) 0.72 / 0.87 / 0.96, Zipf 1.08 / 0.97 / 1.00, so from 896 on, where 56 experts of K = 2048,
    // N = 8192 have 0.71 / 0.86 / 0.92, Zipf 0.99 / 0.95 / 0.91.  Ten MiB (K = 2048, N = 5120) win less and lose more: 128 experts
    // 0.75 / 0.88 / 0.95, Zipf 1.09 / 1.00 / 1.02, 96 experts 0.78 / 0.89 / 0.97, Zipf 1.03 / 1.09 / 1.00, 80 experts 0.82 / 0.99 /
    // 1.05, Zipf 1.13 / 1.01 / 1.03.  With eight columns or fewer per expert (N = 4096, 2048, 1024) 0.79 to 1.07 and 1.01 to
    // 1.15.  144 rows for those.
    const bool fills = narrow || columns >= kComputeUnits;
    const bool beyond = a.K >= 2048 && a.N >= 5120 && own >= (14 << 20) && 2 * columns >= 7 * kComputeUnits;
    const int64_t most = narrow ? 192 : beyond ? 256 : 144;
    // With columns for seven rounds such products are on the wide tiles earlier, since the tall ones are spread among the others:
    // at 40 / 64 / 80 / 100 rows 256 experts of K = 3072, N = 5120 0.96 / 0.90 / 0.88 / 0.86 (Zipf 0.97 / 0.95 / 0.95 / 0.94); of K =
    // 2048, N = 7168 1.00 / 1.02 / 0.95 / 0.94 (0.99 / 0.97 / 0.96 / 0.94), in the layer at 62 / 72 rows 0.99 / 0.97 (0.90 / 0.87);
    // 192 of them 1.00 / 1.01 / 1.01 / 0.97 (1.02 / 0.99 / 0.97 / 0.95), 128 1.00 / 0.99 / 0.98 / 0.96 (1.03 / 0.97 / 0.95 / 0.96);
    // 256 and 160 of K = 2048, N = 8192 1.01 and 1.02 / 1.01 and 1.00 / 1.01 and 1.00 / 0.97 and 0.96 (0.96 and 1.02 / 0.94 and 0.97 /
    // 0.94 and 0.92 / 0.91 and 0.90).
    const int64_t least = narrow ? 96 : beyond && columns >= 7 * kComputeUnits ? (a.K >= 3072 ? 40 : 72) : 112;
    if (avg >= least && avg <= most && a.K >= 1024 && wide_ok && fills) return 256;
    return 128;
}

// The family of one operator call: 0 streaming, 64 / 128 LDS-tiled, 256 weight-streaming tiles, over all experts.
// (Sending the experts above 256 rows of a weight-streaming call to the 128-row tiles measured the same on a Zipf(1.1)
// batch of 32,768 rows, 2149 against 2180 us for the gate_up product, 1136 against 1119 us for the down product, and would
// cost the uniform batches an empty launch.)
static int gemm_family(const GmmArgs& a, bool have_tile_ws)
{
    if (!have_tile_ws || (a.E == 1 && a.R <= 64)) return 0;  // dense, few rows: a workgroup per 64 channels streams
    return tiled_bm(a);
}

// One expert with enough rows and channels for the 256 x 256 tiles to fill the chip: the dense kernel (measured
// against the 128-row tiles: 13 to 17 % faster from 192 tiles on, 20 to 25 % slower at 64 to 128 tiles).
static bool dense_tiles(const GmmArgs& a)
{
    if (a.E != 1 || a.K % 64 != 0) return false;
#ifdef MOE355_DEV_KNOBS
    static const char* force = getenv("MOE355_GEMM");
    if (force && force[0] == 'D') return true;
    if (force && force[0]) return false;
#endif
    return ((a.R + 255) / 256) * ((int64_t)(a.N + 255) / 256) >= 192;
}

// One expert with more rows than the streaming kernel takes in slabs, and 128-row tiles for less than half of the compute
// units (the shared expert of a mixed batch): the 64 x 64 tiles that cut K over their wavefronts.  256 experts of the
// DeepSeek-V3 shape with the shared expert in line, 128 / 192 / 256 / 512 / 1024 tokens 1767 / 1843 / 1882 / 1848 / 1964 us on
// 128-row tiles, 1660 / 1697 / 1738 / 1828 / 1974 on these.  On a side stream the few workgroups of the 128-row tiles hide
// behind the routed products and these do not: 100 / 200 / 400 tokens 1609 / 1712 / 1797 against 1620 / 1738 / 1813.
// Narrow products reach that with many rows, where 64 x 64 tiles pass them around the chip too often (their grid is rounded up
// to eight columns, one for every XCD): us on 128-row tiles / on these at N / K, with the workgroups in brackets, 512 / 7168 at
// 4000 / 6000 rows 52 / 40 (504) and 53 / 57 (752), 512 / 2048 at 6000 / 8000 22.4 / 21.1 (752) and 23.7 / 26.1 (1000), 1024 /
// 4096 at 3000 / 4000 33.0 / 28.6 (752) and 35.1 / 36.4 (1008), 128 / 8192 at 6000 / 16000 58 / 53 (752) and 66 / 130 (2000),
// 64 / 2048 at 4000 / 12000 20.7 / 14.2 (504) and 25.2 / 31.3 (1504).  With a short K there is less to pass: 256 / 256 at 8000 /
// 16000 13.6 / 10.4 (1000) and 16.6 / 18.3 (2000), 512 / 1024 at 8000 17.7 / 18.1 (1000; with SwiGLU 26.7 / 22.4); and with more
// channels: 2048 / 7168 at 2000 63 / 60 (1024), 4096 / 7168 at 1000 66 / 61 (1024).
static bool split_tiles(const GmmArgs& a)
{
    if (a.E != 1 || a.beside || a.K % 64 != 0 || a.R <= 64 || a.R * (int64_t)a.K >= (1ll << 31) || dense_tiles(a)) return false;
    const int64_t workgroups = (a.R + 63) / 64 * ((a.N / 64 + 7) / 8 * 8);
    return ((a.R + 127) / 128) * ((a.N + 255) / 256) < kComputeUnits / 2 && (a.N >= 2048 || workgroups <= (a.K <= 1024 ? 1024 : 768));
}

static size_t tiled_ws_max(int64_t rows, int E)
{
    return (tiled_workspace_bytes(rows, E, 64) + 255) & ~(size_t)255;  // the smallest tile needs the longest tile list
}

// K slabs of the dense few-row product (one expert, at most 64 rows, a long K, too few pairs of tiles to fill
// the chip); 1 = not that case
static int dense_slabs(int64_t R, int K, int N, int E)
{
    const int64_t units = (int64_t)E * (N / 64);
    const int KB = K >> 5;
    if (E != 1 || R > 64 || units >= 256 || units < 1 || KB < 64) return 1;
    int slabs = (int)(512 / units);
    if (slabs > KB / 8) slabs = KB / 8;
    return slabs < 1 ? 1 : slabs;
}

// The tile map that launch_gemm_auto of this product will look for in tile_ws: its number, 0 or 1.
int gemm_tile_specs(int64_t rows, int64_t k, int64_t n, int num_experts, void* tile_ws, TileSpec* specs, int tile_rows)
{
    GmmArgs a = {};
    a.R = rows;
    a.K = (int)k;
    a.N = (int)n;
    a.E = num_experts;
    const int bm = tile_rows ? tile_rows : dense_tiles(a) || split_tiles(a) ? 0 : gemm_family(a, true);
    if (bm) specs[0] = tile_spec(rows, num_experts, bm, tile_ws);
    return bm ? 1 : 0;
}

static int launched(bool ok)
{
    const int rc = launch_status();  // takes the error of a refused step off the thread too
    return ok ? rc : MOE355_E_LAUNCH;
}

template <int EPI>
static int launch_gemm_auto(const GmmArgs& a_in, void* tile_ws, hipStream_t st, void* part_ws = nullptr,
                            size_t part_bytes = 0)
{
    GmmArgs a = a_in;
    hipEvent_t ev0 = t_ev_start, ev1 = t_ev_stop;  // measurement hook: around the GEMM kernels of this call
    t_ev_start = nullptr;
    t_ev_stop = nullptr;
    if (dense_tiles(a)) {
        return launched(launch_dense(EPI, a, st, ev0, ev1));
    }
    if (split_tiles(a)) {
        launch_split(EPI, a, st, ev0, ev1);
        return launch_status();
    }
    const int bm = gemm_family(a, tile_ws != nullptr);
    if (bm) return launched(launch_tiled_any(EPI, bm, a, tile_ws, st, ev0, ev1));
    const int64_t units = (int64_t)a.E * (a.N / 64);
    bool done = false;
    if constexpr (EPI == EPI_I32) {
        // One expert with at most 64 rows (the shared expert of a decode batch: a dense product over a few
        // tokens): too few workgroups for a chip that needs thousands of loads in flight to stream at full rate.
        // K is cut into slabs, one workgroup per (pair of tiles, slab), partial sums added into the zeroed result.
        const int slabs = dense_slabs(a.R, a.K, a.N, a.E);
        if (slabs > 1) {
            const int64_t n4 = a.R * (int64_t)a.N / 4;  // N % 64 == 0
            const dim3 cover((unsigned)((n4 + 255) / 256));
            // with scratch for one plane per slab the partial sums are stored and added up afterwards;
            // without, they are added into the zeroed result with atomics (32 of 47 us at 8 slabs)
            const bool planes = part_ws && part_bytes >= (size_t)slabs * a.R * a.N * 4;
            if (planes) a.acc_part = (int32_t*)part_ws;
            else hipLaunchKernelGGL(zero_i32_kernel, cover, dim3(256), 0, st, a.acc, n4);
            launch_gemm(gmm_stream_kernel<EPI, 4, 4, 3, true>, dim3((unsigned)units, (unsigned)slabs), st, a, ev0,
                        ev1);
            if (planes)
                hipLaunchKernelGGL(slab_sum_kernel, cover, dim3(256), 0, st, a.acc_part, slabs, a.R, a.N, a.gl,
                                   a.acc);
            done = true;
        }
    }
    // Occupancy 3 keeps the SwiGLU epilogue out of scratch memory (131 registers).  With enough units to
    // fill the chip four times over and a short K, the down GEMM lets every wavefront stream a whole unit by
    // itself (no K split, no LDS reduction); otherwise the four wavefronts of a workgroup split K (from
    // K = 2048 on that measured 1.5 % faster on the whole layer, below it the same or slower).
    if (done) {
    } else if (a.gl && a.R < (int64_t)a.E) {
        // fewer rows than experts (a decode batch of a few tokens on the sorted path): a slot per row instead
        // of a place per expert, so that the idle experts cost no dispatch; the workgroup looks up the expert
        // of its slot in the group list, so nothing is requested before that
        a.gl_slots = (int)a.R;
        launch_gemm(gmm_stream_kernel<EPI, 4, 4, 3, false, false>, dim3((unsigned)(a.R * (a.N / 64))), st, a, ev0,
                    ev1);
    } else if (EPI != EPI_SWIGLU && units >= 2048 && a.K < 2048) {
        launch_gemm(gmm_stream_kernel<EPI, 1, 4, 2>, dim3((unsigned)((units + 3) / 4)), st, a, ev0, ev1);
    } else {
        launch_gemm(gmm_stream_kernel<EPI, 4, 4, 3>, dim3((unsigned)units), st, a, ev0, ev1);
    }
    return launch_status();
}

}  // namespace moe355

using namespace moe355;

extern "C" int moe355_profile_next_gemm(void* start_event, void* stop_event)
{
    if ((start_event == nullptr) != (stop_event == nullptr)) return MOE355_E_ARG;
    t_ev_start = (hipEvent_t)start_event;
    t_ev_stop = (hipEvent_t)stop_event;
    return MOE355_OK;
}

extern "C" const char* moe355_gmm_kernel_name(int epilogue, int64_t rows, int64_t k, int64_t n, int num_experts)
{
    if (rows <= 0 || k <= 0 || n <= 0 || num_experts <= 0 || epilogue < 0 || epilogue > 2) return "";
    GmmArgs a = {};
    a.R = rows;
    a.K = (int)k;
    a.N = (int)n;
    a.E = num_experts;
    if (dense_tiles(a)) return "gmm_dense_kernel";
    if (split_tiles(a)) return "gmm_split_kernel";
    const int bm = gemm_family(a, true);  // as launch_gemm_auto decides
    if (bm == 128 && epilogue == EPI_DEQUANT && resident_supported(a)) return "gmm_resident_kernel";
    return bm == 256 ? "gmm_wide_kernel" : bm ? "gmm_tiled_kernel" : "gmm_stream_kernel";
}

extern "C" int moe355_gmm_tile_rows(int64_t rows, int64_t k, int64_t n, int num_experts)
{
    if (rows <= 0 || k <= 0 || n <= 0 || num_experts <= 0) return 0;
    GmmArgs a = {};
    a.R = rows;
    a.K = (int)k;
    a.N = (int)n;
    a.E = num_experts;
    return dense_tiles(a) ? 256 : split_tiles(a) ? 64 : gemm_family(a, true);
}

extern "C" int moe355_format_cast_nz(const int8_t* w, int layout, int64_t num_experts, int64_t n, int64_t k,
                                     int8_t* out, void* stream)
{
    if (num_experts <= 0 || n <= 0 || k <= 0 || !w || !out) return MOE355_E_ARG;
    if (layout != MOE355_W_ENK && layout != MOE355_W_EKN) return MOE355_E_ARG;
    if (n % 32 != 0 || k % 32 != 0) return MOE355_E_SHAPE;
    if (((uintptr_t)w & 15) || ((uintptr_t)out & 15)) return MOE355_E_SHAPE;
    const int64_t total = num_experts * n * k / 16;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipStream_t st = (hipStream_t)stream;
    if (layout == MOE355_W_ENK)
        hipLaunchKernelGGL(format_cast_nz_kernel<MOE355_W_ENK>, dim3((unsigned)blocks), dim3(256), 0, st, w,
                           num_experts, n, k, out);
    else
        hipLaunchKernelGGL(format_cast_nz_kernel<MOE355_W_EKN>, dim3((unsigned)blocks), dim3(256), 0, st, w,
                           num_experts, n, k, out);
    return launch_status();
}

int moe355::gmm_i32_impl(const int8_t* x, const int8_t* weight_nz, const int64_t* group_list, int group_list_type,
                         int64_t rows, int64_t k, int64_t n, int num_experts, int32_t* acc, void* workspace,
                         size_t workspace_bytes, void* stream, bool beside)
{
    int rc = check_gmm(x, weight_nz, group_list, group_list_type, rows, k, n, num_experts);
    if (rc != MOE355_OK) return rc;
    if (rows == 0) return MOE355_OK;
    if (!acc || ((uintptr_t)acc & 15)) return MOE355_E_ARG;
    // the scratch is optional here: without enough of it for the tile map the streaming kernel is used, and
    // what lies behind the tile map serves the partial sums of a product that cuts K into slabs
    const size_t map_bytes = (tiled_ws_max(rows, num_experts) + 255) & ~(size_t)255;
    void* tile_ws = (workspace && !((uintptr_t)workspace & 255) && workspace_bytes >= map_bytes) ? workspace : nullptr;
    void* part_ws = (tile_ws && workspace_bytes > map_bytes) ? (char*)workspace + map_bytes : nullptr;
    const size_t part_bytes = part_ws ? workspace_bytes - map_bytes : 0;
    GmmArgs a = {};
    a.x = x;
    a.w = weight_nz;
    a.gl = group_list;
    a.gl_type = group_list_type;
    a.R = rows;
    a.K = (int)k;
    a.N = (int)n;
    a.E = num_experts;
    a.acc = acc;
    a.beside = beside;
    return launch_gemm_auto<EPI_I32>(a, tile_ws, (hipStream_t)stream, part_ws, part_bytes);
}

extern "C" int moe355_gmm_i32(const int8_t* x, const int8_t* weight_nz, const int64_t* group_list,
                              int group_list_type, int64_t rows, int64_t k, int64_t n, int num_experts, int32_t* acc,
                              void* workspace, size_t workspace_bytes, void* stream)
{
    return gmm_i32_impl(x, weight_nz, group_list, group_list_type, rows, k, n, num_experts, acc, workspace,
                        workspace_bytes, stream, false);
}

extern "C" size_t moe355_gmm_i32_workspace(int64_t rows, int64_t n, int64_t k, int num_experts)
{
    if (rows <= 0 || n <= 0 || num_experts <= 0) return 256;
    size_t bytes = (tiled_ws_max(rows, num_experts) + 255) & ~(size_t)255;
    const int slabs = dense_slabs(rows, (int)k, (int)n, num_experts);
    if (slabs > 1) bytes += (size_t)slabs * rows * n * 4;  // one plane of partial sums per slab
    return bytes;
}

// where the tile maps lie in the gate_up product's workspace: behind the fp32 SwiGLU values
void* moe355::gmm1_tile_ws(void* workspace, int64_t rows, int64_t n)
{
    return (char*)workspace + (((size_t)rows * (size_t)(n / 2) * 4 + 255) & ~(size_t)255);
}

extern "C" size_t moe355_gmm1_swiglu_quant_workspace(int64_t rows, int64_t n, int64_t k, int num_experts)
{
    (void)k;
    (void)num_experts;
    if (rows <= 0 || n <= 0) return 256;
    return (((size_t)rows * (size_t)(n / 2) * 4 + 255) & ~(size_t)255) + tiled_ws_max(rows, num_experts);
}

// a few milliseconds; nobody may ask for more, so that a launch whose workgroups do not meet ends
constexpr int kMeetLooks = 4096;
static thread_local int t_meet_looks = kMeetLooks;

int moe355::take_meeting_looks()
{
    const int looks = t_meet_looks;
    t_meet_looks = kMeetLooks;
    return looks;
}

extern "C" int moe355_next_meeting_looks(int looks)
{
    if (looks < 0) return MOE355_E_ARG;
    t_meet_looks = looks < kMeetLooks ? looks : kMeetLooks;
    return MOE355_OK;
}

// Whether the column workgroups of the gate_up product's tiles meet.  A tile whose columns do not all start in the same round of
// workgroups makes the first of them wait for the rest, holding their place: so a number of columns that divides the places of an
// XCD (64 of the 128-row tiles, 32 of the wide ones) is what matters.  The layer with / without, uniform routing (Zipf(1.1)),
// rows per expert in brackets:
//   - dividing: 8 columns, 64 and 128 experts of 2048 / 1024 (18 to 160) 0.99 .. 0.94 (1.01 .. 0.95); 4 columns, 256 of 2048 / 512 (9 to
//     160) 1.00 .. 0.92 (0.97 .. 0.93), 64 of 1024 / 512 0.99 .. 0.94 (0.97 .. 0.92); 16 columns, 256 of 7168 / 2048 (6 and 16) 0.98 and
//     0.96 (0.97 at 16), 64 of 4096 / 2048 (12 and 36) 1.00 and 0.95 (1.00 and 0.96), 8 of 2048 / 2048 (40 / 250 / 1000) 1.01 / 0.97 / 0.97
//     (1.01 / 0.94 / 0.97); 2 columns, 64 of 1024 / 256, 128 of 2048 / 256, 256 and 32 of 4096 / 256 (9 to 48) 0.98 .. 0.95 (0.99 .. 0.95); one,
//     64 of 2048 / 128 (48) 0.96 (0.93);
//   - others: 6 columns, 128 of 2048 / 768 (54 / 100 / 200 / 300) 0.98 / 0.99 / 0.96 / 0.94 (0.97 / 0.99 / 0.96 / 0.96), 256 of them (18 / 48 /
//     100 / 300) 1.03 / 0.97 / 0.98 / 1.00 (1.00 / 0.99 / 0.96 / 0.99); 11 columns, 60 of 2048 / 1408 (30 / 64 / 128 / 300) 0.98 / 0.96 /
//     0.97 / 0.95 (1.03 / 0.98 / 1.01 / 0.98), 8 of 1024 / 1408 (250 to 2000) 0.96 .. 0.92; 12 columns of 12 and 16 MB an expert, 64 of
//     4096 / 1536 (18 / 36 / 300 / 600) 1.07 / 1.07 / 1.00 / 0.98 (1.00 / 0.99 / 0.99 / 1.00), 128 of them (9 / 36 / 300) 1.02 / 1.02 / 1.00
//     (1.03 / 0.98 / 0.99); 23 columns, 32 of 2880 / 2880 (36 / 60 / 300 / 600) 0.98 / 1.00 / 1.05 / 1.15 (1.04 / 0.99 / 1.00 / 1.12).  So from
//     48 rows on, up to 12 columns and 8 MB.
//   - a launch with workgroups for more than two and up to three per compute unit (128 of 2048 / 768: 768) loses on 128-row tiles, which
//     fill a round and a half (9 / 18 / 27 / 36 rows 1.06 / 1.04 / 1.02 / 1.01, Zipf(1.1) 0.98 / 0.99 / 1.01 / 0.99), and wins on tiles of
//     64 rows, three of which fit a compute unit: 0.99 / 0.97 / 0.95 / 0.94 (0.96 / 0.94 / 0.95 / 0.98; Zipf(0.8) 0.98 / 1.01 / 0.96 / 0.97),
//     at 48 and 60 rows 0.99 and 0.94 (0.99 and 0.97; 1.00 and 1.00).  The same at 18 / 36 / 60 rows of 128 of 2048 / 640 0.96 / 0.93 / 0.90
//     (1.01 / 0.95 / 0.96; Zipf(0.8) 0.96 at 18), 128 of 3072 / 640 0.98 / 0.96 / 0.96 (0.99 / 0.96 / 0.98), 96 of 2560 / 768 0.97 / 0.95 /
//     0.90 (0.95 / 0.95 / 0.97), 96 of 2048 / 896 0.96 / 0.94 / 0.93 (1.00 / 0.99 / 0.97), 256 of 4096 / 384 0.96 / 0.95 / 1.00 (0.90 / 0.93 /
//     0.99), 64 of 1024 / 1536 0.94 / 0.89 / 0.91 (0.94 / 0.97 / 0.97), 64 of 1536 / 1280 0.97 / 0.94 / 0.94 (0.96 / 0.96 / 0.97), at 18 and 36 of
//     256 of 2048 / 384 0.96 and 0.91 (0.92 and 0.98), 100 of 2048 / 768 0.97 and 0.95 (1.05 and 0.91), at 9 of five of them 0.97 .. 0.98
//     (0.95 .. 0.97): 1.5 to 3.9 MB an expert.  Not with 12 MB, whose hot experts read them again for every tile (64 of 4096 / 1536, 36 / 48 / 60
//     rows under Zipf(1.1) 1.06 / 1.08 / 1.09); between 4 and 12 MB nothing was measured.  Up to 48 columns, half of the 96 places of an
//     XCD, so that two launches can wait there: 30 of 768 / 2304 (18 columns) at 36 and 60 rows 0.93 and 0.88 (0.94 and 0.94), 32 of 768 /
//     2560 0.92 and 0.98 (1.03 and 0.98), 24 of 512 / 4096 (32) 0.92 and 0.96 (0.97 and 0.97), 16 of 384 / 5120 (40) 0.81 (0.90) at 60.
//   - wide tiles, 8 columns of 512 channels, 64 experts of 7168 / 2048 (40 / 64 / 96 / 128 / 160 / 200) 0.98 / 0.98 / 0.97 / 0.96 / 0.98 / 1.00
//     (0.98 / 0.97 / 0.98 / 0.98 / 1.04 / 0.99), 256 of them (47 / 94 / 128) 0.94 / 0.95 / 1.00; 4 columns, 64 of 4096 / 1024 (64 / 128 / 200)
//     0.97 / 0.95 / 0.99 (0.99 / 0.97 / 0.98); 3 columns, 128 of 2048 / 768 (125) 0.95 (0.98), 160 of 4096 / 768 (40 / 100 / 160) 0.94 / 0.96
//     / 1.00 (0.99 / 0.97 / 0.98); 6 columns, 128 of 4096 / 1536 (64 / 80 / 112 / 160) 1.03 / 1.04 / 1.03 / 1.08 (1.00 / 0.99 / 1.00 / 1.02);
//     10 columns, 128 of 5120 / 2560 (40 / 96 / 128 / 160) 1.00 / 1.02 / 1.02 / 1.05 (0.98 / 1.01 / 1.02 / 1.00); 8 columns again, 64 and
//     16 of 4096 / 2048 (100) 0.94 and 0.95 (1.00 and 1.03; Zipf(0.8) 1.00 with 16).  So up to 4 columns and with 8, to 144 rows.
//   - beside a shared expert on its side stream, whose workgroups hold places too: 128 of 2048 / 768, 300 / 777 / 2000 / 8192 tokens 1.00 /
//     0.97 / 0.94 / 0.93; 256 of 7168 / 2048, 512 / 1000 / 2048 / 4096 0.99 / 0.95 / 0.99 / 0.97; 64 of 2048 / 2048, 500 / 1000 / 4000 0.95 / 0.94 /
//     0.96: as without.
MeetingPlan moe355::meeting_plan(int64_t rows, int64_t k, int64_t n, int num_experts)
{
    GmmArgs a = {};
    a.R = rows;
    a.K = (int)k;
    a.N = (int)n;
    a.E = num_experts;
    // (the launch that builds the maps clears the words)
    if (dense_tiles(a) || split_tiles(a) || !one_launch_map(rows, num_experts)) return {};
    const int bm = gemm_family(a, true), columns = (a.N / 2 + 127) / 128;
    const int64_t avg = rows / num_experts, own = n * k;
    const MeetingPlan yes = {bm, columns};
    if (bm == 256) {
        const int wide = (columns + 1) / 2;
        return (wide <= 4 || wide == 8) && avg <= 144 ? yes : MeetingPlan{};
    }
    if (bm == 0) return {};
    if (columns <= 16 && (columns & (columns - 1)) == 0) return yes;
    const int64_t least = (int64_t)num_experts * columns;
    if (bm == 128 && least > 2 * kComputeUnits && least <= 3 * kComputeUnits && own <= (4 << 20) && avg < 64 && columns <= 48)
        return {64, columns};
    return columns <= 12 && own <= (8 << 20) && avg >= 48 ? yes : MeetingPlan{};
}

extern "C" int moe355_meeting_tile_rows(int64_t rows, int64_t k, int64_t n, int num_experts)
{
    if (rows <= 0 || k <= 0 || n <= 0 || num_experts <= 0) return 0;
    return moe355::meeting_plan(rows, k, n, num_experts).tile_rows;
}

// The shared expert's gate_up product in line, on the dense tiles.  Without the meeting its int32 sums pass through memory (67 MB each
// way for 4096 rows of 4096 channels; the product and the launch that quantises 109 + 25 us, together 117).  The layer without / with,
// us: 256 experts of 7168 / 2048, 4096 / 5000 / 6000 / 7000 / 8192 tokens 2641 / 2855 / 3328 / 3828 / 4519 and 2617 / 2839 / 3289 / 3799 /
// 4500, Zipf(1.1) 4096 2591 and 2557, int4 4096 2713 and 2698; 64 experts of 2048 / 2048, 4096 / 8000 tokens 674 / 1174 and 656 / 1142, of
// 4096 / 1024, 8192 tokens 1214 and 1198.  The columns need not divide an XCD's 32 places here (64 of 4096 / 1536, 4096 / 7000 tokens
// 1014 / 1596 and 1000 / 1579; 2048 / 2816, 4500 1071 and 1052; 7168 / 2560, 4096 2537 and 2532; 7168 / 1408, 8192 2973 and 2959), but
// those of a row of tiles must all have a place there: dense_split leaves out the wide rectangles (8 experts of 2048 / 512 with 32000
// tokens of 4224 channels, 40192 of 5120 and, with 1024, 64768 of 8192: 1826 / 2383 / 4164 and 1494 / 1846 / 2894).  64 are what a
// wavefront looks at at once.
int moe355::shared_meeting_columns(int64_t rows, int64_t k, int64_t n)
{
    GmmArgs a = {};
    a.R = rows;
    a.K = (int)k;
    a.N = (int)n;
    a.E = 1;
    const int64_t columns = (n / 2 + 127) / 128;
    return columns <= 64 && dense_tiles(a) ? (int)columns : 0;
}

extern "C" int moe355_shared_meeting_columns(int64_t rows, int64_t k, int64_t n, int* on_an_xcd)
{
    const int columns = rows <= 0 || k <= 0 || n <= 0 ? 0 : moe355::shared_meeting_columns(rows, k, n);
    if (on_an_xcd) *on_an_xcd = columns ? dense_split(rows, columns, true).pn : 0;
    return columns;
}

int moe355::shared_meeting_impl(const int8_t* x, const int8_t* weight_nz, const float* weight_scale, const float* x_scale,
                                const int64_t* group_list, int64_t rows, int64_t k, int64_t n, float limit, uint32_t* meet,
                                int looks, int8_t* out, float* out_scale, void* stream)
{
    int rc = check_gmm(x, weight_nz, group_list, MOE355_GL_CUMSUM, rows, k, n, 1);
    if (rc != MOE355_OK) return rc;
    if (((uintptr_t)weight_scale & 15) || ((uintptr_t)out & 15)) return MOE355_E_SHAPE;
    GmmArgs a = {};
    a.x = x;
    a.w = weight_nz;
    a.gl = group_list;
    a.gl_type = MOE355_GL_CUMSUM;
    a.R = rows;
    a.K = (int)k;
    a.N = (int)n;
    a.E = 1;
    a.row_scale = x_scale;
    a.ch_scale = weight_scale;
    a.limit = limit;
    a.meet = meet;
    a.meet_looks = looks;
    a.q = out;
    a.q_scale = out_scale;
    return launched(launch_dense(EPI_MEET_SHARED, a, (hipStream_t)stream, nullptr, nullptr));
}

int moe355::gmm1_impl(const int8_t* x, const int8_t* weight_nz, const int8_t* const* weight_list,
                      const float* weight_scale, const float* const* scale_list, const float* x_scale,
                      const int64_t* group_list, int group_list_type, int64_t rows, int64_t k, int64_t n,
                      int num_experts, float swiglu_limit, int8_t* out, float* out_scale, void* workspace,
                      size_t workspace_bytes, void* stream, const int32_t* row_src, bool tiles_ready, const MeetingPlan& plan,
                      uint32_t* meet)
{
    const void* wany = weight_list ? (const void*)weight_list : (const void*)weight_nz;
    int rc = check_gmm(x, wany, group_list, group_list_type, rows, k, n, num_experts);
    if (rc != MOE355_OK) return rc;
    if (rows == 0) return MOE355_OK;
    if ((!weight_scale && !scale_list) || !x_scale || !out || !out_scale) return MOE355_E_ARG;
    if (((uintptr_t)weight_scale & 15) || ((uintptr_t)out & 3)) return MOE355_E_SHAPE;
    if (!workspace || ((uintptr_t)workspace & 255) ||
        workspace_bytes < moe355_gmm1_swiglu_quant_workspace(rows, n, k, num_experts))
        return MOE355_E_WORKSPACE;
    hipStream_t st = (hipStream_t)stream;
    const int I = (int)(n / 2);
    float* y = (float*)workspace;
    GmmArgs a = {};
    a.x = x;
    a.w = weight_nz;
    a.w_list = weight_list;
    a.gl = group_list;
    a.gl_type = group_list_type;
    a.R = rows;
    a.K = (int)k;
    a.N = (int)n;
    a.E = num_experts;
    a.row_scale = x_scale;
    a.ch_scale = weight_scale;
    a.s_list = scale_list;
    a.limit = swiglu_limit;
    a.y = y;
    a.row_src = row_src;
    a.tiles_ready = tiles_ready;
    void* tile_ws = gmm1_tile_ws(workspace, rows, n);
    if (tiles_ready && plan.columns) {
        a.meet = meet;
        a.meet_looks = plan.looks;
        a.q = out;
        a.q_scale = out_scale;
        hipEvent_t ev0, ev1;
        take_profile_events(ev0, ev1);
        return launched(launch_tiled_any(EPI_MEET, plan.tile_rows, a, tile_ws, st, ev0, ev1));
    }
    rc = launch_gemm_auto<EPI_SWIGLU>(a, tile_ws, st);
    if (rc != MOE355_OK) return rc;
    launch_swiglu_requant(y, group_list, group_list_type, num_experts, rows, I, out, out_scale, st);
    return launch_status();
}

extern "C" int moe355_gmm1_swiglu_quant(const int8_t* x, const int8_t* weight_nz, const float* weight_scale,
                                        const float* x_scale, const int64_t* group_list, int group_list_type,
                                        int64_t rows, int64_t k, int64_t n, int num_experts, float swiglu_limit,
                                        int8_t* out, float* out_scale, void* workspace, size_t workspace_bytes,
                                        void* stream)
{
    return gmm1_impl(x, weight_nz, nullptr, weight_scale, nullptr, x_scale, group_list, group_list_type, rows, k, n,
                     num_experts, swiglu_limit, out, out_scale, workspace, workspace_bytes, stream);
}

extern "C" int moe355_gmm1_swiglu_quant_gather(const int8_t* x, const float* x_scale, const int32_t* row_token,
                                               const int8_t* weight_nz, const float* weight_scale,
                                               const int64_t* group_list, int group_list_type, int64_t rows,
                                               int64_t k, int64_t n, int num_experts, float swiglu_limit, int8_t* out,
                                               float* out_scale, void* workspace, size_t workspace_bytes, void* stream)
{
    if (rows > 0 && !row_token) return MOE355_E_ARG;
    return gmm1_impl(x, weight_nz, nullptr, weight_scale, nullptr, x_scale, group_list, group_list_type, rows, k, n,
                     num_experts, swiglu_limit, out, out_scale, workspace, workspace_bytes, stream, row_token);
}

extern "C" int moe355_gmm1_swiglu_quant_list(const int8_t* x, const int8_t* const* weight_nz_list,
                                             const float* const* weight_scale_list, const float* x_scale,
                                             const int64_t* group_list, int group_list_type, int64_t rows, int64_t k,
                                             int64_t n, int num_experts, float swiglu_limit, int8_t* out,
                                             float* out_scale, void* workspace, size_t workspace_bytes, void* stream)
{
    if (!weight_nz_list || !weight_scale_list) return MOE355_E_ARG;
    return gmm1_impl(x, nullptr, weight_nz_list, nullptr, weight_scale_list, x_scale, group_list, group_list_type,
                     rows, k, n, num_experts, swiglu_limit, out, out_scale, workspace, workspace_bytes, stream);
}

extern "C" size_t moe355_gmm2_dequant_workspace(int64_t rows, int64_t n, int64_t k, int num_experts)
{
    (void)n;
    (void)k;
    if (rows <= 0 || num_experts <= 0) return 256;
    return tiled_ws_max(rows, num_experts);
}

int moe355::gmm2_impl(const int8_t* x, const int8_t* weight_nz, const int8_t* const* weight_list, const float* scale,
                      const float* const* scale_list, const float* per_token_scale, const int64_t* group_list,
                      int group_list_type, int64_t rows, int64_t k, int64_t n, int num_experts, void* out,
                      int out_dtype, void* workspace, size_t workspace_bytes, void* stream, bool tiles_ready, bool beside)
{
    const void* wany = weight_list ? (const void*)weight_list : (const void*)weight_nz;
    int rc = check_gmm(x, wany, group_list, group_list_type, rows, k, n, num_experts);
    if (rc != MOE355_OK) return rc;
    if (out_dtype != MOE355_DT_BF16 && out_dtype != MOE355_DT_F16) return MOE355_E_UNSUPPORTED;
    if (rows > 0 && (!workspace || ((uintptr_t)workspace & 255) ||
                     workspace_bytes < moe355_gmm2_dequant_workspace(rows, n, k, num_experts)))
        return MOE355_E_WORKSPACE;
    if (rows == 0) return MOE355_OK;
    if ((!scale && !scale_list) || !per_token_scale || !out) return MOE355_E_ARG;
    if (((uintptr_t)scale & 15) || ((uintptr_t)out & 15)) return MOE355_E_SHAPE;
    GmmArgs a = {};
    a.x = x;
    a.w = weight_nz;
    a.w_list = weight_list;
    a.gl = group_list;
    a.gl_type = group_list_type;
    a.R = rows;
    a.K = (int)k;
    a.N = (int)n;
    a.E = num_experts;
    a.row_scale = per_token_scale;
    a.ch_scale = scale;
    a.s_list = scale_list;
    a.out = (uint16_t*)out;
    a.out_f16 = out_dtype == MOE355_DT_F16;
    a.tiles_ready = tiles_ready;
    a.beside = beside;
    return launch_gemm_auto<EPI_DEQUANT>(a, workspace, (hipStream_t)stream);
}

extern "C" int moe355_gmm2_dequant(const int8_t* x, const int8_t* weight_nz, const float* scale,
                                   const float* per_token_scale, const int64_t* group_list, int group_list_type,
                                   int64_t rows, int64_t k, int64_t n, int num_experts, void* out, int out_dtype,
                                   void* workspace, size_t workspace_bytes, void* stream)
{
    return gmm2_impl(x, weight_nz, nullptr, scale, nullptr, per_token_scale, group_list, group_list_type, rows, k, n,
                     num_experts, out, out_dtype, workspace, workspace_bytes, stream);
}

extern "C" int moe355_gmm2_dequant_list(const int8_t* x, const int8_t* const* weight_nz_list,
                                        const float* const* scale_list, const float* per_token_scale,
                                        const int64_t* group_list, int group_list_type, int64_t rows, int64_t k,
                                        int64_t n, int num_experts, void* out, int out_dtype, void* workspace,
                                        size_t workspace_bytes, void* stream)
{
    if (!weight_nz_list || !scale_list) return MOE355_E_ARG;
    return gmm2_impl(x, nullptr, weight_nz_list, nullptr, scale_list, per_token_scale, group_list, group_list_type,
                     rows, k, n, num_experts, out, out_dtype, workspace, workspace_bytes, stream);
}

// ------------------------------------------------------------------ pair order (decode batches)
extern "C" int moe355_gmm_pairs_supported(int64_t num_tokens, int top_k, int64_t n, int64_t k)
{
    return num_tokens > 0 && top_k > 0 && num_tokens * top_k <= kPairMax && n > 0 && k > 0 && n % 64 == 0 && k % 32 == 0;
}

// Whether a batch whose ids come straight from the gate runs in pair order: at most 1024 (token, slot) pairs, up to 12
// per expert, and experts that the bit map of the lookup can hold.  Pair order streams every expert; the sorted path of
// a product of a GiB and more has tiles for the hot ones.  DeepSeek-V3 shape, 70 / 80 / 96 tokens with the shared expert
// in line: uniform routing 1500 / 1541 / 1581 us in pair order, 1575 / 1601 / 1641 us sorted; Zipf(1.1) 506 / 538 / 597
// against 481 / 514 / 549; 128 tokens without it 742 against 457 us.
// An expert's weights are read once for every 32 rows.  From 36 rows per expert on (at 32 half of the experts still take one
// pass) that is what a layer of few experts takes its time for, and beyond 128 MiB of such reads it outweighs the longer
// chain of launches of the tiles; beyond 256 MiB where the pair-order launches take a shared expert along, which costs the
// sorted path 30 us of launches more.  us in pair order / sorted, uniform routing (Zipf(1.1)), experts of H / I, two slots:
//   8 of 1024 / 1408, 440 / 500 tokens 44.5 / 49.1 against 40.5 / 41.0 (44.2 / 48.5 against 46.2 / 46.6);
//   8 of 4096 / 2048, 128 / 192 / 256 tokens 79 / 91 / 117 against 75 / 78 / 78 (89 / 116 / 141 against 74 / 76 / 76), with a
//     shared expert 130 / 160 / 200 tokens 91 / 106 / 119 against 102 / 103 / 106;
//   16 of 2048 / 1408, 256 / 288 / 320 tokens 54.6 / 62.6 / 66.8 against 56.3 / 57.0 / 57.6;
//   16 of 4096 / 2048, 256 / 511 tokens 130 / 214 against 92 / 109 (190 / 317 against 114 / 128);
//   8 of 512 / 256, 511 tokens 22 against 36 (22 against 36).
bool moe355::pair_order_impl(int64_t num_tokens, int top_k, int num_logits, int num_experts, int64_t hidden,
                             int64_t intermediate, bool with_shared)
{
    if (!moe355_gmm_pairs_supported(num_tokens, top_k, 2 * intermediate, hidden) ||
        !moe355_gmm_pairs_supported(num_tokens, top_k, hidden, intermediate) ||
        !moe355_gate_quant_supported(num_tokens, top_k, num_logits) || num_experts <= 0 || num_experts > 2048)
        return false;
    const int64_t pairs = num_tokens * top_k;
    if ((int64_t)num_experts * 2 * intermediate * hidden >= (1ll << 30) && pairs > 768) return false;
    const int64_t weight_bytes = 3 * intermediate * hidden;  // of one expert
    if (pairs >= 36 * (int64_t)num_experts && pairs * weight_bytes / 32 >= (with_shared ? 2ll : 1ll) << 27) return false;
    return pairs < 1024 || pairs / num_experts < 12;
}

extern "C" int moe355_pair_order(int64_t num_tokens, int top_k, int num_logits, int num_experts, int64_t hidden,
                                 int64_t intermediate)
{
    return pair_order_impl(num_tokens, top_k, num_logits, num_experts, hidden, intermediate, false);
}

// whether a hot expert's further blocks of 32 rows are workgroups of their own (pair_places)
static bool blocks_of_their_own(int64_t pairs, int64_t n) { return n / 64 < (pairs < 384 ? 48 : 96); }

// pair order: the places of the grid.
// A place per expert lets a workgroup request its first weight tiles before it has seen a single id, and makes every
// idle expert cost the dispatch of its workgroups plus 32 KiB of weights requested for nothing.  A slot (the kernel
// looks up which expert it belongs to, and requests nothing before) costs one exposed lookup, and nothing for idle
// experts.  The exposed lookup only shows in the workgroups that the chip starts with; later ones run beside others
// that stream.  So, with more than two pairs per expert, the experts whose units are resident first have places and the
// rest have slots; with fewer pairs idle experts are the rule and every place is a slot.  Whole layer of the Qwen3
// shape, places / slots / both: 64 tokens uniform 110.1 / 110.4 / 109.1 us, Zipf(1.1) 90 / 78 / 77 us; 127 tokens
// uniform 113.3 / 116.7 / 113.6 us.
// An expert with more than 32 rows takes several passes over its weights, one after the other.  Where an expert has few
// units (the launch is over after two or three rounds of workgroups) its further blocks of 32 rows become workgroups of
// their own: Qwen3 shape (24 and 32 units), Zipf(1.1), 64 / 100 / 127 tokens 77 / 118 / 135 -> 75 / 86 / 93 us, uniform
// routing unchanged.  From 48 units on the passes hide among the other workgroups until the hot experts have a few blocks
// each: DeepSeek-V3 shape, gate_up product (64 units), Zipf(1.1), 33 / 50 / 64 / 90 tokens of eight slots 345 / 417 / 453 / 589 us
// in passes, 347 / 414 / 448 / 573 in workgroups (uniform 40 / 64 / 96 tokens 1234 / 1467 / 1610 and 1235 / 1468 / 1610); its down
// product (112 units) is the same either way.  32 experts of 2880 / 2880 (90 units), four slots, Zipf(1.1), 96 / 127 / 200 tokens
// 168 / 204 / 269 in passes, 154 / 181 / 234 in workgroups, uniform 148 / 157 / 193 and 148 / 157 / 194.
// Those are the longest workgroups of the launch, and at the end of the grid the chip waits for them; but there are
// places for as many as R pairs could need, and in front of the slots an unused one delays them.  So as many as skewed
// routing usually needs, one for every 56 pairs, run in front and the others at the end.  Qwen3 shape, 40 / 64 / 100 / 127
// tokens, all at the end / so / one for every 32 pairs in front: Zipf(1.1) 67.3 / 75.3 / 86.8 / 94.5 against 64.4 / 71.0 / 81.5
// / 90.5 against 63.7 / 70.8 / 82.4 / 88.6 us, uniform routing 103.2 / 108.0 / 110.2 / 111.5 against 103.3 / 108.0 / 110.3 /
// 111.8 against 103.3 / 108.2 / 110.8 / 112.8.
// In front of slots that start behind places of their own, they cost a lookup that the slots of a short launch have to wait for:
// all at the end / so, 48 / 64 / 127 tokens of eight slots, 128 experts of 512 / 256 (1024 units in both products) uniform 30.0 /
// 30.2 / 30.9 against 33.2 / 33.4 / 34.0, Zipf(1.1) 28.6 / 28.8 / 30.8 against 28.3 / 28.7 / 31.4, 64 experts of 512 / 512 (1024,
// 512) uniform 27.9 / 28.4 / 30.5 against 29.2 / 29.8 / 31.8, Zipf 28.9 / 29.8 / 34.9 against 28.6 / 29.9 / 35.2; 128 experts of
// 1024 / 512 (2048, 2048) uniform 49.1 / 49.9 / 52.3 against 49.6 / 50.4 / 54.3, Zipf 43.2 / 46.2 / 53.6 against 41.1 / 43.6 / 52.2.
// 64 of 2048 / 768 (1536, 2048) uniform 65.7 / 66.7 / 72.2 against 65.8 / 67.2 / 73.6, Zipf 60.5 / 67.8 / 84.8 against 59.8 / 66.8 /
// 83.6; 60 of 2048 / 1408 (2640, 1920), four slots, the down product alone, 40 / 64 / 127 tokens uniform 91.6 / 96.2 / 100.1 against
// 91.3 / 95.9 / 100.3, Zipf 62.7 / 68.9 / 88.3 against 60.6 / 66.5 / 85.2.
// So from 1536 units on (two rounds of the gate_up product's workgroups), and with fewer than 12 pairs per expert, beyond which
// most experts are hot: 60 experts of 2048 / 1408, four slots, 160 / 200 / 250 tokens uniform 102.1 / 105.6 / 110.4 against 102.9 /
// 107.5 / 112.7, Zipf 100.7 / 107.2 / 114.1 against 96.9 / 108.9 / 119.3; 32 of 2880 / 2880, 130 / 200 / 250 tokens uniform 158.5 /
// 190.5 / 243.1 against 159.0 / 194.3 / 240.3, Zipf 183.4 / 226.9 / 267.4 against 184.0 / 232.5 / 271.6.  Without places every
// slot makes that lookup, and nothing waits (256 experts of 1024 / 256, 127 tokens of four slots uniform 47.2 against 46.7, Zipf
// 33.8 against 30.8).
// The lookups hold 2048 experts.
static int pair_places(GmmArgs& a, int resident_units)
{
    a.pair_first = a.E;
    a.pair_slots = a.pair_extra = a.pair_early = 0;
    if (a.E <= kPairExperts) {
        a.pair_first = a.R > 2 * (int64_t)a.E ? resident_units / (a.N / 64) - a.sh_blocks : 0;
        if (a.pair_first > a.E) a.pair_first = a.E;
        if (a.pair_first < 0) a.pair_first = 0;
        const int rest = a.E - a.pair_first;
        a.pair_slots = a.R < (int64_t)rest ? (int)a.R : rest;
        // an expert of c rows has (c - 1) / 32 further blocks: over all experts at most (R - 1) / 32
        if (blocks_of_their_own(a.R, a.N)) a.pair_extra = (int)((a.R - 1) / 32);
        if (a.pair_first == 0 || ((int64_t)a.E * (a.N / 64) >= 1536 && a.R < 12 * (int64_t)a.E))
            a.pair_early = a.R / 56 < a.pair_extra ? (int)(a.R / 56) : a.pair_extra;
    }
    return a.sh_blocks + a.pair_first + a.pair_slots + a.pair_extra;
}

extern "C" size_t moe355_gmm1_swiglu_quant_pairs_workspace(int64_t num_tokens, int top_k, int64_t n)
{
    if (num_tokens <= 0 || top_k <= 0 || n <= 0) return 256;
    return (((size_t)num_tokens * top_k * (size_t)(n / 2) * 4 + 255) & ~(size_t)255);
}

// gate_up GEMM + SwiGLU in pair order: fp32 values to y, and with `out` the re-quantised rows.  The weights are one
// tensor (w.one) or per-expert tensors (w.list and w.scale_list).
extern "C" int moe355_pair_blocks_in_front(int64_t num_pairs, int64_t n, int num_experts)
{
    if (num_pairs <= 0 || num_pairs > kPairMax || n <= 0 || n % 64 || num_experts <= 0) return 0;
    GmmArgs a = {};
    a.R = num_pairs;
    a.N = (int)n;
    a.E = num_experts;
    pair_places(a, 768);
    return a.pair_early;
}

int moe355::gmm1_pairs_impl(const int8_t* x, const float* x_scale, const int32_t* topk_ids, int64_t num_tokens,
                            int top_k, const PairWeights& w, int64_t k, int64_t n, int num_experts, float swiglu_limit,
                            float* y, int8_t* out, float* out_scale, void* stream, const PairShared* shared)
{
    if (num_tokens < 0 || top_k <= 0 || k <= 0 || n <= 0 || num_experts <= 0) return MOE355_E_ARG;
    if (num_tokens == 0) return MOE355_OK;
    if (!moe355_gmm_pairs_supported(num_tokens, top_k, n, k)) return MOE355_E_SHAPE;
    if ((int64_t)num_experts * (n / 64) >= 0x7fffffffLL) return MOE355_E_SHAPE;
    if (!x || !x_scale || !topk_ids || !w.complete() || !y) return MOE355_E_ARG;
    if (((uintptr_t)x & 15) || !w.aligned() || ((uintptr_t)y & 15) || ((uintptr_t)out & 3)) return MOE355_E_SHAPE;
    if (shared && !shared->aligned()) return MOE355_E_SHAPE;
    hipStream_t st = (hipStream_t)stream;
    const int64_t rows = num_tokens * top_k;
    GmmArgs a = {};
    a.x = x;
    a.w = w.one;
    a.ch_scale = w.scale;
    a.w_list = w.list;
    a.s_list = w.scale_list;
    a.R = rows;
    a.K = (int)k;
    a.N = (int)n;
    a.E = num_experts;
    a.row_scale = x_scale;
    a.limit = swiglu_limit;
    a.y = y;
    a.pair_ids = topk_ids;
    a.pair_k = top_k;
    a.pair_gather = 1;
    if (shared) shared->into(a, (int)num_tokens);
    hipEvent_t ev0, ev1;
    take_profile_events(ev0, ev1);
    const int64_t units = (int64_t)pair_places(a, 768) * (n / 64);
    // No more workgroups than two for every compute unit: eight K steps in flight instead of four (the small layer's 64 tokens
    // 27.4 -> 26.6 us a call; with more workgroups the third one of a compute unit is worth more: 128 tokens 29.8 -> 31.2)
    if (units <= 2 * kComputeUnits)
        launch_gemm(gmm_stream_kernel<EPI_SWIGLU, 4, 8, 2, false, true, true>, dim3((unsigned)units), st, a, ev0, ev1);
    else launch_gemm(gmm_stream_kernel<EPI_SWIGLU, 4, 4, 3, false, true, true>, dim3((unsigned)units), st, a, ev0, ev1);
    if (out)
        launch_swiglu_requant(y, nullptr, 0, num_experts, rows + a.sh_rows, (int)(n / 2), out, out_scale, st, rows);
    return launch_status();
}

// down GEMM + dequant in pair order on re-quantised rows (x and per_token_scale), or on the fp32 SwiGLU values of the
// gate_up GEMM (y), which the workgroups then re-quantise themselves
int moe355::gmm2_pairs_impl(const int8_t* x, const float* per_token_scale, const float* y, const PairWeights& w,
                            const int32_t* topk_ids, int64_t num_tokens, int top_k, int64_t k, int64_t n,
                            int num_experts, void* out, int out_dtype, void* stream, const PairShared* shared)
{
    if (num_tokens < 0 || top_k <= 0 || k <= 0 || n <= 0 || num_experts <= 0) return MOE355_E_ARG;
    if (out_dtype != MOE355_DT_BF16 && out_dtype != MOE355_DT_F16) return MOE355_E_UNSUPPORTED;
    if (num_tokens == 0) return MOE355_OK;
    if (!moe355_gmm_pairs_supported(num_tokens, top_k, n, k)) return MOE355_E_SHAPE;
    if (y && !moe355_gmm2_requant_pairs_supported(num_tokens, top_k, n, k, num_experts)) return MOE355_E_SHAPE;
    if ((int64_t)num_experts * (n / 64) >= 0x7fffffffLL) return MOE355_E_SHAPE;
    if (!w.complete() || !topk_ids || !out || (!y && (!x || !per_token_scale))) return MOE355_E_ARG;
    if (((uintptr_t)x & 15) || ((uintptr_t)y & 15) || !w.aligned() || ((uintptr_t)out & 15)) return MOE355_E_SHAPE;
    if (shared && !shared->aligned()) return MOE355_E_SHAPE;
    hipStream_t st = (hipStream_t)stream;
    GmmArgs a = {};
    a.x = x;
    a.y_in = y;
    a.w = w.one;
    a.ch_scale = w.scale;
    a.w_list = w.list;
    a.s_list = w.scale_list;
    a.R = num_tokens * top_k;
    a.K = (int)k;
    a.N = (int)n;
    a.E = num_experts;
    a.row_scale = per_token_scale;
    a.out = (uint16_t*)out;
    a.out_f16 = out_dtype == MOE355_DT_F16;
    a.pair_ids = topk_ids;
    a.pair_k = top_k;
    a.pair_gather = 0;
    if (shared && !y) shared->into(a, (int)num_tokens);
    hipEvent_t ev0, ev1;
    take_profile_events(ev0, ev1);
    // a wavefront per unit when there are enough units and K is short, and the units of an expert come in fours (a
    // workgroup collects the pairs of one expert)
    const bool unsplit = (int64_t)num_experts * (n / 64) >= 2048 && k < 2048 && (n / 64) % 4 == 0;
    const int64_t units = (int64_t)pair_places(a, unsplit ? 2048 : 768) * (n / 64);
    const dim3 by_four((unsigned)((units + 3) / 4));
    if (y) {
        const unsigned lds = (unsigned)(32 * (k + 16));
        auto kernel = gmm_stream_kernel<EPI_DEQUANT, 1, 4, 2, false, true, true, 1, 8>;
        if (k <= 768) kernel = gmm_stream_kernel<EPI_DEQUANT, 1, 4, 2, false, true, true, 3, 3>;
        else if (k <= 1024) kernel = gmm_stream_kernel<EPI_DEQUANT, 1, 4, 2, false, true, true, 2, 4>;
        if (ev0 || ev1) hipExtLaunchKernelGGL(kernel, by_four, dim3(256), lds, st, ev0, ev1, 0, a);
        else hipLaunchKernelGGL(kernel, by_four, dim3(256), lds, st, a);
    } else if (unsplit && units >= 2048) {
        launch_gemm(gmm_stream_kernel<EPI_DEQUANT, 1, 4, 2, false, true, true>, by_four, st, a, ev0, ev1);
    } else if (units <= kComputeUnits) {
        launch_gemm(gmm_stream_kernel<EPI_DEQUANT, 4, 12, 2, false, true, true>, dim3((unsigned)units), st, a, ev0, ev1);
    } else {
        launch_gemm(gmm_stream_kernel<EPI_DEQUANT, 4, 4, 3, false, true, true>, dim3((unsigned)units), st, a, ev0, ev1);
    }
    return launch_status();
}

extern "C" int moe355_gmm1_swiglu_quant_pairs(const int8_t* x, const float* x_scale, const int32_t* topk_ids,
                                              int64_t num_tokens, int top_k, const int8_t* weight_nz,
                                              const float* weight_scale, int64_t k, int64_t n, int num_experts,
                                              float swiglu_limit, int8_t* out, float* out_scale, void* workspace,
                                              size_t workspace_bytes, void* stream)
{
    if (num_tokens > 0 && (!out || !out_scale)) return MOE355_E_ARG;
    if (num_tokens > 0 && (!workspace || ((uintptr_t)workspace & 255) ||
                           workspace_bytes < moe355_gmm1_swiglu_quant_pairs_workspace(num_tokens, top_k, n)))
        return MOE355_E_WORKSPACE;
    return gmm1_pairs_impl(x, x_scale, topk_ids, num_tokens, top_k, PairWeights{weight_nz, weight_scale}, k, n,
                           num_experts, swiglu_limit, (float*)workspace, out, out_scale, stream);
}

extern "C" int moe355_gmm2_dequant_pairs(const int8_t* x, const int8_t* weight_nz, const float* scale,
                                         const float* per_token_scale, const int32_t* topk_ids, int64_t num_tokens,
                                         int top_k, int64_t k, int64_t n, int num_experts, void* out, int out_dtype,
                                         void* stream)
{
    return gmm2_pairs_impl(x, per_token_scale, nullptr, PairWeights{weight_nz, scale}, topk_ids, num_tokens, top_k, k,
                           n, num_experts, out, out_dtype, stream);
}

// gate_up GEMM + SwiGLU in pair order, the fp32 values left as they are (the down GEMM below re-quantises them)
extern "C" int moe355_gmm1_swiglu_pairs(const int8_t* x, const float* x_scale, const int32_t* topk_ids,
                                        int64_t num_tokens, int top_k, const int8_t* weight_nz,
                                        const float* weight_scale, int64_t k, int64_t n, int num_experts,
                                        float swiglu_limit, float* y, void* stream)
{
    return gmm1_pairs_impl(x, x_scale, topk_ids, num_tokens, top_k, PairWeights{weight_nz, weight_scale}, k, n,
                           num_experts, swiglu_limit, y, nullptr, nullptr, stream);
}

// the form of the down GEMM that re-quantises: a wavefront per unit (many units, a short K) and 32 rows of K + 16
// bytes in LDS for each of the two workgroups of a compute unit
extern "C" int moe355_gmm2_requant_pairs_supported(int64_t num_tokens, int top_k, int64_t n, int64_t k, int num_experts)
{
    if (!moe355_gmm_pairs_supported(num_tokens, top_k, n, k) || num_experts <= 0) return 0;
    const int64_t units = (int64_t)num_experts * (n / 64);
    if (!(units >= 2048 && k < 2048 && (n / 64) % 4 == 0 && k % 4 == 0 && 32 * (k + 16) <= 48 * 1024)) return 0;
    // Every workgroup of an expert quantises all its rows again.  Rows of up to 768 values go three at a time through a
    // wavefront's registers, and then it pays up to eight rows per expert.  128 experts of 2048 x 768, the layer in us with
    // the launch of its own / one row at a time / three: uniform routing 24 / 48 / 64 / 96 / 127 tokens of eight slots 92.7 /
    // 108.0 / 109.1 / 111.9 / 114.0 against 91.3 / 105.9 / - / - / - against 91.3 / 105.7 / 106.9 / 109.2 / 111.4; Zipf(1.1), 16
    // / 32 / 50 / 64 / 96 / 127 tokens 47.9 / 54.9 / - / 77.4 / 90.3 / 98.2 against 46.2 / 58.5 / 72.4 / - / - / - against 45.0 /
    // 56.0 / 70.2 / 76.3 / 88.6 / 94.8.  Shorter rows gain less: 128 experts of 2048 x 320, 64 / 127 tokens uniform 60.7 / 63.9
    // against 59.6 / 62.1, Zipf 48.0 / 58.6 against 50.3 / 59.5; of 1024 x 256, 160 tokens of four slots 36.4 against 34.1, Zipf
    // 35.2 against 36.7.  Longer rows: up to three and a half rows per expert (two at a time up to 1024 values, one beyond).  Two at
    // a time it would pay further: 64 experts of 2048 x 1024, 28 / 64 / 112 tokens 88.2 / 92.1 / 95.8 against 84.1 / 86.9 / 91.4, Zipf
    // 65.8 / 85.2 / 102.1 against 66.0 / 81.2 / 98.2; left as it is.
    // Three and a half rows are the limit for experts of many channels with few pairs as well, whose hot ones take their rows
    // in passes: there the re-quantisation stands in front of every pass.  32 experts of 4096 x 768, four slots, Zipf(1.1), 40 /
    // 64 / 80 tokens 69.4 / 75.3 / 84.3 against 70.9 / 80.6 / 92.0 (uniform 65.6 / 66.2 / 66.7 against 63.0 / 64.1 / 64.8), 112
    // tokens, which is more than 384 pairs, 80.2 against 78.0.
    const int64_t pairs = num_tokens * top_k;
    return pairs * 2 <= (k <= 768 && blocks_of_their_own(pairs, n) ? 16 : 7) * (int64_t)num_experts;
}

extern "C" int moe355_gmm2_requant_dequant_pairs(const float* y, const int8_t* weight_nz, const float* scale,
                                                 const int32_t* topk_ids, int64_t num_tokens, int top_k, int64_t k,
                                                 int64_t n, int num_experts, void* out, int out_dtype, void* stream)
{
    if (num_tokens > 0 && !y) return MOE355_E_ARG;
    return gmm2_pairs_impl(nullptr, nullptr, y, PairWeights{weight_nz, scale}, topk_ids, num_tokens, top_k, k, n,
                           num_experts, out, out_dtype, stream);
}
