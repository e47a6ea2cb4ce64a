// Grouped int8 GEMM for many rows per expert (prefill): MFMA-bound, LDS-staged tokens.
//
// Workgroup tile: BM tokens x 256 channels, K consumed 64 at a time.  The four wavefronts own 64
// channels each (two 32-channel storage tiles: for the gate_up GEMM a gate tile and its up tile,
// so SwiGLU pairs meet in one lane).  Weights never touch LDS: 16 channels x 64 K of a storage tile are one MFMA A
// operand and are loaded straight into registers, two iterations ahead.  Tokens are shared by the
// four wavefronts: global -> registers (three iterations ahead) -> LDS in MFMA-operand order
// (every B operand, 16 tokens x 64 K, is one conflict-free 1 KiB ds_read_b128 sweep) -> MFMA.
//
// All tiles of this file multiply with v_mfma_i32_16x16x64_i8.  v_mfma_i32_32x32x32_i8 takes the same operand bytes and
// cycles per product but moves four times the accumulators, and these kernels run at the power limit: it only lowers the
// clock.  Loops on int8 values of a normal distribution of width 32, 32x32x32 against 16x16x64, after the first 2 ms:
// operands in registers 3.45 POP/s at 1.80 GHz against 4.09 at 2.09; four token operands from LDS per weight pair 3.16 at
// 1.65 against 3.63 at 1.94; weights from L2 as well 2.67 at 1.59 against 2.97 at 1.88 (zeros: 4.8 at 2.4 GHz for both).
// The kernels back to back: dense 4096 x 7168 x 4096 127.6 -> 115.6 us; 256 experts of 128 rows, gate_up 7168 / 4096 and
// its re-quantisation 1550 -> 1488, down 2048 / 7168 805 -> 782; 128 experts of 512 rows, 2048 / 1536 336 -> 329, 768 / 2048
// 179 -> 174.  Where the weights' way from HBM decides it is the same (128 experts of 48 rows).
// Tiles are enumerated (expert, row block) by a small map kernel from the group list; the 1-D
// grid is remapped so that all column blocks of a row block, and the row blocks of one expert,
// run on the same XCD (workgroup i goes to XCD i % 8) and share its L2.
#include <hip/hip_ext.h>

#include "gmm_common.h"
#include <type_traits>

#include "gmm_tiled.h"
#include "tile_map.h"

namespace moe355 {

__global__ __launch_bounds__(256) void tile_map_kernel(const int64_t* __restrict__ gl, int gl_type, int E, TileSpec spec)
{
    __shared__ int32_t part_rows[16];
    __shared__ int32_t part_tiles[16];
    build_tile_map(
        [&](int e) -> int64_t {
            const int64_t m = (gl_type == MOE355_GL_COUNT) ? gl[e] : gl[e] - (e > 0 ? gl[e - 1] : 0);
            return m < 0 ? 0 : m;
        },
        E, spec, part_rows, part_tiles);
}

constexpr int kBN = 256;  // channels per workgroup (4 wavefronts x 2 storage tiles)
constexpr int kBK = 64;   // K per pipeline stage (one MFMA K step)

// LDS of one workgroup: RING token stages of the tallest tile, reused by the epilogue patches
template <int EPI, int BMT, int RING>
struct TiledLds {
    static constexpr int BM = 32 * BMT;
    static constexpr int STAGE_BYTES = BM * kBK;               // tokens of one stage in LDS
    static constexpr int ROWB = 128 + 16;                      // epilogue patch: bytes per token row (padded)
    static constexpr int PATCHES = (EPI == EPI_I32) ? 2 : 1;   // 32-row patches per wavefront in the epilogue
    static constexpr int EPI_BYTES = 4 * PATCHES * 32 * ROWB;
    static constexpr int SCALES = RING * STAGE_BYTES > EPI_BYTES ? RING * STAGE_BYTES : EPI_BYTES;  // token scales, then channel scales
    static constexpr int BYTES = SCALES + (EPI == EPI_I32 ? 0 : (BM + kBN) * 4);
};

// Epilogue of one wavefront: BMT blocks of 32 tokens x two 32-channel storage tiles (nb0, nb1) out of the MFMA
// accumulators: acc[t][b] holds channels 16 (t % 2) .. + 15 of storage tile t / 2 for tokens 16 b .. + 15.  There a lane
// owns one token and runs of four channels; written like that every store would touch 64 different cache lines.  The
// wavefront instead turns 32 tokens at a time through a private LDS patch (token-major, 128 data bytes per
// token and tile) and stores whole 128-byte row segments: 8 lanes per token row.
// FLAG, SwiGLU epilogue: the clamp is compiled in (as compares and selects it costs 8 of about 50 vector
// instructions per output, and the epilogue is bound by their number); dequant epilogue: the output is fp16
// instead of bf16.  The caller branches once.
// IN_LDS: the scales lie in LDS, rs_lds by row of the tile and cs_lds by channel of the wavefront's two storage tiles.
template <int EPI, int BMT, bool FLAG, bool IN_LDS>
__device__ __forceinline__ void tiled_epilogue_body(const GmmArgs& a, int e, v4i (&acc)[4][2 * BMT], int64_t row0,
                                                    int64_t row_end, int nb0, int nb1, int8_t* patch, int lane,
                                                    const float* rs_lds, const float* cs_lds)
{
    constexpr int ROWB = TiledLds<EPI, BMT, 3>::ROWB;
    const int tok = lane & 15;
    const int run = 4 * (lane >> 4);  // this lane's first channel inside a group of 16
    v4f s0[2], s1[2];
    if constexpr (EPI != EPI_I32 && IN_LDS) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            s0[t] = *(const v4f*)(cs_lds + 16 * t + run);
            s1[t] = *(const v4f*)(cs_lds + 32 + 16 * t + run);
        }
    } else if constexpr (EPI != EPI_I32) {
        const float* cs = expert_scales(a, e);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            s0[t] = gload4f(cs + nb0 * 32 + 16 * t + run);
            s1[t] = gload4f(cs + nb1 * 32 + 16 * t + run);
        }
    }
    // every token scale is requested before the first store: the memory counter retires in order, so a load
    // behind a block's stores would wait for their acknowledgement, once per token block.  The rows' tokens are looked up
    // in one go: a branch per row would wait for each look-up before it requests the next.
    float rs_all[2 * BMT];
    if constexpr (EPI != EPI_I32 && IN_LDS) {
#pragma unroll
        for (int b = 0; b < 2 * BMT; ++b) rs_all[b] = rs_lds[b * 16 + tok];
    } else if constexpr (EPI != EPI_I32) {
        int32_t at[2 * BMT];  // rows are fewer than 2^31
#pragma unroll
        for (int b = 0; b < 2 * BMT; ++b) {
            const int64_t row = row0 + b * 16 + tok;
            at[b] = (int32_t)(row < row_end ? row : row_end - 1);
        }
        if (a.row_src) {
#pragma unroll
            for (int b = 0; b < 2 * BMT; ++b) at[b] = a.row_src[at[b]];
        }
#pragma unroll
        for (int b = 0; b < 2 * BMT; ++b) rs_all[b] = a.row_scale[at[b]];
    } else {
#pragma unroll
        for (int b = 0; b < 2 * BMT; ++b) rs_all[b] = 0.0f;
    }
    // ... and has arrived before it: the stores below sit behind "row < row_end" branches, and a wait for a
    // load that is still in flight at that point would have to assume that none of them was issued, which
    // turns it into a wait for every store of the block before
#pragma unroll
    for (int b = 0; b < 2 * BMT; ++b) asm volatile("" : "+v"(rs_all[b]));
#pragma unroll
    for (int b = 0; b < BMT; ++b) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float rs = rs_all[2 * b + h];
            int8_t* const prow = patch + (16 * h + tok) * ROWB;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const v4i c0 = acc[t][2 * b + h], c1 = acc[2 + t][2 * b + h];
                const int ch = 16 * t + run;  // first of this lane's four channels inside the storage tile
                if constexpr (EPI == EPI_I32) {
                    *(v4i*)(prow + ch * 4) = c0;
                    *(v4i*)(prow + 32 * ROWB + ch * 4) = c1;
                } else if constexpr (EPI == EPI_DEQUANT) {
                    v4u16 o0, o1;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        o0[j] = f32_to_half<FLAG ? MOE355_DT_F16 : MOE355_DT_BF16>(((float)c0[j] * rs) * s0[t][j]);
                        o1[j] = f32_to_half<FLAG ? MOE355_DT_F16 : MOE355_DT_BF16>(((float)c1[j] * rs) * s1[t][j]);
                    }
                    // both tiles are adjacent in the output row: 64 bf16 = 128 bytes per token
                    *(v4u16*)(prow + ch * 2) = o0;
                    *(v4u16*)(prow + 64 + ch * 2) = o1;
                } else {
                    v4f yv;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        float gg = ((float)c0[j] * rs) * s0[t][j];
                        float uu = ((float)c1[j] * rs) * s1[t][j];
                        if constexpr (FLAG) {
                            gg = gg > a.limit ? a.limit : gg;
                            uu = uu > a.limit ? a.limit : uu;
                            uu = uu < -a.limit ? -a.limit : uu;
                        }
                        yv[j] = m_silu(gg) * uu;
                    }
                    *(v4f*)(prow + ch * 4) = yv;
                }
            }
        }
        wave_lds_order();
        // read back row-major: lane -> (row r8 + 8*p, 16-byte column c16)
        const int c16 = lane & 7, r8 = lane >> 3;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int r = r8 + 8 * p;
            const int64_t orow = row0 + b * 32 + r;
            if (orow < row_end) {
                if constexpr (EPI == EPI_I32) {
                    *(v4i*)(a.acc + orow * a.N + nb0 * 32 + c16 * 4) = *(const v4i*)(patch + r * ROWB + c16 * 16);
                    *(v4i*)(a.acc + orow * a.N + nb1 * 32 + c16 * 4) =
                        *(const v4i*)(patch + 32 * ROWB + r * ROWB + c16 * 16);
                } else if constexpr (EPI == EPI_DEQUANT) {
                    // Written through the L2: written back by it in the ordinary way they slowed the weight streams of every
                    // other workgroup (K loops 8 % longer), and store16_through has the rest.
                    store16_through(a.out + orow * a.N + nb0 * 32 + c16 * 8, *(const v4i*)(patch + r * ROWB + c16 * 16));
                } else {
                    store16_through(a.y + orow * (a.N >> 1) + nb0 * 32 + c16 * 4, *(const v4i*)(patch + r * ROWB + c16 * 16));
                }
            }
        }
        wave_lds_order();
    }
}

// ------------------------------------------------------------------ where the column workgroups of a tile meet
// A row of SwiGLU values is quantised with its maximum, and its columns are in several workgroups.  Written as fp32 and quantised by
// a launch of its own, the values of a prefill batch pass through HBM twice, and what a product writes costs it more than what
// it reads: beside a stream of weights at 7 TB/s the writes go at 1.7 to 2.6 (128 experts of 49 rows, 2048 / 1536: 72.8 us, 64.5
// without the stores).  So (EPI_MEET) the workgroups of a tile exchange the maxima of their columns, keep the values in registers
// until the others' are there, and store int8.
// - Every workgroup stores the maxima of its rows over its columns into a word of its own per row (with the sign set: a word of
//   zero is not there yet) and looks at the others' until none is missing: no counter, no order, no fence, since a word is all that
//   is handed over.  The routing launch clears the words.
// - They run at the same time, because a launch starts its workgroups in order, those of a tile are neighbours, and those of them that
//   run on one XCD find a place there all at once (at most 48 of 96 for the 64-row tiles, 16 of 64 for the 128-row ones, 8 of 32 for
//   the wide ones, of a tall tile's two entries 16; dense_split for the dense ones).  No result rests on that: a workgroup
//   that has looked meet_looks times (a few milliseconds) computes the maxima that are still missing itself.
// What it costs is that they wait for the slowest, which is why the number of columns matters (meeting_plan in gmm.hip).  us a layer
// with / without, 128 experts of 2048 / 768, 777 / 2000 / 4000 / 8192 tokens 138 / 184 / 292 / 496 against 143 / 194 / 313 / 531; 256 of
// 7168 / 2048, 500 / 1500 / 3000 tokens 1712 / 1831 / 2049 against 1770 / 1956 / 2157; 8 of 1024 / 1408, 6000 tokens 105 against 115.
// Exchanged by atomic maxima and a counter per tile it took 2 us a tile more, with atomics inside the XCD's L2 the same
// (4096 / 7168: 6 % more).
//
// a look at a word that another workgroup writes
__device__ __forceinline__ uint32_t look(const uint32_t* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// a sum with its scales, in the order of the routed experts or of the shared one
template <bool SHARED>
__device__ __forceinline__ float scaled(int sum, float rs, float cs)
{
    return SHARED ? ((float)sum * cs) * rs : ((float)sum * rs) * cs;
}

// The maxima of the tile's rows over column block c, by the workgroup itself and one product after the other: only where the
// workgroup that is meant for that block has not come.  sum: rows words of LDS
template <bool LIMIT, bool SHARED>
__device__ __forceinline__ void maxima_of_column(const GmmArgs& a, int e, int64_t row0, int rows, int c, int channels, uint32_t* sum)
{
    for (int i = threadIdx.x; i < rows; i += (int)blockDim.x) sum[i] = 0u;
    __syncthreads();
    const int I = a.N >> 1, first = c * channels, n = I - first < channels ? I - first : channels;
    const int8_t* we = expert_weights(a, e);
    const float* cs = expert_scales(a, e);
    for (int i = threadIdx.x; i < rows * n; i += (int)blockDim.x) {
        const int r = i / n, ch = first + i % n;
        const int64_t src = a.row_src ? (int64_t)a.row_src[row0 + r] : row0 + r;
        int g = 0, u = 0;
        for (int k = 0; k < a.K; k += 16) {
            const v4i x = gload16(a.x + src * a.K + k);
            auto add = [&](int ch, int s) {
                const v4i w = gload16(we + ((int64_t)(ch >> 5) * (a.K >> 5) + (k >> 5)) * 1024 + (k >> 4 & 1) * 512 + (ch & 31) * 16);
#pragma unroll
                for (int j = 0; j < 4; ++j) s = __builtin_amdgcn_sdot4(x[j], w[j], s, false);
                return s;
            };
            g = add(ch, g);
            u = add(ch + I, u);
        }
        float gg = scaled<SHARED>(g, a.row_scale[src], cs[ch]), uu = scaled<SHARED>(u, a.row_scale[src], cs[ch + I]);
        if constexpr (LIMIT) {
            gg = gg > a.limit ? a.limit : gg;
            uu = uu > a.limit ? a.limit : uu;
            uu = uu < -a.limit ? -a.limit : uu;
        }
        const float y = __builtin_fabsf(m_silu(gg) * uu);
        if (y > 0.0f) atomicMax(sum + r, __float_as_uint(y));  // (not where it is NaN)
    }
    __syncthreads();
}

// What one workgroup has of a tile.  nt: its column block, of `columns`; g: this wavefront's channel group (a gate tile nb0 and
// its up tile); lrow: its first row behind row0.  Tall tiles whose two column blocks are done by one workgroup, one after the
// other: `first` leaves its values in y and goes on, `second` stores both.
struct TilePart {
    int e, lrow, g, nb0, nt, columns;
    int64_t row0, row_end;
    bool active, first, second;
};

// acc: the wavefront's 16 NB2 rows.  lds: ROWS * (32 GROUPS + 16) bytes (the maxima of every quarter of a wavefront, then the int8
// rows), behind them 64 KiB for the values of the widest tiles.  scales: those of the rows (ROWS of them), then 64 of the channels for
// each group.
template <int NB2, int GROUPS, int ROWS, bool LIMIT, bool SHARED>
__device__ __forceinline__ void meet_body(const GmmArgs& a, const TilePart& p, v4i (&acc)[4][NB2], int8_t* lds, float* scales)
{
    constexpr int PITCH = 32 * GROUPS + 16;
    const int tid = threadIdx.x;
    const int lane = tid & 63, tok = lane & 15, quarter = lane >> 4, run = 4 * quarter;
    const int64_t row0 = p.row0, row_end = p.row_end;
    const int nt = p.nt, columns = p.columns, lrow = p.lrow, g = p.g;
    const int rows = (int)(row_end - row0 < ROWS ? row_end - row0 : ROWS);
    float* const part = (float*)lds + (g * 4 + quarter) * ROWS + lrow + tok;
    int* const met = (int*)(scales + ROWS);  // (in the place of channel scales that have been read by then)
    const float* const cs = scales + ROWS + g * 64;
    // With ten groups of 16 rows and more there is no room for all values beside the sums: those of the first four go to LDS.  That
    // is enough for ten.  For twelve it is not: gmm_wide_kernel<EPI_MEET> spills 58 registers in the epilogue of the 192-row body
    // (for up to six groups there is room in LDS, which has not been tried).
    constexpr int STASH = NB2 > 8 ? 4 : 0;
    constexpr int STASH_AT = (ROWS * PITCH + (ROWS + 64 * GROUPS) * 4 + 15) / 16 * 16;  // behind the scales
    v4f* const stash = (v4f*)(lds + STASH_AT) + g * (STASH * 2 * 64) + lane;
    v4f y[2][NB2 - STASH];  // (a wavefront without channels has sums of zero and scales of zero)
#pragma unroll
    for (int b = 0; b < NB2; ++b) {
        const float rs = scales[lrow + b * 16 + tok];
        float m = 0.0f;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            // (read again for every 16 rows: with six blocks there is no room for them beside the sums)
            const v4f s0 = *(const v4f*)(cs + 16 * t + run), s1 = *(const v4f*)(cs + 32 + 16 * t + run);
            v4f yv;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float gg = scaled<SHARED>(acc[t][b][j], rs, s0[j]);
                float uu = scaled<SHARED>(acc[2 + t][b][j], rs, s1[j]);
                if constexpr (LIMIT) {
                    gg = gg > a.limit ? a.limit : gg;
                    uu = uu > a.limit ? a.limit : uu;
                    uu = uu < -a.limit ? -a.limit : uu;
                }
                yv[j] = m_silu(gg) * uu;
            }
            bool nan = false;  // (arithmetic makes no signalling NaNs)
            m = max_abs(m, yv, nan);
            if (b < STASH) stash[(b * 2 + t) * 64] = yv;
            else y[t][b < STASH ? 0 : b - STASH] = yv;
        }
        part[b * 16] = m;
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    if (tid == 0) *met = 1;
    float amax = 0.0f;
    if (tid < rows) {
#pragma unroll
        for (int i = 0; i < 4 * GROUPS; ++i) {
            const float o = ((const float*)lds)[i * ROWS + tid];
            amax = o > amax ? o : amax;
        }
    }
    if (columns > 1) {
        __syncthreads();  // (and the note below is reset)
        uint32_t* const word = a.meet + row0;
        if (tid < rows)
            __hip_atomic_store(word + nt * a.R + tid, __float_as_uint(amax) | 1u << 31, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (p.first && p.active) {
#pragma unroll
            for (int b = 0; b < NB2; ++b) {
                const int64_t row = row0 + lrow + b * 16 + tok;
                if (row >= row_end) continue;
#pragma unroll
                for (int t = 0; t < 2; ++t) *(v4f*)(a.y + row * (a.N >> 1) + p.nb0 * 32 + 16 * t + run) = y[t][b < STASH ? 0 : b - STASH];
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        if (p.first) return;
        // A look takes what every column has left for one row, until nothing is missing there; what the others have left for the
        // other rows of the tile came with it or follows at once.
        const int last = rows > 64 ? rows - 1 : 0;
        if (tid < 64) {
            int looks = a.meet_looks;
            for (; looks > 0; --looks) {
                const uint32_t w = lane < columns ? look(word + lane * a.R + last) : 1u;
                if (!__any(w == 0u)) break;
                __builtin_amdgcn_s_sleep(4);
            }
            if (tid == 0 && looks <= 0) *met = 0;
        }
        __syncthreads();
        if (*met && tid < rows) {
            for (int c = 0, looks = a.meet_looks;;) {
                uint32_t w[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) w[i] = c + i < columns ? look(word + (c + i) * a.R + tid) : 1u << 31;
                int here = 0;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    if (here < i || w[i] == 0u) continue;
                    const float o = __uint_as_float(w[i] & ~(1u << 31));
                    amax = o > amax ? o : amax;
                    ++here;
                }
                c += here;
                if (c >= columns) break;
                if (here < 8 && looks-- <= 0) {
                    *met = 0;
                    break;
                }
            }
        }
        __syncthreads();
        if (!*met) {
            for (int c = 0; c < columns; ++c) {
                if (c == nt) continue;
                // Column by column, what has come by now is taken (with looks of 0, for tests, nothing is): while one column is
                // computed the others come, and to compute them too would hold the compute unit that they wait for.
                uint32_t w = tid < rows && a.meet_looks > 0 ? look(word + c * a.R + tid) : 0u;
                __syncthreads();  // (everybody has read the note and the maxima)
                if (tid == 0) *met = 1;
                __syncthreads();
                if (tid < rows && w == 0u) *met = 0;
                __syncthreads();
                if (!*met) {
                    maxima_of_column<LIMIT, SHARED>(a, p.e, row0, rows, c, 32 * GROUPS, (uint32_t*)lds);
                    if (tid < rows) w = ((const uint32_t*)lds)[tid];
                }
                if (tid < rows) {
                    const float o = __uint_as_float(w & ~(1u << 31));
                    amax = o > amax ? o : amax;
                }
            }
        }
    }
    const int I = a.N >> 1;
    if (tid < rows) {
        const float s = SHARED ? amax * (float)(1.0 / 127.0) : amax / 127.0f;
        scales[tid] = SHARED ? s : 1.0f / s;
        if (nt == 0) a.q_scale[row0 + tid] = amax == 0.0f ? 0.0f : s;
    }
    __syncthreads();
    auto quantise_block = [&](bool mine, int block) __attribute__((always_inline)) {
        if (mine) {
#pragma unroll
            for (int b = 0; b < NB2; ++b) {
                const float by = scales[lrow + b * 16 + tok];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const v4f v = b < STASH ? stash[(b * 2 + t) * 64] : y[t][b < STASH ? 0 : b - STASH];
                    *(uint32_t*)(lds + (lrow + b * 16 + tok) * PITCH + g * 32 + 16 * t + run) =
                        SHARED ? quantise_over(v, by) : quantise_times(v, by);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
        constexpr int PIECES = 2 * GROUPS;  // of 16 bytes in a row
        for (int i = tid; i < rows * PIECES; i += (int)blockDim.x) {
            const int r = i / PIECES, ch = block * 32 * GROUPS + i % PIECES * 16;
            if (ch < I) store16_through(a.q + (row0 + r) * I + ch, *(const v4i*)(lds + r * PITCH + i % PIECES * 16));
        }
    };
    quantise_block(p.active, nt);
    if (p.second) {
        // the column block in front of this one, whose values this wavefront has left in y
        const bool rows_here = row0 + lrow < row_end;
        if (rows_here) {
#pragma unroll
            for (int b = 0; b < NB2; ++b) {
                const int64_t row = row0 + lrow + b * 16 + tok;
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const float* from = a.y + (row < row_end ? row : row_end - 1) * I + ((nt - 1) * GROUPS + g) * 32;
                    y[t][b < STASH ? 0 : b - STASH] = *(const v4f*)(from + 16 * t + run);
                }
            }
        }
        __syncthreads();  // the pieces of the block before are out of LDS
        quantise_block(rows_here, nt - 1);
        if (nt == 1 && tid < rows) a.q_scale[row0 + tid] = amax == 0.0f ? 0.0f : amax / 127.0f;
    }
}

template <int NB2, int GROUPS, int ROWS, bool SHARED = false>
__device__ __forceinline__ void meet_epilogue(const GmmArgs& a, const TilePart& p, v4i (&acc)[4][NB2], int8_t* lds, float* scales)
{
    if (a.limit > 0.0f) meet_body<NB2, GROUPS, ROWS, true, SHARED>(a, p, acc, lds, scales);
    else meet_body<NB2, GROUPS, ROWS, false, SHARED>(a, p, acc, lds, scales);
}

template <int EPI, int BMT, bool IN_LDS = false>
__device__ __forceinline__ void tiled_epilogue(const GmmArgs& a, int e, v4i (&acc)[4][2 * BMT], int64_t row0,
                                               int64_t row_end, int nb0, int nb1, int8_t* patch, int lane,
                                               const float* rs_lds = nullptr, const float* cs_lds = nullptr)
{
    if constexpr (EPI == EPI_SWIGLU) {
        if (a.limit > 0.0f) {
            tiled_epilogue_body<EPI, BMT, true, IN_LDS>(a, e, acc, row0, row_end, nb0, nb1, patch, lane, rs_lds, cs_lds);
            return;
        }
    }
    if constexpr (EPI == EPI_DEQUANT) {
        if (a.out_f16) {
            tiled_epilogue_body<EPI, BMT, true, IN_LDS>(a, e, acc, row0, row_end, nb0, nb1, patch, lane, rs_lds, cs_lds);
            return;
        }
    }
    tiled_epilogue_body<EPI, BMT, false, IN_LDS>(a, e, acc, row0, row_end, nb0, nb1, patch, lane, rs_lds, cs_lds);
}

// One tile of BMT token blocks: rows [row0, row_end) of expert e (at most 32 * BMT of them are computed),
// column block nt.
// RING = depth of the operand ring in registers: weights are requested RING - 1 K blocks ahead, tokens RING.
// REM: K / 64 modulo RING when K / 64 >= RING (the closing steps are then specialised), -1 for any K.
// ONCE: the tile is the only row block of its expert, so its weights are read once: non-temporal loads, as the
// streaming kernel uses them.  With several row blocks the others find the weights in L2, and must.
template <int EPI, int BMT, int RING, int REM, bool ONCE>  // BMT = token blocks of 32 per tile (BM = 32 * BMT)
__device__ __forceinline__ void tiled_body(const GmmArgs& a, int e, int64_t row0, int64_t row_end, int nt,
                                           int8_t* lds_raw, int columns)
{
    constexpr int STAGE_BYTES = TiledLds<EPI, BMT, RING>::STAGE_BYTES;
    constexpr int CHUNKS = STAGE_BYTES / 16 / 256;        // 16-byte chunks per thread per stage
    constexpr int ROWB = TiledLds<EPI, BMT, RING>::ROWB;
    constexpr int PATCHES = TiledLds<EPI, BMT, RING>::PATCHES;
    static_assert(CHUNKS >= 1, "a stage is at least one 16-byte chunk per thread");
    int8_t (*Bs)[STAGE_BYTES] = reinterpret_cast<int8_t (*)[STAGE_BYTES]>(lds_raw);

    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int lane = tid & 63;

    const int NB = a.N >> 5, KB = a.K >> 5;
    const int half_tiles = NB >> 1;
    // storage tiles of this wavefront
    int nb0, nb1;
    if constexpr (gated(EPI)) {
        nb0 = nt * 4 + wave;          // gate tile
        nb1 = nb0 + half_tiles;       // its up tile
    } else {
        nb0 = nt * 8 + 2 * wave;
        nb1 = nb0 + 1;
    }
    const bool have = gated(EPI) ? (nb0 < half_tiles) : (nb1 < NB);
    const int8_t* we = expert_weights(a, e);
    const int8_t* w0 = we + ((int64_t)(have ? nb0 : 0) * KB) * 1024 + weight_lane(lane);
    const int8_t* w1 = we + ((int64_t)(have ? nb1 : 0) * KB) * 1024 + weight_lane(lane);

    const int n_iter = a.K / kBK;

    v4i Areg[RING][4];   // [stage][16 channels]
    v4i Breg[RING][CHUNKS];

    // Loads past the last K block or the last row are redirected to valid addresses instead of being
    // skipped (their results are never used): the loop body stays free of branches, so the compiler can
    // keep several stages of loads in flight with partial s_waitcnt counts.
    const int last_it = n_iter - 1;
    auto weight_tile = [](const int8_t* p) { return ONCE ? gload16_nt(p) : gload16(p); };
    auto load_A = [&](int it, int st) {
        const int itc = it < last_it ? it : last_it;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            Areg[st][t] = weight_tile(w0 + (int64_t)itc * 2048 + t * 256);
            Areg[st][2 + t] = weight_tile(w1 + (int64_t)itc * 2048 + t * 256);
        }
    };
    const int8_t* xrow[CHUNKS];
    int lds_off[CHUNKS];
    int64_t xr[CHUNKS];
#pragma unroll
    for (int j = 0; j < CHUNKS; ++j) {
        xr[j] = row0 + (tid & 15) + 16 * ((tid >> 6) + 4 * j);
        if (xr[j] > row_end - 1) xr[j] = row_end - 1;  // rows past the expert's end duplicate its last row
    }
    if (a.row_src) {  // the rows' values lie in their tokens' rows
#pragma unroll
        for (int j = 0; j < CHUNKS; ++j) xr[j] = a.row_src[xr[j]];
    }
#pragma unroll
    for (int j = 0; j < CHUNKS; ++j) {
        // 16 consecutive lanes take 16 consecutive token rows at the same K chunk: their 16-byte LDS
        // writes then fall into 16 different bank groups (no conflicts), and a load instruction still
        // covers 16 rows x 64 contiguous bytes
        const int row = (tid & 15) + 16 * ((tid >> 6) + 4 * j);
        const int kc = (tid >> 4) & 3;
        xrow[j] = a.x + xr[j] * a.K + kc * 16;
        lds_off[j] = (row >> 4) * 1024 + kc * 256 + (row & 15) * 16;
    }
    auto load_B = [&](int it, int st) {
        const int itc = it < last_it ? it : last_it;
#pragma unroll
        for (int j = 0; j < CHUNKS; ++j) Breg[st][j] = *(const v4i*)(xrow[j] + (int64_t)itc * kBK);
    };
    auto store_B = [&](int st) {
#pragma unroll
        for (int j = 0; j < CHUNKS; ++j) *(v4i*)(&Bs[st][lds_off[j]]) = Breg[st][j];
    };

    v4i acc[4][2 * BMT];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int b = 0; b < 2 * BMT; ++b) acc[t][b] = (v4i){0};

    // B operands (fragments of 16 tokens x 64 K, 1 KiB) of half the tokens live in registers; the two halves of a
    // stage are double-buffered so that LDS reads of one half run under the MFMAs of the other.
    v4i bf0[BMT], bf1[BMT];
    auto read_frags = [&](v4i* dst, int st) {
#pragma unroll
        for (int b = 0; b < BMT; ++b) dst[b] = *(const v4i*)(&Bs[st][(b * 64 + lane) * 16]);
    };

    // ---- prologue.  After it the loads still in flight are, oldest first, A(0) B(1) A(1) B(2) ...: the same
    // order every iteration leaves behind, so the wait counts the compiler derives at the loop head are exact.
    // Every load of the prologue is requested before the first wait, so that the fill of the pipeline costs
    // one memory latency, not two.
    load_B(0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r + 1 < RING; ++r) {
        load_A(r, r);
        load_B(r + 1, r + 1);
    }
    // the scales of the epilogue too: requested behind the K loop they cost it two or three memory latencies with nothing
    // else left to do
    float* const rs_lds = (float*)(lds_raw + TiledLds<EPI, BMT, RING>::SCALES);
    float* const cs_lds = rs_lds + 32 * BMT + wave * 64;
    float rs_own = 0.0f, cs_own = 0.0f;
    if constexpr (EPI != EPI_I32) {
        if (tid < 32 * BMT) {
            int64_t r = row0 + tid < row_end ? row0 + tid : row_end - 1;
            if (a.row_src) r = a.row_src[r];
            rs_own = a.row_scale[r];
        }
        if (have) cs_own = expert_scales(a, e)[(lane < 32 ? nb0 * 32 : nb1 * 32 - 32) + lane];
    }
    __builtin_amdgcn_sched_barrier(0);
    store_B(0);
    if constexpr (EPI != EPI_I32) {
        if (tid < 32 * BMT) rs_lds[tid] = rs_own;
        cs_lds[lane] = cs_own;
    }
    __syncthreads();
    read_frags(bf0, 0);

    // One pipeline step on stage U (compile-time ring position) for K block I.  LA / LB: request the weights of
    // K block I + RING - 1 / the tokens of K block I + RING; SB: move the tokens of K block I + 1 to LDS.
#define MOE355_STEP(U, I, LA, LB, SB)                                                            \
    {                                                                                            \
        /* first half of the tokens: its MFMAs go first; the LDS traffic of the second half and */ \
        /* of the next stage is issued in the gaps while the matrix pipe is busy             */  \
        _Pragma("unroll") for (int b = 0; b < BMT; ++b)                                          \
        {                                                                                        \
            _Pragma("unroll") for (int t = 0; t < 4; ++t)                                        \
                acc[t][b] = mfma_i8_16(Areg[(U)][t], bf0[b], acc[t][b]);                         \
            bf1[b] = *(const v4i*)(&Bs[(U)][((BMT + b) * 64 + lane) * 16]);                      \
            if ((SB) && b == 0) store_B(((U) + 1) % RING); /* B(I+1): registers -> LDS */        \
            __builtin_amdgcn_sched_barrier(0);                                                   \
        }                                                                                        \
        __syncthreads(); /* B(I+1) visible to all wavefronts */                                  \
        _Pragma("unroll") for (int b = 0; b < BMT; ++b)                                          \
        {                                                                                        \
            _Pragma("unroll") for (int t = 0; t < 4; ++t)                                        \
                acc[t][BMT + b] = mfma_i8_16(Areg[(U)][t], bf1[b], acc[t][BMT + b]);             \
            if (SB) bf0[b] = *(const v4i*)(&Bs[((U) + 1) % RING][(b * 64 + lane) * 16]);         \
            if ((LA) && b == 0) load_A((I) + RING - 1, ((U) + RING - 1) % RING);                 \
            if ((LB) && b == (BMT > 1 ? 1 : 0)) load_B((I) + RING, (U));                         \
            __builtin_amdgcn_sched_barrier(0);                                                   \
        }                                                                                        \
    }
    if constexpr (REM < 0) {
        // any K: whole passes through the ring run without any condition inside (exact wait counts), the remainder
        // is peeled; requests past the last K block are redirected to it (load_A, load_B)
        const int n_full = (n_iter / RING) * RING;
        for (int i0 = 0; i0 < n_full; i0 += RING) {
            MOE355_STEP(0, i0, 1, 1, 1)
            MOE355_STEP(1, i0 + 1, 1, 1, 1)
            MOE355_STEP(2, i0 + 2, 1, 1, 1)
        }
        if (n_iter - n_full >= 1) MOE355_STEP(0, n_full, 1, 1, 1)
        if (n_iter - n_full >= 2) MOE355_STEP(1, n_full + 1, 1, 1, 1)
    } else {
        // K / 64 = 3 q + REM with q >= 1 (the host picks the instantiation).  The last RING steps request nothing
        // that lies past the last K block (the weights of the last block are requested RING - 1 steps before it,
        // its tokens RING steps before); their ring positions follow from REM, so every step is written out with
        // its requests decided at compile time: no condition inside a step, exact waits, and a tile of 12 K blocks
        // issues 66 loads per wavefront instead of 80.
        static_assert(RING == 3, "the closing steps are written for a ring of three");
        const int n_pass = (n_iter - RING - REM) / RING;  // whole passes that request both operands
        int it = 0;
        for (int ps = 0; ps < n_pass; ++ps, it += RING) {
            MOE355_STEP(0, it, 1, 1, 1)
            MOE355_STEP(1, it + 1, 1, 1, 1)
            MOE355_STEP(2, it + 2, 1, 1, 1)
        }
        if constexpr (REM >= 1) MOE355_STEP(0, it, 1, 1, 1)
        if constexpr (REM >= 2) MOE355_STEP(1, it + 1, 1, 1, 1)
        it += REM;
        MOE355_STEP(REM % RING, it, 1, 0, 1)
        MOE355_STEP((REM + 1) % RING, it + 1, 0, 0, 1)
        MOE355_STEP((REM + 2) % RING, it + 2, 0, 0, 0)
    }
#undef MOE355_STEP

    __syncthreads();  // all wavefronts are done reading the token stages; LDS is reused below
    if constexpr (EPI == EPI_MEET) {
        meet_epilogue<2 * BMT, 4, 32 * BMT>(a, TilePart{e, 0, wave, nb0, nt, columns, row0, row_end, have, false, false}, acc, lds_raw,
                                            rs_lds);
    } else {
        if (have)
            tiled_epilogue<EPI, BMT, EPI != EPI_I32>(a, e, acc, row0, row_end, nb0, nb1, lds_raw + wave * (PATCHES * 32 * ROWB), lane,
                                                     rs_lds, cs_lds);
    }
}

// The last tile of an expert is usually short.  Tiles of at most 64 rows run the two-block body (half the
// MFMAs and half the token traffic of a full tile) inside the same launch, next to the full tiles of their
// expert, so that they still find the expert's weights in the L2 of their XCD.
template <int EPI, int BMT, int RING, int REM>
__global__ __launch_bounds__(256, (BMT <= 2 ? 3 : 2)) void gmm_tiled_kernel(GmmArgs a, TileMap tm, int max_tiles, int n_col_blocks)
{
    __shared__ __attribute__((aligned(16))) int8_t lds_raw[TiledLds<EPI, BMT, RING>::BYTES];
    // ---- which tile: XCD-aware remap of the 1-D grid over the tiles that exist (workgroup i runs on
    // XCD i % 8; each XCD gets one contiguous eighth of the tile list, in order)
    const int total = tm.count[0] * n_col_blocks;
    const int per_xcd = (total + 7) / 8;
    const int slot = (int)(blockIdx.x / 8);
    const int first = (int)(blockIdx.x % 8) * per_xcd, end = first + per_xcd < total ? first + per_xcd : total;
    // EPI_MEET: every other XCD takes its share from the end, so that a tile that two XCDs share is worked on by both at once
    const int item = EPI == EPI_MEET && (blockIdx.x & 1) ? end - 1 - slot : first + slot;
    if (item < first || item >= end) return;
    const int mt = item / n_col_blocks;
    const int nt = item % n_col_blocks;
    const int e = tm.expert[mt];
    const int64_t row0 = tm.row_begin[mt];
    int64_t row_end = tm.row_end[mt];
    if (row_end > a.R) row_end = a.R;
    if (row0 >= row_end) return;
    // Tiles that are their expert's only one read its weights once, with non-temporal loads (the tiles of an expert follow one
    // another in the list).  Qwen3 shape, whole layer, 300 / 777 tokens 146 / 167 -> 138 / 156 us (short tiles); the products
    // of 128 experts of 75 rows, 2048 / 1536 and 768 / 2048, 94.5 -> 91.0 and 51.5 -> 48.5, of 256 experts of 80 rows, 2048 /
    // 7168, 721 -> 697 (full tiles); skewed batches, where all four bodies run at once, + 1 to - 1.4 %.
    const bool once = (mt == 0 || tm.expert[mt - 1] != e) && (mt + 1 == tm.count[0] || tm.expert[mt + 1] != e);
    if (row_end - row0 <= 64) {
        constexpr int SHORT = BMT > 2 ? 2 : BMT;
        if (once) tiled_body<EPI, SHORT, RING, REM, true>(a, e, row0, row_end, nt, lds_raw, n_col_blocks);
        else tiled_body<EPI, SHORT, RING, REM, false>(a, e, row0, row_end, nt, lds_raw, n_col_blocks);
        return;
    }
    // With a short K full tiles that way only where they are many: a few among short ones are the last to end.  128 experts of
    // 2048 / 768, the layer with non-temporal / plain full tiles at 49 / 53 / 59 / 66 / 75 rows per expert 1.01 / 1.01 / 0.98 /
    // 0.97 / 0.97; 256 experts of 7168 / 2048, 47 rows 0.98.
    if (once && (a.K >= 4096 || a.R >= 56 * (int64_t)a.E)) tiled_body<EPI, BMT, RING, REM, true>(a, e, row0, row_end, nt, lds_raw, n_col_blocks);
    else tiled_body<EPI, BMT, RING, REM, false>(a, e, row0, row_end, nt, lds_raw, n_col_blocks);
}

// ------------------------------------------------------------------ weight-streaming tiles
// Tiles for shapes whose grouped GEMM is bound by streaming the weights (a few hundred rows per expert at
// most).  A workgroup of eight wavefronts works on up to 256 rows of one expert, so that an expert with up to
// 256 rows fetches its weights from HBM exactly once; every wavefront computes its token blocks x one channel
// group (two storage tiles) with the accumulator layout and the epilogue of the 128-row tiles.
//   wide tile (at most 192 rows left): wavefront g = channel group g of 8, all 4, 5 or 6 token blocks of 32
//   -> 128 / 160 / 192 x 512;
//   tall tile (193..256 rows left): wavefront (h, g) = token half h x channel group g of 4 -> 256 x 256, twice
//   the token traffic per weight byte (tokens come from L2, and that traffic costs weight bandwidth).
// Both operands reach LDS by LDS-direct loads (no register staging, so the prefetch depth costs no registers),
// each into a ring of its own.  A weight stage holds the weights of 64 K values (2 KiB of every storage tile,
// copied as they lie; an MFMA operand of 16 channels is four pieces of 256 bytes of them, 512 apart), a token stage the
// tokens' 64 bytes (row-major, the 16-byte chunks exchanged by row).
// The compiler does not count LDS-direct loads against the LDS reads that consume them: the wait for a stage
// is written by hand, before the barrier that publishes the stage.
constexpr int kWideLdsBytes = 163840;

constexpr int ring_gcd(int a, int b) { return b == 0 ? a : ring_gcd(b, a % b); }

template <int N>
__device__ __forceinline__ void wait_vmcnt()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

#define MOE355_GPTR(p) ((const __attribute__((address_space(1))) void*)(p))
#define MOE355_LPTR(p) ((__attribute__((address_space(3))) void*)(p))

// NBLK: 32-row token blocks per wavefront (4 in a tall tile; 4, 5 or 6 in a wide one, so that an expert a little
// above 128 rows keeps the wide shape instead of paying the token traffic of a tall tile).
// once: the tile is its expert's only one, nobody else reads its weights: non-temporal loads, which stream from HBM at 7.1
// TB/s where plain ones reach 6.3 (these copies alone, 256 experts of 4096 x 7168).  256 experts, 7168 / 4096, 80 / 128 rows
// 1328 / 1362 -> 1175 / 1333 us; 2048 / 7168, 128 rows 757 -> 696.
template <int EPI, bool WIDE, int NBLK = 4>
__device__ __forceinline__ void stream_tile_body(const GmmArgs& a, int e, int64_t row0, int64_t row_end, int nt,
                                                 bool once, int8_t* lds, int columns = 0, bool first = false,
                                                 bool second = false)
{
    static_assert(WIDE ? (NBLK >= 1 && NBLK <= 8) : NBLK == 4, "tall tiles have two halves of four blocks");
    constexpr int GROUPS = WIDE ? 8 : 4;            // channel groups (two storage tiles each) per workgroup
    constexpr int A_BYTES = GROUPS * 4096;          // weights of a stage
    constexpr int X_BYTES = WIDE ? NBLK * 2048 : 16384;  // tokens of a stage
    // Two rings.  The weights come from HBM: their ring takes the LDS that is left once the tokens (L2 hits,
    // a third of the latency) have a ring of at least three stages.  wide: 4 + 4 (4 + 3 with five token
    // blocks); tall: 6 + 4.
    constexpr int SX = WIDE ? (NBLK > 4 ? 3 : 4) : 4;
    constexpr int SW = (kWideLdsBytes - SX * X_BYTES) / A_BYTES;
    constexpr int XBASE = SW * A_BYTES;
    constexpr int CYCLE = SW / ring_gcd(SW, SX) * SX;  // steps after which both rings are back at stage 0
    constexpr int NA = WIDE ? 4 : 2;                // weight loads per wavefront and stage
    constexpr int ROWB = TiledLds<EPI, 4, 3>::ROWB;
    constexpr int PATCHES = TiledLds<EPI, 4, 3>::PATCHES;
    static_assert(8 * PATCHES * 32 * ROWB <= SW * A_BYTES + SX * X_BYTES, "epilogue patches fit the stages");
    static_assert(SW * A_BYTES + SX * X_BYTES <= kWideLdsBytes && SX >= 3 && SW >= SX, "stages fit LDS");
    static_assert(CYCLE % SW == 0 && CYCLE % SX == 0, "the unrolled steps return to stage 0 of both rings");

    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int h = WIDE ? 0 : wave >> 2;
    const int g = WIDE ? wave : wave & 3;
    const int NB = a.N >> 5, KB = a.K >> 5;
    const int half_tiles = NB >> 1;
    auto tiles_of = [&](int cg, int& t0, int& t1) -> bool {
        if constexpr (gated(EPI)) {
            t0 = cg;
            t1 = cg + half_tiles;
            return cg < half_tiles;
        } else {
            t0 = 2 * cg;
            t1 = t0 + 1;
            return t1 < NB;
        }
    };
    // what this wavefront computes
    int nb0, nb1;
    const bool have = tiles_of(nt * GROUPS + g, nb0, nb1);
    const int64_t hrow0 = row0 + 128 * h;
    const bool active = have && hrow0 < row_end;

    // what this wavefront copies.  Weights: tall -- storage tile wave % 2 of group wave / 2; wide -- both
    // storage tiles of group wave; always the stage's 64 K values (2 KiB contiguous per tile).
    const int8_t* we = expert_weights(a, e);
    const int8_t* wsrc[WIDE ? 2 : 1];
    if constexpr (WIDE) {
        wsrc[0] = we + (int64_t)(have ? nb0 : 0) * KB * 1024 + lane * 16;
        wsrc[1] = we + (int64_t)(have ? nb1 : 0) * KB * 1024 + lane * 16;
    } else {
        int l0, l1;
        const bool lhave = tiles_of(nt * GROUPS + (wave >> 1), l0, l1);
        wsrc[0] = we + (int64_t)(lhave ? ((wave & 1) ? l1 : l0) : 0) * KB * 1024 + lane * 16;
    }
    // Tokens: one load covers 16 rows x the 64 K bytes of a stage, four neighbouring lanes on one row (one
    // 64-byte line per lane quad).  LDS slot of (row r, 16-byte chunk c) inside its 16-row KiB:
    // 4 * (r % 16) + (c ^ f(r)), f = 0, 3, 2, 1 for r / 4 % 4 = 0, 1, 2, 3 -- 64 bytes apart, sixteen rows at one chunk
    // then lie in all sixteen 16-byte bank groups, and so do rows 0..3 and 12..15 at a chunk and rows 4..11 at its
    // neighbour (c ^ 1), which is how the LDS takes the lanes of a 16-byte read.  Wavefront w copies rows 32 w .. 32 w + 31 (tall: two loads) or
    // 16 w .. 16 w + 15 (wide); 16-row blocks that lie past the expert's last row are not loaded at all
    // (their products are never stored).
    // A wide tile of more than four blocks has more than eight 16-row pieces: wavefront w also copies piece
    // w + 8 when that exists.
    constexpr int XROWS = WIDE ? 16 : 32;
    constexpr int XSECOND = WIDE ? 8 * 16 : 16;     // rows between the first and the second piece of a wavefront
    constexpr bool X2 = !WIDE || NBLK > 4;
    const int xchunk = (lane & 3) ^ (-(lane >> 4) & 3);
    const int64_t xfirst = row0 + wave * XROWS;
    const bool x2 = X2 && (WIDE ? wave + 8 < 2 * NBLK : true) && xfirst + XSECOND < row_end;
    const int n_xloads = xfirst >= row_end ? 0 : (x2 ? 2 : 1);
    int64_t xr0 = xfirst + (lane >> 2), xr1 = xr0 + XSECOND;
    if (xr0 > row_end - 1) xr0 = row_end - 1;  // rows past the expert's end duplicate its last row
    if (xr1 > row_end - 1) xr1 = row_end - 1;
    if (a.row_src) {  // the rows' values lie in their tokens' rows
        xr0 = a.row_src[xr0];
        xr1 = a.row_src[xr1];
    }
    const int8_t* xsrc0 = a.x + xr0 * a.K + xchunk * 16;
    const int8_t* xsrc1 = a.x + xr1 * a.K + xchunk * 16;
    // operand reads of this lane: token l % 16 of a block, chunk l / 16
    const int r16 = lane & 15;
    const int frag_off = XBASE + h * 8192 + r16 * 64 + (((lane >> 4) ^ (-(r16 >> 2) & 3)) * 16);
    const int a_off = g * 4096 + weight_lane(lane);

    const int n_iter = a.K / kBK;
    const int last_it = n_iter - 1;
    // loads past the last K block are redirected to it (never used), so that the number of loads in flight,
    // which the hand-written waits rely on, is the same in every step
    auto load_weights = [&](int it, int st) {
        const int itc = it < last_it ? it : last_it;
        int8_t* base = lds + st * A_BYTES + wave * (NA * 1024);
#pragma unroll
        for (int j = 0; j < NA; ++j) {
            const int8_t* wp = wsrc[j / 2] + (int64_t)itc * 2048 + (j & 1) * 1024;
            if (once) __builtin_amdgcn_global_load_lds(MOE355_GPTR(wp), MOE355_LPTR(base + j * 1024), 16, 0, 2 /* non-temporal */);
            else __builtin_amdgcn_global_load_lds(MOE355_GPTR(wp), MOE355_LPTR(base + j * 1024), 16, 0, 0);
        }
    };
    auto load_tokens = [&](int it, int st) {
        const int itc = it < last_it ? it : last_it;
        int8_t* base = lds + XBASE + st * X_BYTES;
        if (n_xloads >= 1)
            __builtin_amdgcn_global_load_lds(MOE355_GPTR(xsrc0 + (int64_t)itc * kBK),
                                             MOE355_LPTR(base + wave * (XROWS * 64)), 16, 0, 0);
        if constexpr (X2) {
            if (n_xloads >= 2)
                __builtin_amdgcn_global_load_lds(MOE355_GPTR(xsrc1 + (int64_t)itc * kBK),
                                                 MOE355_LPTR(base + (WIDE ? (wave + 8) * 1024 : wave * 2048 + 1024)),
                                                 16, 0, 0);
        }
    };

    v4i acc[4][2 * NBLK];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int b = 0; b < 2 * NBLK; ++b) acc[t][b] = (v4i){0};

    // the scales of the epilogue, in front of everything else in the queue of answers
    constexpr int ROWS = WIDE ? 32 * NBLK : 256;
    float rs_own = 0.0f, cs_own = 0.0f;
    if constexpr (meets(EPI)) {
        if ((int)threadIdx.x < ROWS) {
            int64_t r = row0 + threadIdx.x < row_end ? row0 + threadIdx.x : row_end - 1;
            if (a.row_src) r = a.row_src[r];
            rs_own = a.row_scale[r];
        }
        if (have) cs_own = expert_scales(a, e)[(lane < 32 ? nb0 * 32 : nb1 * 32 - 32) + lane];
        asm volatile("" : "+v"(rs_own), "+v"(cs_own));  // (here: the waits below count what is requested behind it)
    }

    // Every step requests the tokens SX - 1 steps ahead and then the weights SW - 1 steps ahead; the steps before
    // the first one do the same for what lies at or after K block 0, so that the order of the requests, which the
    // hand-written waits count on, is the same from the start.
#pragma unroll
    for (int j = 1 - SW; j < 0; ++j) {
        if (j + SX - 1 >= 0) load_tokens(j + SX - 1, j + SX - 1);
        load_weights(j + SW - 1, j + SW - 1);
    }

    // Requests that may still be in flight when the step d before the last one (d = kSteady: any step that is at
    // least SW - 1 before it) waits for the stage `ahead` steps after its own: everything requested behind that
    // stage's tokens.  The last SW - 1 steps request no weights and the last SX - 1 no tokens (nothing lies past the
    // last K block), so the counts shrink towards the end; each of those steps is compiled with its own.
    constexpr int kSteady = 1 << 20;
    auto in_flight = [](int d, int ahead, int nx) constexpr {
        int n = (SW > SX && d >= SW - SX + ahead) ? NA : 0;  // the weights requested right behind those tokens
        for (int m = 1; m <= SX - 2 - ahead; ++m) n += (d + m >= SX - 1 ? nx : 0) + (d + m >= SW - 1 ? NA : 0);
        return n;
    };
    // the steps d = SW - 2 .. 0 before the end (those that exist), each with its distance as a type
    auto closing_steps = [&](auto& step_fn, auto dfirst) {
        auto one = [&](auto self, auto dtag) -> void {
            constexpr int D = decltype(dtag)::value;
            if (D < n_iter) {
                const int it = last_it - D;
                step_fn(dtag, it % SW, it % SX, it);
            }
            if constexpr (D > 0) self(self, std::integral_constant<int, D - 1>{});
        };
        one(one, dfirst);
    };
    const int n_main = n_iter > SW - 1 ? n_iter - (SW - 1) : 0;  // steps that request both operands
    const int n_full = (n_main / CYCLE) * CYCLE;
    if constexpr (WIDE) {
        // One K block on stage uw of the weights and ux of the tokens.  Requests retire in order.  The younger of
        // the two requests that this step needs is its tokens (its weights, in the same step, if the rings are
        // equally deep): what was requested after it may still be in flight.  The barrier then covers the other
        // wavefronts and also says that everybody is done reading the stages that the next requests overwrite.
        auto step = [&](auto dtag, int uw, int ux, int it) {
            constexpr int D = decltype(dtag)::value;
            if (n_xloads == 2) wait_vmcnt<in_flight(D, 0, 2)>();
            else if (n_xloads == 1) wait_vmcnt<in_flight(D, 0, 1)>();
            else wait_vmcnt<in_flight(D, 0, 0)>();
            __builtin_amdgcn_s_barrier();
            if constexpr (D >= SX - 1) load_tokens(it + SX - 1, (ux + SX - 1) % SX);
            if constexpr (D >= SW - 1) load_weights(it + SW - 1, (uw + SW - 1) % SW);
            if (active) {
                const int8_t* wbase = lds + uw * A_BYTES;
                const int8_t* xbase = lds + ux * X_BYTES;
                v4i w[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) w[t] = *(const v4i*)(wbase + a_off + (t >> 1) * 2048 + (t & 1) * 256);
#pragma unroll
                for (int b = 0; b < 2 * NBLK; ++b) {
                    const v4i f = *(const v4i*)(xbase + frag_off + b * 1024);
#pragma unroll
                    for (int t = 0; t < 4; ++t) acc[t][b] = mfma_i8_16(w[t], f, acc[t][b]);
                }
            }
        };
        constexpr std::integral_constant<int, kSteady> steady{};
        for (int i0 = 0; i0 < n_full; i0 += CYCLE) {
#pragma unroll
            for (int u = 0; u < CYCLE; ++u) step(steady, u % SW, u % SX, i0 + u);
        }
#pragma unroll
        for (int u = 0; u + 1 < CYCLE; ++u)
            if (n_full + u < n_main) step(steady, u % SW, u % SX, n_full + u);
        // the closing steps: ring positions known at run time only (three or four steps of a tile's dozens)
        closing_steps(step, std::integral_constant<int, SW - 2>{});
    } else {
        // Tall tiles are bound by the matrix units, and every wavefront meets the others at the barrier of every K
        // block: operand reads that start behind that barrier leave all eight wavefronts, both of each SIMD, without
        // an MFMA to issue until the first LDS answer is back.  So the operands stay half a K block (64 of the 128
        // tokens) ahead in registers, across the barrier: a block waits for the stage AFTER its own (one stage less of
        // prefetch distance: the operands of a tall tile are L2 hits), runs its first half on operands read during the
        // block before, reads the second half's tokens under those MFMAs and the next block's weights and first tokens
        // under the second's.  Reads and MFMAs are placed one by one (sched_barrier): an MFMA that waits for the matrix
        // pipe holds up whatever is queued behind it in the wavefront.
        v4i fa[4], fb[2][NBLK];  // [16 channels] / [half][16 tokens]
        auto read_weights = [&](int uw, int t) {
            fa[t] = *(const v4i*)(lds + uw * A_BYTES + a_off + (t >> 1) * 2048 + (t & 1) * 256);
        };
        auto read_tokens = [&](int half, int ux, int b) {
            fb[half][b] = *(const v4i*)(lds + ux * X_BYTES + frag_off + (half * NBLK + b) * 1024);
        };
        // the stage of K block 0 has landed (for everybody): its first operands
        auto wait_stage = [&]() {
            // the younger request of the stage waited for is its tokens; behind them: the weights of that step and
            // every request of the later steps (the steps before the first have requested everything, redirected
            // to the last K block where a tile has fewer blocks than the rings are deep)
            if (n_xloads == 2) wait_vmcnt<in_flight(kSteady, 0, 2)>();
            else if (n_xloads == 1) wait_vmcnt<in_flight(kSteady, 0, 1)>();
            else wait_vmcnt<in_flight(kSteady, 0, 0)>();
        };
        auto wait_next_stage = [&](auto dtag) {
            constexpr int D = decltype(dtag)::value;
            if (n_xloads == 2) wait_vmcnt<in_flight(D, 1, 2)>();
            else if (n_xloads == 1) wait_vmcnt<in_flight(D, 1, 1)>();
            else wait_vmcnt<in_flight(D, 1, 0)>();
        };
        static_assert(SX >= 4, "a block reads the stage after its own: three stages in flight plus the one overwritten");
        wait_stage();
        __builtin_amdgcn_s_barrier();
        if (active) {
#pragma unroll
            for (int t = 0; t < 4; ++t) read_weights(0, t);
#pragma unroll
            for (int b = 0; b < NBLK; ++b) read_tokens(0, 0, b);
        }
        auto step = [&](auto dtag, int uw, int ux, int it) {
            constexpr int D = decltype(dtag)::value;
            if constexpr (D > 0) wait_next_stage(dtag);  // stage it + 1 has landed
            __builtin_amdgcn_s_barrier();
            if constexpr (D >= SX - 1) load_tokens(it + SX - 1, (ux + SX - 1) % SX);
            if constexpr (D >= SW - 1) load_weights(it + SW - 1, (uw + SW - 1) % SW);
            if (active) {
                static_assert(NBLK == 4, "one token read beside every group of channels");
                // the first half of the tokens, reading the second
#pragma unroll
                for (int t = 0; t < 4; ++t) {
#pragma unroll
                    for (int b = 0; b < NBLK; ++b) acc[t][b] = mfma_i8_16(fa[t], fb[0][b], acc[t][b]);
                    read_tokens(1, ux, t);
                    __builtin_amdgcn_sched_barrier(0);
                }
                // the second half, reading the next block's first tokens and, where they have just been used for the
                // last time, its weights
#pragma unroll
                for (int t = 0; t < 4; ++t) {
#pragma unroll
                    for (int b = 0; b < NBLK; ++b) acc[t][NBLK + b] = mfma_i8_16(fa[t], fb[1][b], acc[t][NBLK + b]);
                    if constexpr (D > 0) {
                        read_tokens(0, (ux + 1) % SX, t);
                        read_weights((uw + 1) % SW, t);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        constexpr std::integral_constant<int, kSteady> steady{};
        for (int i0 = 0; i0 < n_full; i0 += CYCLE) {
#pragma unroll
            for (int u = 0; u < CYCLE; ++u) step(steady, u % SW, u % SX, i0 + u);
        }
#pragma unroll
        for (int u = 0; u + 1 < CYCLE; ++u)
            if (n_full + u < n_main) step(steady, u % SW, u % SX, n_full + u);
        closing_steps(step, std::integral_constant<int, SW - 2>{});
    }

    wait_vmcnt<0>();  // the redirected loads past the end still write LDS
    __builtin_amdgcn_s_barrier();
    if constexpr (meets(EPI)) {
        constexpr int SCALES = ROWS * (32 * GROUPS + 16);
        static_assert(16 * GROUPS * ROWS <= SCALES && SCALES + (ROWS + GROUPS * 64) * 4 + 16 + (NBLK > 4 ? 65536 : 0) <= kWideLdsBytes &&
                      ROWS <= 512, "maxima, rows, scales and values fit LDS; a thread for every row");
        float* const scales = (float*)(lds + SCALES);
        if ((int)threadIdx.x < ROWS) scales[threadIdx.x] = rs_own;
        if (WIDE || h == 0) scales[ROWS + g * 64 + lane] = cs_own;
        __syncthreads();
        const TilePart part = {e, 128 * h, g, nb0, nt, columns, row0, row_end, active, first, second};
        meet_epilogue<2 * NBLK, GROUPS, ROWS, EPI == EPI_MEET_SHARED>(a, part, acc, lds, scales);
    } else {
        if (active) tiled_epilogue<EPI, NBLK>(a, e, acc, hrow0, row_end, nb0, nb1, lds + wave * (PATCHES * 32 * ROWB), lane);
    }
}

template <int EPI>
__global__ __launch_bounds__(512, 1) void gmm_wide_kernel(GmmArgs a, TileMap tm, int max_tiles, int n_col_blocks,
                                                          int columns)
{
    extern __shared__ __attribute__((aligned(16))) int8_t wide_lds[];
    // Workgroup i runs on XCD i % 8.  The tiles (listed longest first) go round the XCDs, tile t to XCD t % 8, and
    // the `columns` workgroups of a tile (a column: 512 channels, two column blocks) follow each other on that XCD,
    // so they run at the same time and share the tile's tokens in its L2.  Nothing here depends on the number of
    // tiles: the tile's entries are requested together with the count they are checked against.
    const int slot = (int)(blockIdx.x / 8);
    const int mt = (slot / columns) * 8 + (int)(blockIdx.x % 8);
    const int col = slot % columns;
    if (mt >= max_tiles) return;
    const int count = tm.count[0];
    const int listed = tm.expert[mt];
    const int64_t row0 = tm.row_begin[mt];
    int64_t row_end = tm.row_end[mt];
    if (mt >= count) return;
    const int e = listed & ~(kOnlyTile | kFirstHalf | kSecondHalf);
    const bool once = listed & kOnlyTile;
    if (row_end > a.R) row_end = a.R;
    if (row0 >= row_end) return;
    // An expert of a few rows (the cold ones of a skewed batch) runs the same body with one or two token blocks:
    // the matrix units draw their power whether a block's rows exist or not, and the kernel's clock follows it.
    if (row_end - row0 <= 32) {
        stream_tile_body<EPI, true, 1>(a, e, row0, row_end, col, once, wide_lds, columns);
    } else if (row_end - row0 <= 64) {
        stream_tile_body<EPI, true, 2>(a, e, row0, row_end, col, once, wide_lds, columns);
    } else if (row_end - row0 <= 128) {
        stream_tile_body<EPI, true>(a, e, row0, row_end, col, once, wide_lds, columns);
    } else if (row_end - row0 <= 160) {
        stream_tile_body<EPI, true, 5>(a, e, row0, row_end, col, once, wide_lds, columns);
    } else if (row_end - row0 <= 192) {
        stream_tile_body<EPI, true, 6>(a, e, row0, row_end, col, once, wide_lds, columns);
    } else {
        // a tall tile is one column block wide: the column's two blocks have an entry each, or are done one after the other
        const bool second = listed & kSecondHalf;
        if (second && 2 * col + 1 >= n_col_blocks) return;
        const bool two = !(listed & (kFirstHalf | kSecondHalf)) && 2 * col + 1 < n_col_blocks;
        stream_tile_body<EPI, false>(a, e, row0, row_end, second ? 2 * col + 1 : 2 * col, once, wide_lds, n_col_blocks, two);
        if (two) {
            __syncthreads();  // the first block's epilogue is out of LDS
            stream_tile_body<EPI, false>(a, e, row0, row_end, 2 * col + 1, once, wide_lds, n_col_blocks, false, true);
        }
    }
}

// One expert that owns every row (a dense product: the shared expert of a prefill batch): 256 x 256 tiles of the
// tall form, one workgroup per tile and compute unit, found by arithmetic on the expert's row count.  This shape
// is bound by the matrix units and, before them, by what the XCDs fetch: a tile reads 256 token rows and 256
// weight channels over the whole of K, and only tiles on the same XCD share those reads in its L2.  The 8 XCDs
// (workgroup i runs on XCD i % 8) therefore split the tile grid into xm x xn rectangles of pm x pn tiles, as
// square as the shape allows, instead of every XCD streaming all the weights.
template <int EPI>
__global__ __launch_bounds__(512, 1) void gmm_dense_kernel(GmmArgs a, int xn, int pm, int pn, int n_col_blocks)
{
    extern __shared__ __attribute__((aligned(16))) int8_t wide_lds[];
    const int xcd = (int)(blockIdx.x % 8);
    const int slot = (int)(blockIdx.x / 8);
    const int mt = (xcd / xn) * pm + slot / pn;
    const int nt = (xcd % xn) * pn + slot % pn;
    if (nt >= n_col_blocks) return;
    int64_t rows = a.gl[0];  // one group: its count and its running total are the same number
    if (rows > a.R) rows = a.R;
    const int64_t row0 = (int64_t)mt * 256;
    if (row0 >= rows) return;
    stream_tile_body<EPI, false>(a, 0, row0, rows, nt, false, wide_lds, n_col_blocks);
}

// ------------------------------------------------------------------ host side
TileSpec tile_spec(int64_t rows, int E, int BM, void* workspace)
{
    TileSpec t;
    t.BM = BM;
    t.by_length = BM == 256;
    t.flag_only = 0;
    t.max_tiles = (int)(rows / BM + E);
    const size_t arr = (size_t)(((size_t)t.max_tiles * 4 + 255) / 256) * 256;
    t.tm.count = (int32_t*)workspace;
    t.tm.expert = (int32_t*)((char*)workspace + 256);
    t.tm.row_begin = (int32_t*)((char*)workspace + 256 + arr);
    t.tm.row_end = (int32_t*)((char*)workspace + 256 + 2 * arr);
    return t;
}

size_t tiled_workspace_bytes(int64_t rows, int E, int BM)
{
    const int64_t max_tiles = rows / BM + E;
    return 256 + (size_t)(((max_tiles * 4 + 255) / 256) * 256) * 3;
}

template <int EPI, int BMT, int RING>
static void launch_tiled(const GmmArgs& a, void* workspace, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1)
{
    constexpr int BM = 32 * BMT;
    const TileSpec spec = tile_spec(a.R, a.E, BM, workspace);
    const TileMap tm = spec.tm;
    const int max_tiles = spec.max_tiles;
    if (!a.tiles_ready)
        hipLaunchKernelGGL(tile_map_kernel, dim3(1), dim3(256), 0, st, a.gl, a.gl_type, a.E, spec);
    const int channels = gated(EPI) ? a.N / 2 : a.N;
    const int per_block = gated(EPI) ? kBN / 2 : kBN;
    const int n_col_blocks = (channels + per_block - 1) / per_block;
    const int total = max_tiles * n_col_blocks;
    const int grid = ((total + 7) / 8) * 8;
    auto launch = [&](auto kernel) {
        if (ev0 || ev1)
            hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, st, ev0, ev1, 0, a, tm, max_tiles, n_col_blocks);
        else
            hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, st, a, tm, max_tiles, n_col_blocks);
    };
    // the closing steps of the K loop are compiled for K / 64 modulo the ring depth
    const int n_iter = a.K / kBK;
    if (n_iter < RING) launch(gmm_tiled_kernel<EPI, BMT, RING, -1>);
    else if (n_iter % RING == 0) launch(gmm_tiled_kernel<EPI, BMT, RING, 0>);
    else if (n_iter % RING == 1) launch(gmm_tiled_kernel<EPI, BMT, RING, 1>);
    else launch(gmm_tiled_kernel<EPI, BMT, RING, 2>);
}

template <int EPI>
static bool launch_wide(const GmmArgs& a, void* workspace, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1)
{
    constexpr int BM = 256;
    constexpr int lds_bytes = kWideLdsBytes;
    static OncePerDevice once;
    if (!allow_dynamic_lds(once, (const void*)gmm_wide_kernel<EPI>, lds_bytes)) return false;
    const TileSpec spec = tile_spec(a.R, a.E, BM, workspace);
    const TileMap tm = spec.tm;
    const int max_tiles = spec.max_tiles;
    if (!a.tiles_ready)
        hipLaunchKernelGGL(tile_map_kernel, dim3(1), dim3(256), 0, st, a.gl, a.gl_type, a.E, spec);
    const int channels = gated(EPI) ? a.N / 2 : a.N;
    const int per_block = gated(EPI) ? kBN / 2 : kBN;
    const int n_col_blocks = (channels + per_block - 1) / per_block;
    const int columns = (n_col_blocks + 1) / 2;
    const int grid = 8 * ((max_tiles + 7) / 8) * columns;  // one workgroup per (tile, column), no idle ones
    if (ev0 || ev1)
        hipExtLaunchKernelGGL((gmm_wide_kernel<EPI>), dim3(grid), dim3(512), lds_bytes, st, ev0, ev1, 0, a, tm,
                              max_tiles, n_col_blocks, columns);
    else
        hipLaunchKernelGGL((gmm_wide_kernel<EPI>), dim3(grid), dim3(512), lds_bytes, st, a, tm, max_tiles,
                           n_col_blocks, columns);
    return true;
}

// The split of the 8 XCDs over rows x columns with the smallest rectangle perimeter (= bytes fetched per XCD).  Workgroups that
// exchange maxima hold their places until the last one of their row of tiles has come, so all of a row that fall to an XCD must find
// a place there: 32 workgroups run on one, 16 columns leave room for such a launch on another stream.  A split like that exists up to
// 128 columns.
DenseSplit dense_split(int64_t rows, int columns, bool meet)
{
    const int row_tiles = (int)((rows + 255) / 256), most = meet ? 16 : columns;
    DenseSplit best = {};
    for (int c = 1; c <= 8; c *= 2) {
        const DenseSplit s = {c, (row_tiles + 8 / c - 1) / (8 / c), (columns + c - 1) / c};
        if (s.pn <= most && (best.xn == 0 || s.pm + s.pn < best.pm + best.pn)) best = s;
    }
    return best;
}

template <int EPI>
static bool launch_dense_t(const GmmArgs& a, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1)
{
    constexpr int lds_bytes = kWideLdsBytes;
    static OncePerDevice once;
    if (!allow_dynamic_lds(once, (const void*)gmm_dense_kernel<EPI>, lds_bytes)) return false;
    const int channels = gated(EPI) ? a.N / 2 : a.N;
    const int per_block = gated(EPI) ? kBN / 2 : kBN;
    const int n_col_blocks = (channels + per_block - 1) / per_block;
    const auto [xn, pm, pn] = dense_split(a.R, n_col_blocks, meets(EPI));
    const int grid = 8 * pm * pn;
    if (ev0 || ev1)
        hipExtLaunchKernelGGL((gmm_dense_kernel<EPI>), dim3(grid), dim3(512), lds_bytes, st, ev0, ev1, 0, a, xn, pm, pn,
                              n_col_blocks);
    else
        hipLaunchKernelGGL((gmm_dense_kernel<EPI>), dim3(grid), dim3(512), lds_bytes, st, a, xn, pm, pn, n_col_blocks);
    return true;
}

bool launch_dense(int epi, const GmmArgs& a, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1)
{
    if (epi == EPI_I32) return launch_dense_t<EPI_I32>(a, st, ev0, ev1);
    if (epi == EPI_SWIGLU) return launch_dense_t<EPI_SWIGLU>(a, st, ev0, ev1);
    if (epi == EPI_MEET_SHARED) return launch_dense_t<EPI_MEET_SHARED>(a, st, ev0, ev1);
    return launch_dense_t<EPI_DEQUANT>(a, st, ev0, ev1);
}

bool launch_tiled_any(int epi, int bm, const GmmArgs& a, void* workspace, hipStream_t st, hipEvent_t ev0,
                      hipEvent_t ev1)
{
#define MOE355_TILED(E_, B_) launch_tiled<E_, B_, 3>(a, workspace, st, ev0, ev1)
    if (bm == 256) {
        if (epi == EPI_I32) return launch_wide<EPI_I32>(a, workspace, st, ev0, ev1);
        if (epi == EPI_SWIGLU) return launch_wide<EPI_SWIGLU>(a, workspace, st, ev0, ev1);
        if (epi == EPI_MEET) return launch_wide<EPI_MEET>(a, workspace, st, ev0, ev1);
        return launch_wide<EPI_DEQUANT>(a, workspace, st, ev0, ev1);
    }
    if (bm == 128) {
        if (epi == EPI_I32) MOE355_TILED(EPI_I32, 4);
        else if (epi == EPI_SWIGLU) MOE355_TILED(EPI_SWIGLU, 4);
        else if (epi == EPI_MEET) MOE355_TILED(EPI_MEET, 4);
        else if (resident_supported(a)) {
            if (!a.tiles_ready) {
                const TileSpec spec = tile_spec(a.R, a.E, bm, workspace);
                hipLaunchKernelGGL(tile_map_kernel, dim3(1), dim3(256), 0, st, a.gl, a.gl_type, a.E, spec);
            }
            return launch_resident(a, workspace, st, ev0, ev1);
        } else MOE355_TILED(EPI_DEQUANT, 4);
    } else {
        if (epi == EPI_I32) MOE355_TILED(EPI_I32, 2);
        else if (epi == EPI_SWIGLU) MOE355_TILED(EPI_SWIGLU, 2);
        else if (epi == EPI_MEET) MOE355_TILED(EPI_MEET, 2);
        else MOE355_TILED(EPI_DEQUANT, 2);
    }
#undef MOE355_TILED
    return true;
}

}  // namespace moe355
