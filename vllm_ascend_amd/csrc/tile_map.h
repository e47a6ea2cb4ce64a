// The list of (expert, row block) tiles of a grouped GEMM, built on the device by one workgroup: on its own in front of
// the GEMM (tile_map_kernel), or by an extra workgroup of the routing launch, which knows the row counts first.
#pragma once

#include "moe355_common.h"

namespace moe355 {

// in the list by length and where it is asked for: the tile is its expert's only one
constexpr int32_t kOnlyTile = 1 << 30;

// (expert, row block) tiles of one launch
struct TileMap {
    int32_t* count;      // [1]
    int32_t* expert;     // [max_tiles] (and kOnlyTile)
    int32_t* row_begin;  // [max_tiles]
    int32_t* row_end;    // [max_tiles] end of the expert's rows
};

struct TileSpec {
    TileMap tm;
    int BM, max_tiles;
    // the 256-row weight-streaming tiles: the tiles are listed longest first -- 161..192 rows, 129..160, up to 128,
    // then the tall ones (more than 192 rows, which become two shorter column items) -- so that the workgroups that
    // start last are the short ones and the compute units finish closer together
    int by_length;
    int flag_only;  // kOnlyTile also in a list in the order of the experts
};

// One workgroup of any size, every thread calls it; rows_of(e) = rows of expert e (not negative).  Thread t owns
// experts [t*seg, (t+1)*seg).  part_a, part_b: 16 ints of LDS each.
template <typename RowsOf>
__device__ __forceinline__ void build_tile_map(RowsOf rows_of, int E, const TileSpec& spec, int32_t* part_a,
                                               int32_t* part_b)
{
    const TileMap& tm = spec.tm;
    const int BM = spec.BM, max_tiles = spec.max_tiles, tid = threadIdx.x;
    const int seg = (E + (int)blockDim.x - 1) / (int)blockDim.x;
    const int e0 = tid * seg;
    auto put = [&](int32_t t, int e, int64_t begin, int64_t end) {
        if (t < max_tiles) {
            tm.expert[t] = e;
            tm.row_begin[t] = (int32_t)begin;
            tm.row_end[t] = (int32_t)end;
        }
    };
    if (spec.by_length) {
        // class of a tile with m rows left in its expert; per-thread counts per class, two classes per scan
        auto cls = [](int64_t m) -> int { return m > 192 ? 3 : (m > 160 ? 0 : (m > 128 ? 1 : 2)); };
        int32_t rows = 0, n01 = 0, n23 = 0;  // counts packed 16 + 16 bits (at most max_tiles < 32768 tiles)
        for (int j = 0; j < seg; ++j) {
            const int e = e0 + j;
            if (e < E) {
                const int64_t m = rows_of(e);
                rows += (int32_t)m;
                for (int64_t r0 = 0; r0 < m; r0 += BM) {
                    const int c = cls(m - r0);
                    if (c < 2) n01 += 1 << (16 * c);
                    else n23 += 1 << (16 * (c - 2));
                }
            }
        }
        int32_t all_rows, all01, all23;
        const int32_t rows_before = block_scan_exclusive_i32(rows, part_a, all_rows);
        const int32_t b01 = block_scan_exclusive_i32(n01, part_b, all01);
        const int32_t b23 = block_scan_exclusive_i32(n23, part_b, all23);
        const int32_t total[4] = {all01 & 0xffff, all01 >> 16, all23 & 0xffff, all23 >> 16};
        const int32_t all_tiles = total[0] + total[1] + total[2] + total[3];
        if (tid == 0) tm.count[0] = all_tiles < max_tiles ? all_tiles : max_tiles;
        int32_t next[4] = {b01 & 0xffff, total[0] + (b01 >> 16), total[0] + total[1] + (b23 & 0xffff),
                           total[0] + total[1] + total[2] + (b23 >> 16)};
        int64_t row = rows_before;
        for (int j = 0; j < seg; ++j) {
            const int e = e0 + j;
            if (e < E) {
                const int64_t m = rows_of(e);
                for (int64_t r0 = 0; r0 < m; r0 += BM)
                    put(next[cls(m - r0)]++, m <= BM ? e | kOnlyTile : e, row + r0, row + m);
                row += m;
            }
        }
        return;
    }
    int32_t rows = 0, tiles = 0;
    for (int j = 0; j < seg; ++j) {
        const int e = e0 + j;
        if (e < E) {
            const int64_t m = rows_of(e);
            rows += (int32_t)m;
            tiles += (int32_t)((m + BM - 1) / BM);
        }
    }
    // exclusive prefix of rows and tiles over the threads (experts in order)
    int32_t all_rows, all_tiles;
    const int32_t rows_before = block_scan_exclusive_i32(rows, part_a, all_rows);
    const int32_t tiles_before = block_scan_exclusive_i32(tiles, part_b, all_tiles);
    if (tid == 0) tm.count[0] = all_tiles < max_tiles ? all_tiles : max_tiles;
    int64_t row = rows_before;
    int32_t t = tiles_before;
    for (int j = 0; j < seg; ++j) {
        const int e = e0 + j;
        if (e < E) {
            const int64_t m = rows_of(e);
            for (int64_t r0 = row; r0 < row + m; r0 += BM) put(t++, spec.flag_only && m <= BM ? e | kOnlyTile : e, r0, row + m);
            row += m;
        }
    }
}

}  // namespace moe355
