// The list of (expert, row block) tiles of a grouped GEMM, built on the device by one workgroup: on its own in front of
// the GEMM (tile_map_kernel), or by an extra workgroup of the routing launch, which knows the row counts first.
#pragma once

#include "moe355_common.h"

namespace moe355 {

// in the list by length and where it is asked for: the tile is its expert's only one
constexpr int32_t kOnlyTile = 1 << 30;
// in the list by length: an entry of one half of a tall tile's columns (neither: both of them)
constexpr int32_t kFirstHalf = 1 << 29, kSecondHalf = 1 << 28;

// (expert, row block) tiles of one launch
struct TileMap {
    int32_t* count;      // [1]
    int32_t* expert;     // [max_tiles] (and kOnlyTile, kFirstHalf, kSecondHalf)
    int32_t* row_begin;  // [max_tiles]
    int32_t* row_end;    // [max_tiles] end of the expert's rows
};

struct TileSpec {
    TileMap tm;
    int BM, max_tiles;
    // the 256-row weight-streaming tiles, listed longest first -- 161..192 rows, 129..160, up to 128 -- so that the workgroups
    // that start last are the short ones and the compute units finish closer together, and the tall ones (more than 192 rows),
    // where enough of them share their weights with another tile, spread evenly among them: the tall tiles of a hot expert find their weights in the caches and wait for the matrix units,
    // the cold experts' tiles for their weights from HBM, and so both are busy all the time.  In eights, because entry t
    // runs on XCD t % 8.  A tall tile has an entry for either half of its columns as long as the list has room for that (a
    // workgroup per entry and column is launched for as many tiles as the rows can make), beyond it one for both.
    // Both halves are in the same eight entries, since their workgroups wait for each other (EPI_MEET in gmm_tiled.hip).
    // Layers under Zipf(1.1), 256 experts of 7168 / 2048, 2048 / 3000 / 4096 tokens: tall ones whole and last 1662 / 2165 / 2520 us,
    // halves last 1631 / 2108 / 2510, halves first 1617 / 2075 / 2443, spread 1567 / 1998 / 2254; 128 experts of 2048 / 768, 1900
    // tokens 223 whole and last, 214 spread.  4096 tokens of uniform routing, a few of whose experts are tall because of the
    // router's bias, gate_up alone 1295 whole and last, 1325 halves first.
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
    if (spec.by_length) {  // BM is 256
        // class of a tile with m rows left in its expert; per-thread counts per class, two classes per scan
        auto cls = [](int64_t m) -> int { return m > 192 ? 3 : (m > 160 ? 0 : (m > 128 ? 1 : 2)); };
        // tiles in front of an expert's last one, all of them tall
        auto full_tiles = [](int64_t m) -> int32_t { return (int32_t)((uint32_t)(m - 1) >> 8); };
        int32_t rows = 0, n01 = 0, n23 = 0;  // counts packed 16 + 16 bits (at most max_tiles < 32768 tiles)
        int32_t shared = 0;                  // tall tiles whose weights another tile of the expert reads too
        for (int j = 0; j < seg; ++j) {
            const int e = e0 + j;
            if (e < E) {
                const int64_t m = rows_of(e);
                rows += (int32_t)m;
                if (m == 0) continue;
                const int32_t full = full_tiles(m);
                const int c = cls(m - (int64_t)full * 256);
                n23 += full << 16;
                shared += full + (full > 0 && c == 3 ? 1 : 0);
                if (c < 2) n01 += 1 << (16 * c);
                else n23 += 1 << (16 * (c - 2));
            }
        }
        int32_t all_rows, all01, all23;
        const int32_t rows_before = block_scan_exclusive_i32(rows, part_a, all_rows);
        // part_a is free behind the first scan; its sums are visible behind the second one and read before the third one is over
        const int32_t shared_wave = wave_scan_inclusive_i32(shared);
        if ((tid & 63) == 63) part_a[tid >> 6] = shared_wave;
        const int32_t b01 = block_scan_exclusive_i32(n01, part_b, all01);
        int32_t all_shared = 0;
        for (int w = 0; w < (int)(blockDim.x + 63) >> 6; ++w) all_shared += part_a[w];
        const int32_t b23 = block_scan_exclusive_i32(n23, part_b, all23);
        const int32_t total[4] = {all01 & 0xffff, all01 >> 16, all23 & 0xffff, all23 >> 16};
        const int32_t all_tiles = total[0] + total[1] + total[2] + total[3];
        const int32_t room = max_tiles > all_tiles ? max_tiles - all_tiles : 0;
        // Whole and last: fewer than one tall tile in 16, which has no phase of its own to mix, and tall tiles that are their
        // experts' only ones, which wait for HBM as the others do; halves would only read their tokens twice.  Few of the first
        // kind, 4096 tokens of uniform routing, gate_up / down 1344 / 792 us spread, 1318 / 778 so; under Zipf(0.6), where one in 8 to
        // 16 is tall, the layer at 2048 tokens 2175 spread, 2261 so.  Of the second kind, uniform routing, layers as they were
        // before there were halves / spread / so: 8 experts of 4096 / 14336, 187 / 200 / 220 rows each 471 / 525 / 469, 473 / 634 / 473, 484 /
        // 600 / 484; 128 of 4096 / 1536, 210 rows 777 / 803 / 778; 96 of 8192 / 2048, 200 rows 1301 / 1361 / 1304.  With 240 to 256 rows,
        // where some experts spill over into a second tile, spreading wins: 256 of 7168 / 2048 3580 / 3475 at 240, 64 of 8192 /
        // 2560 1453 / 1340 at 250, 96 of 8192 / 2048 1562 / 1505 under Zipf(0.1) at 220, where one tile in eight is tall and shared.
        // Between (one in 33, 24, 22, 21, 17): 1.01, 0.98, 0.95, 1.01, 0.97 of the time.
        const bool few = 16 * total[3] < all_tiles || 24 * all_shared < all_tiles;
        // Tall tiles with one entry: an even number in front, so that pairs of halves start at even places.  One more is the first of
        // the others (the last one of all: the layers of 128 experts of 4096 / 1024, 2000 tokens under Zipf(0.8), 4 % slower).
        const int32_t whole = few ? total[3] : total[3] > room ? total[3] - room : 0, extra = few ? 0 : whole & 1;
        const int32_t in_front = whole - extra, tall = 2 * (total[3] - extra) - in_front, others = all_tiles - total[3] + extra;
        if (tid == 0) tm.count[0] = all_tiles < max_tiles ? others + tall : max_tiles;
        // eight entries, one for every XCD, are a block; the blocks of tall entries lie at ((2 b + 1) n / 2 a) of the a of them among
        // n blocks, and what fills no block at the end, the tall ones last (so that their pairs start at even places there too, an odd one
        // of the others behind them)
        const int32_t a8 = few ? 0 : tall >> 3, n8 = a8 + (others >> 3);  // at most 8192 and 12288
        // x / d where the quotient is at most 12288: by the reciprocal it is off by one at most.  One lane walks the tiles
        // of a hot expert, and 64-bit divisions for each of them made the launch of 4096 tokens under Zipf(1.1) 30 us
        // instead of 16.
        auto divide = [](int32_t x, int32_t d, float by) {
            const int32_t q = (int32_t)((float)x * by), rest = x - q * d;
            return rest < 0 ? q - 1 : rest >= d ? q + 1 : q;
        };
        const float by_a = 1.0f / (float)(2 * a8), by_n = 1.0f / (float)(2 * n8);
        auto tall_at = [&](int32_t i) {
            if ((i >> 3) < a8) return divide((2 * (i >> 3) + 1) * n8, 2 * a8, by_a) * 8 + (i & 7);
            return (few ? others : others & ~1) + i;
        };
        auto other_at = [&](int32_t i) {
            int32_t at = i >> 3, before = 0;
            if (!few && i == others - 1 && (others & 1)) return tall + i;
            if (at >= n8 - a8) return a8 * 8 + i;
            for (int32_t next = -1; next != before;) {  // the tall blocks in front of it: those at `at` or before
                next = before;
                const int32_t reach = 2 * (at + before + 1) * a8 - n8;
                before = reach <= 0 ? 0 : divide(reach + 2 * n8 - 1, 2 * n8, by_n);
                if (before > a8) before = a8;
            }
            return (at + before) * 8 + (i & 7);
        };
        int32_t next[3] = {extra + (b01 & 0xffff), extra + total[0] + (b01 >> 16), extra + total[0] + total[1] + (b23 & 0xffff)};
        int32_t next_tall = (b23 >> 16) - extra;
        int64_t row = rows_before;
        for (int j = 0; j < seg; ++j) {
            const int e = e0 + j;
            if (e < E) {
                const int64_t m = rows_of(e);
                if (m == 0) continue;
                const int32_t full = full_tiles(m);
                const int c = cls(m - (int64_t)full * 256), listed = m <= BM ? e | kOnlyTile : e;
                for (int32_t t = 0; t < full + (c == 3 ? 1 : 0); ++t) {
                    const int32_t i = next_tall++;
                    const int64_t begin = row + (int64_t)t * 256;
                    if (i < in_front) {
                        put(i < 0 ? other_at(0) : tall_at(i), listed, begin, row + m);
                    } else {
                        put(tall_at(2 * i - in_front), listed | kFirstHalf, begin, row + m);
                        put(tall_at(2 * i - in_front + 1), listed | kSecondHalf, begin, row + m);
                    }
                }
                if (c < 3) put(other_at(next[c]++), listed, row + (int64_t)full * 256, row + m);
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
