// Host interface of the LDS-tiled grouped GEMM (gmm_tiled.hip).
#pragma once

#include "gmm_common.h"
#include "tile_map.h"

namespace moe355 {

// bytes of scratch for the tile map (BM = rows per tile: 64, 128 or 256)
size_t tiled_workspace_bytes(int64_t rows, int E, int BM);

// the tile map of a product over `rows` rows, laid out in a workspace of tiled_workspace_bytes()
TileSpec tile_spec(int64_t rows, int E, int BM, void* workspace);

// epi: EPI_*; bm: 64 or 128 (LDS-tiled kernel) or 256 (weight-streaming tiles).  ev0/ev1: optional events recorded around
// the GEMM kernel itself.  false: the device refused the kernel its LDS, nothing was launched.
bool launch_tiled_any(int epi, int bm, const GmmArgs& a, void* workspace, hipStream_t st, hipEvent_t ev0,
                      hipEvent_t ev1);

// The down product on the list of 128-row tiles (in the workspace) with a tile's tokens in LDS for the whole of K
// (gmm_resident.hip).
bool resident_supported(const GmmArgs& a);
bool launch_resident(const GmmArgs& a, void* workspace, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1);

// One expert owning every row: 64 x 64 tiles with K cut over the wavefronts (gmm_split.hip), no tile map either.
void launch_split(int epi, const GmmArgs& a, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1);

// One expert owning every row (a.E == 1): 256 x 256 tiles placed by arithmetic, no tile map, no scratch.  xn of the 8 XCDs lie side
// by side, each with a rectangle of pm x pn tiles; meet: the workgroups of a row of tiles exchange its maxima (EPI_MEET_SHARED).
struct DenseSplit {
    int xn, pm, pn;
};
DenseSplit dense_split(int64_t rows, int columns, bool meet);
bool launch_dense(int epi, const GmmArgs& a, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1);

}  // namespace moe355
