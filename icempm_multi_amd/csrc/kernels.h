// kernels.h -- host-side launchers of the HIP kernels (one per .hip file).
#pragma once

#include <hip/hip_runtime.h>
#include "mpm_common.h"

namespace icempm {

// kernels_fp64.hip / kernels_mixed.hip share these signatures.
// Tile kernels: mode bit 1 = G2P from grid[rbuf], bit 2 = P2G into grid[wbuf].
// Bit 4 folds the grid update in: G2P stages node velocities computed from the
// momenta of grid[rbuf] (instead of reading velocities a grid update wrote),
// and the launch also clears the flagged segments of grid[zbuf], adds the
// indenter force of the nodes inside the indenter and advances the clocks.
enum TileMode {
    kTileG2P = 1,
    kTileP2G = 2,
    kTileFused = 3,
    kTileFromMomenta = 4,
    kTileTail = kTileG2P | kTileFromMomenta,     // last G2P of a call
    kTileChain = kTileFused | kTileFromMomenta,  // grid update + G2P(n) + P2G(n+1)
};

namespace fp64 {
// record_mode: 1/0 = write P, Q or not; -1 = decide from the scene clock.
hipError_t launch_tiles(const StepArgs &a, int mode, int rbuf, int wbuf, int zbuf, int record_mode, hipStream_t s);
hipError_t launch_p2g_direct(const StepArgs &a, int scene, int n_pts, int wbuf, hipStream_t s);
hipError_t launch_g2p_direct(const StepArgs &a, int scene, int n_pts, int rbuf, int record_pq, hipStream_t s);
// One substep of a scene's points in their own order: grid update folded in,
// G2P from grid[rbuf]'s momenta and, with next, P2G into grid[wbuf]; clears
// grid[zbuf].  a.n_work: workgroups of 256 points.
hipError_t launch_points(const StepArgs &a, int scene, bool next, int rbuf, int wbuf, int zbuf, hipStream_t s);
// Grid update of both precision forms: their grids share one layout (3 FP64
// lines per buffer) and the update works in FP64.
hipError_t launch_update(const StepArgs &a, int buf, int zero_other, int advance_clock, int n_blocks, hipStream_t s);
hipError_t launch_update_at(StepArgs a, int buf, const SceneClock &clock, SceneClock *slot, int n_blocks,
                            hipStream_t s);
hipError_t launch_clear(const StepArgs &a, int buf, int n_blocks, hipStream_t s);
size_t tile_lds_bytes(const StepArgs &a, int mode);
// Workgroups of the tile kernel for this mode and window that one CU holds at
// once (registers and LDS); 0 if the runtime cannot tell.
int tiles_resident_per_cu(const StepArgs &a, int mode);
}  // namespace fp64

namespace mixed {
// record_mode: 1/0 = write P, Q or not; -1 = decide from the scene clock.
hipError_t launch_tiles(const StepArgs &a, int mode, int rbuf, int wbuf, int zbuf, int record_mode, hipStream_t s);
hipError_t launch_p2g_direct(const StepArgs &a, int scene, int n_pts, int wbuf, hipStream_t s);
hipError_t launch_g2p_direct(const StepArgs &a, int scene, int n_pts, int rbuf, int record_pq, hipStream_t s);
size_t tile_lds_bytes(const StepArgs &a, int mode);
// Workgroups of the tile kernel for this mode and window that one CU holds at
// once (registers and LDS); 0 if the runtime cannot tell.
int tiles_resident_per_cu(const StepArgs &a, int mode);
}  // namespace mixed

// kernels_common.hip
// Clock of every scene: t += dt; ind_x = x0 + t*V; step counter (model.cpp:39-41).
hipError_t launch_fill_zero(void *ptr, size_t bytes, hipStream_t s);

// binning.hip -- device RemoveDisabledAndSort and tile tables.
struct BinWork {
    int *keys;          // per point: bin (cell) index within its scene, -1 if disabled
    int *cell_count;    // concatenated per-scene cell histograms (+1 slot per scene)
    int *cell_fill;     // scatter cursors
    int *cell_start;    // exclusive scan (global point indices)
    int *perm;          // sorted position -> previous point index
    int *scan_tmp;      // block sums of the scan
    int *scene_count;   // per scene: kept points after the sort
    int *sorted_keys;   // per sorted point: its reference cell key
    long long n_cells_total;
    long long n_pts_total;   // size of the point index space
};
// elem_bytes: 8 (FP64 SoA) or 4 (mixed SoA).
hipError_t launch_sort(const StepArgs &a, const SceneDev *host_scenes, int nscenes, BinWork &w, int elem_bytes,
                       void *pts_src, void *pts_dst, hipStream_t s);
// Tile shapes to count the tiles of (launch_tile_census: counts[i] = tiles of
// shape i that hold points, by the points as last sorted).
struct TileShapes {
    static constexpr int kMax = 8;
    int n = 0;
    int tx[kMax], ty[kMax];
};
// The tiles of one shape: how many take k + 1 passes of a workgroup (the last
// entry: that many and more), the most passes, the points of all.
struct TileCensus {
    static constexpr int kPasses = 64;
    int tiles[kPasses];
    int most, points;
};
hipError_t launch_tile_census(const StepArgs &a, const TileShapes &shapes, const BinWork &w, TileCensus *out,
                              hipStream_t s);
// Phase calls' times: stamps of launches (StepArgs::stamp, kStampStride words
// each), summed by class into ticks.
constexpr int kStampSlots = 32, kStampStride = 2 + kStampBlocks;
struct StampClasses {
    int n = 0;
    unsigned char cls[kStampSlots];
};
hipError_t launch_sum_stamps(const unsigned long long *stamps, const StampClasses &classes, unsigned long long *ticks,
                             hipStream_t s);
// The tile table of the binned kernels (mpm_common.h) and its builder's memory.
struct TileTable {
    long long max_tiles = 0;      // places of tiles
    long long max_live = 0;       // tiles that can hold points
    int n_work = 0;               // workgroups of a tile launch
    int n_few = 0;                // workgroups where no more tiles than these are found (0: always n_work)
    TileWork *work = nullptr;
    TileItem *tiles = nullptr;    // in spatial order
    TileItem *list = nullptr;     // by workgroup
    TileRun *runs = nullptr;
    int *n_tiles = nullptr;
    int *flag = nullptr, *pos = nullptr, *weight = nullptr, *scan_tmp = nullptr;
};
// Lays the table out from base (null: only counts); returns its bytes.
size_t tile_table_layout(char *base, long long max_tiles, long long max_points, int tx, int n_work, TileTable &t);
hipError_t launch_build_tiles(const StepArgs &a, const SceneDev *host_scenes, int nscenes, long long n_points,
                              const TileTable &t, hipStream_t s);

}  // namespace icempm
