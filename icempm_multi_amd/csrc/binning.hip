// binning.hip -- on-device HostSideSOA::RemoveDisabledAndSort
// (simulation/hssoa/host_side_soa.cpp:50-61) and the tile tables of the
// binned kernels.
//
// Counting sort by the reference's cell key (proxypoint2d.cpp:164-169):
//   key = (int)(x/h + 0.5)*GridY + (int)(y/h + 0.5)
// 1. keys + per-cell histogram (int atomics), disabled points dropped;
// 2. exclusive scan of the concatenated per-scene histograms -> cell_start;
// 3. scatter of point indices into their cells (atomic cursors);
// 4. each cell's indices sorted ascending, so ties keep their previous order
//    and the result is the stable order, independent of atomic timing;
// 5. gather of the 16 SoA lines into the second point buffer.
// Built with -ffp-contract=off so that x*hinv+0.5 is rounded twice, as on the host.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "kernels.h"

namespace icempm {

namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ int scene_of_point(const SceneDev *sc, int nscenes, long long i)
{
    int lo = 0, hi = nscenes - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (sc[mid].pt_off <= i) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ int scene_of_cell(const SceneDev *sc, int nscenes, long long j)
{
    int lo = 0, hi = nscenes - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (sc[mid].cell_off <= j) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// (int)(x*hinv + 0.5), reference rounding (two roundings, C truncation)
__device__ __forceinline__ int cell_index_fp64(double x, double hinv) { return (int)(x * hinv + 0.5); }

// the same on a fixed-point coordinate x/h = q*2^-fb - origin, exactly
__device__ __forceinline__ int cell_index_fixed(unsigned q, int fb, int origin)
{
    const long long v = (long long)q + (1LL << (fb - 1)) - ((long long)origin << fb);
    return v >= 0 ? (int)(v >> fb) : -(int)((-v) >> fb);
}

template <int EB>
__global__ void __launch_bounds__(kBlock) k_keys(StepArgs a, BinWork w, const void *src)
{
    const long long i = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (i >= w.n_pts_total) return;
    const int s = scene_of_point(a.scenes, a.nscenes, i);
    const SceneDev &S = a.scenes[s];
    const long long local = i - S.pt_off;
    if (local < 0 || local >= S.n_pts) { w.keys[i] = -2; return; }
    int ix, iy;
    if (EB == 8) {
        const double *P = (const double *)src;
        const long long ud = __double_as_longlong(P[i]);
        if (ud & kDisabled) { w.keys[i] = -1; return; }
        ix = cell_index_fp64(P[kLinePosX * a.pitch + i], S.c.hinv);
        iy = cell_index_fp64(P[(kLinePosX + 1) * a.pitch + i], S.c.hinv);
    } else {
        const unsigned *P = (const unsigned *)src;
        if (P[i] & (unsigned)kDisabled) { w.keys[i] = -1; return; }
        ix = cell_index_fixed(P[kLinePosX * a.pitch + i], S.c.frac_bits, S.c.origin);
        iy = cell_index_fixed(P[(kLinePosX + 1) * a.pitch + i], S.c.frac_bits, S.c.origin_y);
    }
    const int col = min(max(ix - S.c.xoff + S.c.halo, 0), S.c.ncols - 1);
    const int row = min(max(iy, 0), S.c.gridY - 1);
    const int bin = col * S.c.gridY + row;
    w.keys[i] = bin;
    atomicAdd(&w.cell_count[S.cell_off + bin], 1);
}

// Block-level exclusive scan; block totals to `sums` (may be null).
__global__ void __launch_bounds__(1024) k_scan_block(const int *in, int *out, int *sums, long long n)
{
    __shared__ int sh[1024];
    const long long i = (long long)blockIdx.x * 1024 + threadIdx.x;
    const int v = i < n ? in[i] : 0;
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const int t = threadIdx.x >= off ? sh[threadIdx.x - off] : 0;
        __syncthreads();
        sh[threadIdx.x] += t;
        __syncthreads();
    }
    if (i < n) out[i] = sh[threadIdx.x] - v;
    if (sums && threadIdx.x == 1023) sums[blockIdx.x] = sh[1023];
}

__global__ void __launch_bounds__(1024) k_scan_add(int *out, const int *sums, long long n)
{
    const long long i = (long long)blockIdx.x * 1024 + threadIdx.x;
    if (i < n) out[i] += sums[blockIdx.x];
}

// cell_start = (global exclusive scan) - (scan at the scene's first cell) + pt_off
__global__ void __launch_bounds__(kBlock) k_cell_start(StepArgs a, BinWork w)
{
    const long long j = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (j >= w.n_cells_total) return;
    const int s = scene_of_cell(a.scenes, a.nscenes, j);
    const SceneDev &S = a.scenes[s];
    w.cell_start[j] = w.cell_count[j] - w.cell_count[S.cell_off] + (int)S.pt_off;
}

__global__ void __launch_bounds__(kBlock) k_scatter(StepArgs a, BinWork w)
{
    const long long i = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (i >= w.n_pts_total) return;
    const int bin = w.keys[i];
    if (bin < 0) return;
    const int s = scene_of_point(a.scenes, a.nscenes, i);
    const long long cell = a.scenes[s].cell_off + bin;
    const int slot = w.cell_start[cell] + atomicAdd(&w.cell_fill[cell], 1);
    w.perm[slot] = (int)i;
}

__global__ void __launch_bounds__(kBlock) k_sort_cells(StepArgs a, BinWork w)
{
    const long long j = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (j >= w.n_cells_total) return;
    const int s = scene_of_cell(a.scenes, a.nscenes, j);
    if (j - a.scenes[s].cell_off >= a.scenes[s].ncells) return;   // the per-scene end slot
    const int b = w.cell_start[j], e = w.cell_start[j + 1];
    for (int k = b + 1; k < e; k++) {
        const int v = w.perm[k];
        int m = k - 1;
        while (m >= b && w.perm[m] > v) { w.perm[m + 1] = w.perm[m]; m--; }
        w.perm[m + 1] = v;
    }
}

// Gathers the sorted points of every scene into dst; keys[] becomes the
// reference key of each sorted point.  Writes the new point counts.
template <typename T>
__global__ void __launch_bounds__(kBlock) k_gather(StepArgs a, BinWork w, const T *src, T *dst, int *sorted_keys)
{
    const long long j = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (j >= w.n_pts_total) return;
    const int s = scene_of_point(a.scenes, a.nscenes, j);
    const SceneDev &S = a.scenes[s];
    const int kept = w.cell_start[S.cell_off + S.ncells] - (int)S.pt_off;
    if (j == S.pt_off) w.scene_count[s] = kept;
    if (j - S.pt_off >= kept) return;
    const int from = w.perm[j];
#pragma unroll
    for (int line = 0; line < kNumPtsLines; line++) dst[line * a.pitch + j] = src[line * a.pitch + from];
    const int bin = w.keys[from];
    const int col = bin / S.c.gridY, row = bin % S.c.gridY;
    sorted_keys[j] = (col - S.c.halo + S.c.xoff) * S.c.gridY + row;
}

// Tile builder: half a wave per tile, a lane per column (tx <= 32).  Its
// launches have at most kBuildBlocks workgroups, which take the tiles in turn:
// a launch of 2^32 threads (2^27 tiles) and more is refused, and small pinned
// shapes on huge grids have up to 2^31 tiles.
constexpr int kTileLanes = 32, kBuildBlocks = 65536;

// Place of tile t of the table: its scene and first cell.
__device__ __forceinline__ const SceneDev &tile_place(const StepArgs &a, int t, int &scene, int &col0, int &row0)
{
    int lo = 0, hi = a.nscenes - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (a.scenes[mid].tile_off <= t) lo = mid;
        else hi = mid - 1;
    }
    const SceneDev &S = a.scenes[lo];
    const int local = t - S.tile_off;
    scene = lo;
    col0 = (local / S.n_tiles_y) * a.tx;
    row0 = (local % S.n_tiles_y) * a.ty;
    return S;
}

__device__ __forceinline__ int half_wave_min(int v)
{
#pragma unroll
    for (int k = kTileLanes / 2; k > 0; k >>= 1) v = min(v, __shfl_xor(v, k, kTileLanes));
    return v;
}

// f(t, k) for every tile t of the table, by its lanes k.
template <class F>
__device__ __forceinline__ void for_each_tile(int n_tiles_all, F &&f)
{
    const int k = threadIdx.x & (kTileLanes - 1);
    constexpr int per = kBlock / kTileLanes;
    for (long long t = (long long)blockIdx.x * per + threadIdx.x / kTileLanes; t < n_tiles_all;
         t += (long long)gridDim.x * per)
        f((int)t, k);
}

// 1 per tile that holds points.
__global__ void __launch_bounds__(kBlock) k_tile_count(StepArgs a, int n_tiles_all, int *tile_flag)
{
    for_each_tile(n_tiles_all, [&](int t, int k) {
        int sc, col0, row0;
        const SceneDev &S = tile_place(a, t, sc, col0, row0);
        int empty = 1;
        if (k < a.tx && col0 + k < S.c.ncols) {
            const int *cs = a.cell_start + S.cell_off + (long long)(col0 + k) * S.c.gridY;
            empty = cs[min(row0 + a.ty, S.c.gridY)] == cs[row0];
        }
        empty = half_wave_min(empty);
        if (k == 0) tile_flag[t] = !empty;
    });
}

// The box of a tile's cells that hold points, and the runs of the box's
// columns.  Each lane bisects its column: cell_start is nondecreasing, so the
// first and last occupied rows are found in log2(ty) steps (one thread per
// tile, column after column, took 12 us for any scene).
__device__ __forceinline__ void emit_tile(const StepArgs &a, int t, int k, int n_tiles_all, const int *tile_flag,
                                          const int *tile_pos, TileItem *tiles, TileRun *runs, int *weight,
                                          int tile_cost, int *n_tiles)
{
    const int live = tile_flag[t], pos = tile_pos[t];
    if (t == n_tiles_all - 1 && k == 0) *n_tiles = pos + live;
    if (!live) return;
    int sc, col0, row0;
    const SceneDev &S = tile_place(a, t, sc, col0, row0);
    const int rend = min(row0 + a.ty, S.c.gridY);
    int c_lo = kTileLanes, c_hi = 0, r_lo = a.ty, r_hi = 0, s0 = 0, n = 0;   // c_hi, r_hi: negated for the minimum
    if (k < a.tx && col0 + k < S.c.ncols) {
        const int *cs = a.cell_start + S.cell_off + (long long)(col0 + k) * S.c.gridY;
        s0 = cs[row0];
        const int s1 = cs[rend];
        n = s1 - s0;
        if (n > 0) {
            c_lo = k;
            c_hi = -k;
            int l = row0, h = rend - 1;           // first row r with cs[r + 1] > s0
            int l2 = row0, h2 = rend - 1;         // last row r with cs[r] < s1
            while (l < h || l2 < h2) {
                const int m = (l + h) >> 1, m2 = (l2 + h2 + 1) >> 1;
                const int v = cs[m + 1], v2 = cs[m2];
                if (l < h) {
                    if (v > s0) h = m;
                    else l = m + 1;
                }
                if (l2 < h2) {
                    if (v2 < s1) l2 = m2;
                    else h2 = m2 - 1;
                }
            }
            r_lo = l - row0;
            r_hi = -(l2 - row0);
        }
    }
    c_lo = half_wave_min(c_lo);
    c_hi = -half_wave_min(c_hi);
    r_lo = half_wave_min(r_lo);
    r_hi = -half_wave_min(r_hi);
    int end = n;   // inclusive prefix sum over the columns
#pragma unroll
    for (int o = 1; o < kTileLanes; o <<= 1) {
        const int v = __shfl_up(end, o, kTileLanes);
        if (k >= o) end += v;
    }
    const int total = __shfl(end, kTileLanes - 1, kTileLanes);
    if (k >= c_lo && k <= c_hi) {
        TileRun r;
        r.off = s0 - (end - n);
        r.end = end;
        runs[(long long)pos * a.tx + k - c_lo] = r;
    }
    if (k == 0) {
        TileItem it{};
        it.scene = sc;
        it.col0 = col0 + c_lo;
        it.row0 = row0 + r_lo;
        it.dims = (c_hi - c_lo + 1) | ((r_hi - r_lo + 1) << 16);
        it.total = total;
        it.runs = pos;
        tiles[pos] = it;
        weight[pos] = total + tile_cost;
    }
}

__global__ void __launch_bounds__(kBlock) k_tile_emit(StepArgs a, int n_tiles_all, const int *tile_flag,
                                                      const int *tile_pos, TileItem *tiles,
                                                      TileRun *runs, int *weight, int tile_cost, int *n_tiles)
{
    for_each_tile(n_tiles_all, [&](int t, int k) {
        emit_tile(a, t, k, n_tiles_all, tile_flag, tile_pos, tiles, runs, weight, tile_cost, n_tiles);
    });
}

// Smallest of the wave's values, in every lane.
__device__ __forceinline__ unsigned wave_min(unsigned v)
{
    // DPP: row_shr 1, 2, 4, 8 within 16 lanes, then row_bcast 15 and 31
    v = min(v, (unsigned)__builtin_amdgcn_update_dpp(-1, (int)v, 0x111, 0xf, 0xf, false));
    v = min(v, (unsigned)__builtin_amdgcn_update_dpp(-1, (int)v, 0x112, 0xf, 0xf, false));
    v = min(v, (unsigned)__builtin_amdgcn_update_dpp(-1, (int)v, 0x114, 0xf, 0xf, false));
    v = min(v, (unsigned)__builtin_amdgcn_update_dpp(-1, (int)v, 0x118, 0xf, 0xf, false));
    v = min(v, (unsigned)__builtin_amdgcn_update_dpp(-1, (int)v, 0x142, 0xa, 0xf, false));
    v = min(v, (unsigned)__builtin_amdgcn_update_dpp(-1, (int)v, 0x143, 0xc, 0xf, false));
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// Splits the tiles among the workgroups of a tile launch.  The table is cut
// into `parts` ranges, one per XCD (the workgroups of a range run on one XCD,
// see xcd_block), of equal count if no workgroup gets two tiles, else of equal
// summed weight (points, plus tile_cost per tile).  One workgroup per range.
//
// Where a workgroup gets at most kPackTiles tiles on average, each tile goes to
// the workgroup with the least weight so far, the heavy tiles first: the launch
// lasts as long as its most loaded workgroup, and the tiles of a scene of floes
// hold between 1 and all of their points (1.2M points of floes: 63.8 -> 54.5 us
// per substep in FP64, 57 -> 48 in the mixed form).  The order of weights is coarse
// (eighths of the largest) and full tiles count alike, so that tiles of about
// one size go in turn and workgroups at work at the same time are neighbours, whose window
// nodes overlap in the XCD's L2 (with neighbours one after the other in one
// workgroup instead, the launch of the 4M-point sheet was 13% slower at 14x32
// cells).
//
// Past that, and where there is at most one tile each, the workgroups take the
// range's tiles in turn: the loads then differ by little, and the assignment,
// which is serial, would take longer than it saves.  pre: exclusive prefix sums
// of the weights.
constexpr int kPackTiles = 8, kPackBins = 256, kPackLane = kPackBins / 64;

__global__ void __launch_bounds__(kBlock) k_tile_split(const TileItem *tiles, const int *weight, const int *pre,
                                                       const int *n_tiles, TileItem *list, TileWork *work, int n_work,
                                                       int n_few, int parts)
{
    static_assert(kPackBins == kBlock, "one workgroup's tile count per thread");
    __shared__ int base[kPackBins + 1];
    __shared__ int wt[kPackTiles * kPackBins], place[kPackTiles * kPackBins];   // of the range's tiles
    const int tid = threadIdx.x, n = *n_tiles, part = blockIdx.x;
    if (n_few > 0 && n <= n_few) n_work = n_few;
    const int per = n_work / parts;
    // first tile of range k: the first whose middle (doubled) reaches k parts of the weight
    auto start = [&](int k) {
        if (n <= n_work) return (int)((long long)n * k / parts);
        const unsigned long long w2 = 2ull * ((long long)pre[n - 1] + weight[n - 1]);
        int lo = 0, hi = n;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if ((2ull * pre[mid] + weight[mid]) * parts >= w2 * k) hi = mid;
            else lo = mid + 1;
        }
        return lo;
    };
    const int t0 = start(part), t1 = start(part + 1);
    const bool pack = n > n_work && per <= kPackBins && t1 - t0 <= kPackTiles * per;
    if (pack)
        for (int t = t0 + tid; t < t1; t += kBlock) wt[t - t0] = weight[t];
    __syncthreads();
    if (pack && tid < 64) {
        // workgroup b of the range is kept by lane b / J
        const int J = (per + 63) / 64;
        unsigned load[kPackLane];
        int count[kPackLane];
#pragma unroll
        for (int j = 0; j < kPackLane; j++) {
            load[j] = j < J && tid * J + j < per ? 0u : ~0u;
            count[j] = 0;
        }
        unsigned most = 1;
        for (int t = tid; t < t1 - t0; t += 64) most = max(most, (unsigned)wt[t]);
        most = ~wave_min(~most);
        for (int c = 7; c >= 0; c--) {
            for (int first = 0; first < t1 - t0; first += 64) {
                const int t = first + tid;
                const int w = t < t1 - t0 ? wt[t] : 0;
                const int cls = min(7, (int)(8.0f * (float)w / (float)most));
                for (unsigned long long m = __ballot(t < t1 - t0 && cls == c); m; m &= m - 1) {
                    const int i = __builtin_ctzll(m);
                    // (the full tiles count alike: theirs go in turn)
                    const unsigned wi = c == 7 ? most : (unsigned)__builtin_amdgcn_readlane(w, i);
                    const unsigned mine = min(min(load[0], load[1]), min(load[2], load[3]));
                    const unsigned least = wave_min(mine);
                    const int owner = __builtin_ctzll(__ballot(mine == least));
                    bool todo = tid == owner;
#pragma unroll
                    for (int j = 0; j < kPackLane; j++)
                        if (todo && load[j] == least) {
                            load[j] += wi;
                            place[first + i] = (tid * J + j) << 16 | count[j]++;
                            todo = false;
                        }
                }
            }
        }
#pragma unroll
        for (int j = 0; j < kPackLane; j++)
            if (j < J && tid * J + j < kPackBins) base[tid * J + j + 1] = count[j];
    }
    __syncthreads();
    if (!pack) {
        for (int t = t0 + tid; t < t1; t += kBlock) list[t] = tiles[t];
        for (int i = tid; i < per; i += kBlock) {
            TileWork out{};
            out.first = t0 + i;
            out.end = t1;
            out.step = per;
            if (out.first < out.end) out.item = tiles[out.first];
            work[part * per + i] = out;
        }
        return;
    }
    // counts to exclusive sums
    if (tid >= per) base[tid + 1] = 0;
    if (tid == 0) base[0] = 0;
    __syncthreads();
    for (int o = 1; o <= kPackBins; o <<= 1) {
        const int v = tid + 1 >= o ? base[tid + 1 - o] : 0;
        __syncthreads();
        if (tid + 1 >= o) base[tid + 1] += v;
        __syncthreads();
    }
    for (int t = t0 + tid; t < t1; t += kBlock) {
        const int p = place[t - t0];
        list[t0 + base[p >> 16] + (p & 0xffff)] = tiles[t];
    }
    __syncthreads();
    if (tid < per) {
        TileWork out{};
        out.first = t0 + base[tid];
        out.end = t0 + base[tid + 1];
        out.step = 1;
        if (out.first < out.end) out.item = list[out.first];
        work[part * per + tid] = out;
    }
}

// Tiles that hold points under each of several shapes, counted by their passes
// of kBlock points.  A workgroup's counts are kept in LDS.
struct CensusBlock {
    TileCensus *here;   // of shapes.n shapes
    __device__ __forceinline__ void clear(int n)
    {
        for (int i = threadIdx.x; i < n * TileCensus::kPasses; i += kBlock)
            here[i / TileCensus::kPasses].tiles[i % TileCensus::kPasses] = 0;
        if ((int)threadIdx.x < n) here[threadIdx.x].most = here[threadIdx.x].points = 0;
        __syncthreads();
    }
    __device__ __forceinline__ void add(int shape, int points)
    {
        const int passes = (points + kBlock - 1) / kBlock;
        atomicAdd(&here[shape].tiles[min(passes, TileCensus::kPasses) - 1], 1);
        atomicMax(&here[shape].most, passes);
        atomicAdd(&here[shape].points, points);
    }
    __device__ __forceinline__ void flush(int n, TileCensus *out)
    {
        __syncthreads();
        for (int k = threadIdx.x; k < n * TileCensus::kPasses; k += kBlock) {
            const int i = k / TileCensus::kPasses, q = k % TileCensus::kPasses;
            if (here[i].tiles[q]) atomicAdd(&out[i].tiles[q], here[i].tiles[q]);
        }
        if ((int)threadIdx.x < n && here[threadIdx.x].points) {
            atomicMax(&out[threadIdx.x].most, here[threadIdx.x].most);
            atomicAdd(&out[threadIdx.x].points, here[threadIdx.x].points);
        }
    }
};

// By the cells: a thread per tile of shape blockIdx.y adds up its columns.
__global__ void __launch_bounds__(kBlock) k_tile_census_cells(StepArgs a, TileShapes shapes, TileCensus *out)
{
    __shared__ TileCensus one;
    CensusBlock b{&one};
    b.clear(1);
    const int tx = shapes.tx[blockIdx.y], ty = shapes.ty[blockIdx.y], tid = threadIdx.x;
    for (int sc = 0; sc < a.nscenes; sc++) {
        const SceneDev &S = a.scenes[sc];
        const int ntx = (S.c.ncols + tx - 1) / tx, nty = (S.c.gridY + ty - 1) / ty;
        const long long n = (long long)ntx * nty;
        for (long long t = (long long)blockIdx.x * kBlock + tid; t < n; t += (long long)gridDim.x * kBlock) {
            const int col0 = (int)(t / nty) * tx, row0 = (int)(t % nty) * ty, rend = min(row0 + ty, S.c.gridY);
            int points = 0;
            for (int c = col0; c < min(col0 + tx, S.c.ncols); c++) {
                const int *cs = a.cell_start + S.cell_off + (long long)c * S.c.gridY;
                points += cs[rend] - cs[row0];
            }
            if (points) b.add(0, points);
        }
    }
    b.flush(1, out + blockIdx.y);
}

// By the sorted points, whose keys say where a run of one tile's points in one
// column starts: the thread of the tile's first such point adds up its columns.
__global__ void __launch_bounds__(kBlock) k_tile_census_points(StepArgs a, BinWork w, TileShapes shapes, TileCensus *out)
{
    __shared__ TileCensus all[TileShapes::kMax];
    CensusBlock b{all};
    b.clear(shapes.n);
    for (long long j = (long long)blockIdx.x * kBlock + threadIdx.x; j < w.n_pts_total; j += (long long)gridDim.x * kBlock) {
        const SceneDev &S = a.scenes[scene_of_point(a.scenes, a.nscenes, j)];
        const int *const cells = a.cell_start + S.cell_off, gridY = S.c.gridY, ncols = S.c.ncols;
        if (j >= cells[S.ncells]) continue;   // past the scene's points
        const bool first_point = j == S.pt_off;
        const int key = w.sorted_keys[j], before = first_point ? key : w.sorted_keys[j - 1];
        if (!first_point && key == before) continue;
        const int shift = (S.c.halo - S.c.xoff) * gridY;
        const int col = (key + shift) / gridY, row = (key + shift) % gridY;
        const int col_b = (before + shift) / gridY, row_b = (before + shift) % gridY;
        for (int i = 0; i < shapes.n; i++) {
            const int tx = shapes.tx[i], ty = shapes.ty[i];
            const int row0 = row / ty * ty, rend = min(row0 + ty, gridY);
            if (!first_point && col_b == col && row_b >= row0) continue;   // the same tile
            const int col0 = col / tx * tx, cend = min(col0 + tx, ncols);
            int points = 0;
            for (int c = col0; c < cend; c++) {
                const int *cs = cells + (long long)c * gridY;
                const int n = cs[rend] - cs[row0];
                if (c < col && n > 0) {   // an earlier point's tile
                    points = 0;
                    break;
                }
                points += n;
            }
            if (points) b.add(i, points);
        }
    }
    b.flush(shapes.n, out);
}

inline unsigned nblk(long long n, int b) { return (unsigned)((n + b - 1) / b); }

}  // namespace

// Exclusive scan of n ints (in may equal out), multi-level.
hipError_t scan_exclusive(const int *in, int *out, long long n, int *tmp, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    const long long nb = (n + 1023) / 1024;
    if (nb == 1) {
        hipLaunchKernelGGL(k_scan_block, dim3(1), dim3(1024), 0, s, in, out, nullptr, n);
        return hipGetLastError();
    }
    int *sums = tmp;
    hipLaunchKernelGGL(k_scan_block, dim3((unsigned)nb), dim3(1024), 0, s, in, out, sums, n);
    hipError_t e = scan_exclusive(sums, sums, nb, tmp + nb, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_scan_add, dim3((unsigned)nb), dim3(1024), 0, s, out, sums, n);
    return hipGetLastError();
}

hipError_t launch_sort(const StepArgs &a, const SceneDev *host_scenes, int nscenes, BinWork &w, int elem_bytes,
                       void *pts_src, void *pts_dst, hipStream_t s)
{
    (void)host_scenes;
    (void)nscenes;
    hipError_t e;
    const size_t cbytes = (size_t)w.n_cells_total * sizeof(int);
    if ((e = launch_fill_zero(w.cell_count, cbytes, s)) != hipSuccess) return e;
    if ((e = launch_fill_zero(w.cell_fill, cbytes, s)) != hipSuccess) return e;
    const unsigned gp = nblk(w.n_pts_total, kBlock), gc = nblk(w.n_cells_total, kBlock);
    if (elem_bytes == 8) hipLaunchKernelGGL(k_keys<8>, dim3(gp), dim3(kBlock), 0, s, a, w, pts_src);
    else hipLaunchKernelGGL(k_keys<4>, dim3(gp), dim3(kBlock), 0, s, a, w, pts_src);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = scan_exclusive(w.cell_count, w.cell_count, w.n_cells_total, w.scan_tmp, s)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_cell_start, dim3(gc), dim3(kBlock), 0, s, a, w);
    hipLaunchKernelGGL(k_scatter, dim3(gp), dim3(kBlock), 0, s, a, w);
    hipLaunchKernelGGL(k_sort_cells, dim3(gc), dim3(kBlock), 0, s, a, w);
    if (elem_bytes == 8)
        hipLaunchKernelGGL(k_gather<double>, dim3(gp), dim3(kBlock), 0, s, a, w, (const double *)pts_src,
                           (double *)pts_dst, w.sorted_keys);
    else
        hipLaunchKernelGGL(k_gather<unsigned>, dim3(gp), dim3(kBlock), 0, s, a, w, (const unsigned *)pts_src,
                           (unsigned *)pts_dst, w.sorted_keys);
    return hipGetLastError();
}

// By the points where there are more than 10 cells per point: 160k points on
// 16384 x 16384 cells take 26 us by the points, 1040 by the cells (all of them
// are read for each of seven shapes), 4.0M points on 1.1M cells 122 and 17.
hipError_t launch_tile_census(const StepArgs &a, const TileShapes &shapes, const BinWork &w, TileCensus *out,
                              hipStream_t s)
{
    const hipError_t e = launch_fill_zero(out, sizeof(TileCensus) * shapes.n, s);
    if (e != hipSuccess) return e;
    if (w.n_cells_total > 10 * w.n_pts_total) {
        const unsigned g = std::min(nblk(std::max<long long>(w.n_pts_total, 1), kBlock), 2048u);
        hipLaunchKernelGGL(k_tile_census_points, dim3(g), dim3(kBlock), 0, s, a, w, shapes, out);
    } else {
        const unsigned g = (unsigned)std::min<long long>(std::max<long long>(w.n_cells_total / (32 * kBlock), 1), 256);
        hipLaunchKernelGGL(k_tile_census_cells, dim3(g, shapes.n), dim3(kBlock), 0, s, a, shapes, out);
    }
    return hipGetLastError();
}

// The parts of a tile table of max_tiles places in one allocation, no more of
// which than there are points can hold any (a small shape on a huge grid has
// many times more places): the
// workgroups' work, the items, their runs, the tile count, and the builder's
// own ints (scene offsets, flags, positions or weight sums, weights, scan sums).
size_t tile_table_layout(char *base, long long max_tiles, long long max_points, int tx, int n_work, TileTable &t)
{
    size_t at = 0;
    auto part = [&](size_t bytes) {
        char *p = base + at;
        at = (at + bytes + 63) / 64 * 64;
        return p;
    };
    const long long live = std::min(max_tiles, max_points);
    t.max_tiles = max_tiles;
    t.max_live = live;
    t.n_work = n_work;
    t.work = (TileWork *)part(sizeof(TileWork) * n_work);
    t.tiles = (TileItem *)part(sizeof(TileItem) * live);
    t.list = (TileItem *)part(sizeof(TileItem) * live);
    t.runs = (TileRun *)part(sizeof(TileRun) * tx * live);
    t.n_tiles = (int *)part(sizeof(int));
    t.flag = (int *)part(sizeof(int) * max_tiles);
    t.pos = (int *)part(sizeof(int) * max_tiles);
    t.weight = (int *)part(sizeof(int) * live);
    t.scan_tmp = (int *)part(sizeof(int) * (max_tiles / 1000 + 64));
    return at;
}

hipError_t launch_build_tiles(const StepArgs &a, const SceneDev *host_scenes, int nscenes, long long n_points,
                              const TileTable &t, hipStream_t s)
{
    long long total = 0;
    for (int i = 0; i < nscenes; i++) total += (long long)host_scenes[i].n_tiles_x * host_scenes[i].n_tiles_y;
    if (total > t.max_tiles || total == 0 || a.tx > kTileLanes || t.n_work <= 0) return hipErrorInvalidValue;
    // a tile's staging and flush cost about as much as 250 points (the sums of
    // the weights stay below 2^31)
    const int tile_cost = (int)std::max<long long>(0, std::min<long long>(250, (0x7fffffff - n_points) / total - 1));
    hipError_t e;
    const unsigned g = std::min(nblk(total * kTileLanes, kBlock), (unsigned)kBuildBlocks);
    hipLaunchKernelGGL(k_tile_count, dim3(g), dim3(kBlock), 0, s, a, (int)total, t.flag);
    // positions of the non-empty tiles: exclusive scan of the 0/1 flags
    if ((e = scan_exclusive(t.flag, t.pos, total, t.scan_tmp, s)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_tile_emit, dim3(g), dim3(kBlock), 0, s, a, (int)total, t.flag, t.pos, t.tiles,
                       t.runs, t.weight, tile_cost, t.n_tiles);
    // (weights past the live tiles are not read from the sums)
    if ((e = scan_exclusive(t.weight, t.pos, std::min(total, t.max_live), t.scan_tmp, s)) != hipSuccess) return e;
    const int parts = t.n_work % 8 ? 1 : 8;
    hipLaunchKernelGGL(k_tile_split, dim3(parts), dim3(kBlock), 0, s, t.tiles, t.weight, t.pos, t.n_tiles, t.list,
                       t.work, t.n_work, t.n_few, parts);
    return hipGetLastError();
}

}  // namespace icempm
