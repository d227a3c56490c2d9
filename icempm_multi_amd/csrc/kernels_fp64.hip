// kernels_fp64.hip -- FP64 binned P2G / G2P tile kernels for gfx950 (CDNA4).
//
// Replaces partition_kernel_p2g and partition_kernel_g2p
// (simulation/kernels.cuh:46-122, 305-414); the grid update between them is in
// kernels_fp64_update.hip.
//
// Layout: points are the reference's SoA (16 lines of `pitch` doubles); each
// scene's grid is 3 lines (mass, momentum->velocity x, y) of `gpitch`
// doubles with node (col, row) at col*gridY + row, col = gx + halo.
//
// The binned kernels work on tiles of TX x TY cells: a workgroup stages the
// grid velocities of the tile's node window in LDS (G2P gathers), and sums
// the P2G contributions of the tile's points in an LDS window (ds_add_f64)
// that is flushed with one global atomic per touched node and line.  The
// point runs of a tile come from the cell_start table of the last sort; a
// point that drifted out of the window since then falls back to global memory.
//
// Products and sums may contract to FMA (as the reference's nvcc build does by
// default); the FP64 oracle rounds each operation, so the two agree to a few
// ulps per operation plus the reordering of the atomic sums.
#include <hip/hip_runtime.h>

#include "kernels.h"
#include "point_fp64.h"
#include "tile_common.h"

namespace icempm {
namespace fp64 {

// A point set aside by its tile (its G2P stencil left the tile's LDS window):
// G2P from the momenta of grid rb with every node velocity formed from global
// memory, the state stored as the tile kernel stores it, and (p2g) P2G into
// grid wb with global atomics.
__device__ __forceinline__ void deferred_point(const StepArgs &a, bool p2g, int rb, int wb, int pt)
{
    const PtRef R{(double *)a.pts, a.pitch};
    const int sc = a.defer_scene[pt];
    const SceneDev &S = a.scenes[sc];
    const SceneConsts &c = S.c;
    const SceneClock clk = next_clock(c, a.clocks[sc]);
    const bool record = (clk.step % c.update_every) == 0;
    long long ud = as_ll(R.at(kLineUtility, pt));
    double x, y, F[4], Jp, v[2], B[4], pp, qq;
    load_state(R, pt, x, y, F, Jp);
    unsigned e;
    StressTerms terms;
    terms.valid = false;
    const glb_d *gr = (const glb_d *)(a.grid_mem + S.grid_off[rb]);
    if (!g2p_point(c, (const glb_d *)S.fail_tab, gr, S.gpitch, &clk, nullptr, 0, 0, 0, 0, 0, false, x, y, v, B, F, Jp,
                   ud, pp, qq, e, terms)) {
        atomicMax(&a.err[sc], e);
        return;
    }
    if (!p2g) {
        store_state(R, pt, x, y, v, F, B, Jp, ud, record, pp, qq);
        return;
    }
    store_state_fused(R, pt, x, y, F, Jp, ud, record, pp, qq);
    glb_d *gw = (glb_d *)(a.grid_mem + S.grid_off[wb]);
    const long long gp = S.gpitch;
    const int gridY = c.gridY;
    P2GStencil st;
    const unsigned e2 = p2g_stencil(c, x, y, v, B, F, Jp, ud, terms, st);
    if (e2) {
        atomicMax(&a.err[sc], e2);
        return;
    }
    st.nodes(c, [&](int i, int j, double dm, double dpx, double dpy) {
        const long long gi = (long long)(st.bxc + i) * gridY + st.by + j;
        glb_add(gw + gi, dm);
        glb_add(gw + gp + gi, dpx);
        glb_add(gw + 2 * gp + gi, dpy);
        mark_dirty(a, S, wb, gi);
    });
}

// Waves per SIMD the tile kernel is built for; the second for launches whose
// tiles all run at once at two (StepArgs::few): 25.6k points 7.1 us per substep,
// 8.0 with three; the 4M-point sheet 140 with two, 127 with three.
constexpr int kWaves = 3, kWavesFew = 2;

// ---------------------------------------------------------------------------
// Binned tile kernel: G2P from grid[rbuf] and/or P2G into grid[wbuf].
// 3 waves per SIMD (up to 168 VGPRs; the fused kernel spills 7 outside the
// point loop), or 2 (181 VGPRs, none) for launches of few workgroups.
// What keeps it there: the scene invariants of the point loop (4/h, kappa/2,
// sqrt(2) mu, the failure-surface and tension-branch terms) come from the host
// in scalar registers, and the water stress uses J^-5 = 1/(J^2 J^2 J) rather
// than pow(), whose polynomial constants the compiler would otherwise keep in
// vector registers across the loop (242 VGPRs, 2 waves per SIMD, before).
// ---------------------------------------------------------------------------
//
// WHC is the LDS row stride, the height of the largest window (ty + 2 +
// 2*margin), when fixed at compile time for the common tile shapes (0: read
// from the arguments).  A compile-time stride turns the stencil's LDS offsets
// into instruction immediates.  A tile's window covers the box of its cells
// that held points at the last sort (TileItem), so it may be smaller.
//
// With kTileFromMomenta (the chain of a stepping call) grid[rbuf] holds the
// momenta of the last P2G: the staging forms each window node's velocity
// (the grid update of kernels.cuh:164-301, per node), the launch clears
// grid[zbuf] for the next P2G, adds the indenter force and writes the advanced
// clocks to the other slot.  Without it grid[rbuf] holds velocities.
template <int MODE, int WHC, int WAVES>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(WAVES)))
k_tiles(StepArgs a, int rbuf, int wbuf, int zbuf, int record_mode)
{
    constexpr bool DO_G2P = (MODE & kTileG2P) != 0;
    constexpr bool DO_P2G = (MODE & kTileP2G) != 0;
    constexpr bool FROM_M = (MODE & kTileFromMomenta) != 0;
    extern __shared__ __attribute__((aligned(16))) double lds_raw[];
    __shared__ TileRun runs_raw[kMaxTX];
    __shared__ double ftab[kFailTab];   // failure-surface table of the tile's scene
    lds_run *const runs = (lds_run *)runs_raw;

    // The LDS regions hold the largest window, a.win_w columns of WS nodes; a
    // tile's own window (TileWindow) takes its first columns and rows.
    const int WS = WHC > 0 ? WHC : a.win_h;
    const int WNmax = a.win_w * WS;
    lds_d *lds = (lds_d *)lds_raw;
    lds_d *vw = lds;                            // 2*WNmax: (vx, vy) per window node
    // Two accumulation windows of 3*WNmax, (m, px, py) per node: even lanes add
    // into the first, odd lanes into the second.  The adjacent lanes of a
    // 16-lane row hold points 4 apart in the sorted order, which share a cell
    // (and so every LDS address) whenever the cell holds more than 4 points;
    // with a window each they never collide.  The flush adds the two.
    lds_d *acc = lds + (DO_G2P ? 2 * WNmax : 0);
    lds_d *const acc_lane = acc + ((threadIdx.x & 1) ? 3 * WNmax : 0);
    const int tid = threadIdx.x;
    const PtRef R{(double *)a.pts, a.pitch};
    int block = blockIdx.x;
    if (!FROM_M) stamp_begin(a);
    if (FROM_M && side_work(a, rbuf, zbuf, block)) return;
    const int n_blocks = a.n_work;
    TileWork work = scalar_load(a.tile_work + xcd_block(block, n_blocks));

    // Tile distribution.  Static: the tiles of the workgroup's TileWork.
    // Dynamic: each XCD (block % 8, the hardware's round-robin dispatch order)
    // owns a contiguous eighth of the tile list; its blocks pull tiles with an
    // atomic counter and then help the other XCDs' ranges.  Every block counts
    // itself done once at the end; the last one clears the counters for the
    // next launch.
    __shared__ int s_tile;
    const bool dyn = a.dyn_tiles != 0;
    const int nq = (n_blocks >= 8 && (n_blocks & 7) == 0) ? 8 : 1;
    const int q0 = nq == 8 ? (block & 7) : 0;
    int qk = 0;                      // queues visited so far (dynamic)
    int aside = -1;                  // first of the points this thread set aside
    int tab_scene = -1;              // scene whose failure table ftab holds
    for (;;) {
        if (dyn) {
            const int ntiles = scalar_copy(a.n_tiles);
            if (tid == 0) {
                int t = -1;
                for (; qk < nq; qk++) {
                    const int q = (q0 + qk) % nq;
                    const int hi = (int)((long long)ntiles * (q + 1) / nq);
                    const int got = (int)((long long)ntiles * q / nq) + atomicAdd(a.tile_queue + q, 1);
                    if (got < hi) { t = got; break; }
                }
                s_tile = t;
            }
            __syncthreads();
            work.first = __builtin_amdgcn_readfirstlane(s_tile);   // uniform: keeps tile data in scalar registers
            if (work.first < 0) break;
            work.end = work.first + 1;
            work.step = 1;
            work.item = scalar_load(a.tiles + work.first);
        }
        // a lone scene's data is loaded without waiting for the tile item
        const SceneDev *S = a.scenes;
        const SceneClock *clock = a.clocks;
        if (a.nscenes > 1) {
            asm volatile("");
            S += work.item.scene;
            clock += work.item.scene;
        }
        SceneLanes sl;
        sl.load(S);
        SceneClock clk = scalar_load(clock);
        pin(work);
        if (work.first >= work.end) break;
        const TileItem ti = work.item;
        // What the tile's loads need first; the rest of the constants are read
        // out of the lanes while those loads are under way.  The serial start is
        // what bounds a small scene: 7.5 -> 6.8 us per substep at 1.6k points,
        // 25.1 -> 24.0 us at 410k.
        const int gridY = sl.copy<int>(offsetof(SceneDev, c) + offsetof(SceneConsts, gridY));
        const int ncols = sl.copy<int>(offsetof(SceneDev, c) + offsetof(SceneConsts, ncols));
        const long long gp = sl.copy<long long>(offsetof(SceneDev, gpitch));
        char *const grids = a.grid_mem + sl.copy<long long>(offsetof(SceneDev, grid_off));
        const glb_d *gr = (const glb_d *)(grids + rbuf * a.grid_buf_bytes);
        glb_d *gw = (glb_d *)(grids + wbuf * a.grid_buf_bytes);
        const TileWindow W(ti, a.margin);
        const int wc0 = W.c0, wr0 = W.r0, win_w = W.w, win_h = W.h, WN = W.nodes();
        const int ncol = ti.dims & 0xffff, total = ti.total;

        // The loads of a tile are issued before any is waited for: the point
        // runs, a new scene's table, the window's momenta, and (after the runs are in LDS) the
        // first points.  kU window nodes per thread cover any window that fits the
        // LDS (64 B per node of 64 KiB).
        constexpr int kU = 4;
        double m[kU], px[kU], py[kU];
        TileRun my_run{0, kRunEnd};
        if (tid < ncol) my_run = a.tile_runs[(long long)ti.runs * a.tx + tid];
        static_assert(kFailTab <= kBlock, "one table entry per thread");
        const bool new_table = DO_G2P && ti.scene != tab_scene;
        double my_fail = 0;
        if (new_table && tid < kFailTab) my_fail = S->fail_tab[tid];
        if (DO_G2P && FROM_M) {
#pragma unroll
            for (int u = 0; u < kU; u++) {
                m[u] = px[u] = py[u] = 0;
                if (u * kBlock >= WN) continue;   // uniform
                const int i = tid + u * kBlock;
                const int qc = W.col_of(i), qr = i - qc * win_h;
                const int col = wc0 + qc, row = wr0 + qr;
                const bool in = i < WN && col >= 0 && col < ncols && row >= 0 && row < gridY;
                const long long gi = (long long)col * gridY + row;
                m[u] = in ? (double)gr[gi] : 0.0;
                px[u] = in ? (double)gr[gp + gi] : 0.0;
                py[u] = in ? (double)gr[2 * gp + gi] : 0.0;
            }
        }
        const SceneConsts c = sl.copy<SceneConsts>(offsetof(SceneDev, c));
        int *const dflag = a.dirty + wbuf * a.dirty_stride + sl.copy<long long>(offsetof(SceneDev, seg_off));
        // the substep's clock: advanced here from the current slot, or already
        // advanced by the grid update
        pin(clk);
        if (FROM_M) clk = next_clock(c, clk);
        bool record = false;
        if (DO_G2P) record = record_mode >= 0 ? record_mode != 0 : (clk.step % c.update_every) == 0;
        // The runs of the last tile were last read in its point loop, before
        // the barrier that precedes its flush (the barrier at the end of the
        // tile where there is no flush).
        if (tid < kMaxTX) {
            runs[tid].off = my_run.off;
            runs[tid].end = my_run.end;
        }
        // the failure-surface table of the tile's scene, kept while the scene
        // stays the same
        if (new_table) {
            if (tid < kFailTab) ftab[tid] = my_fail;
            tab_scene = ti.scene;
        }
        __syncthreads();   // runs and table in LDS; the last tile's window is flushed

        // points of the tile, strided over the workgroup: consecutive lanes take
        // consecutive points of a run, so every SoA access is coalesced
        unsigned err = 0;
        RunCursor cursor;
        // lane_spread: the lanes of one atomic instruction then hold points of
        // different cells (about 4 points per cell), so their LDS targets differ.
        //   0: lane l takes point l of its wave's 64-point group;
        //   1: point (l%16)*4 + l/16 of the group (16 cells per group);
        //   2: the wave takes a 128-point group in two passes, lane l taking
        //      point (l%32)*4 + l/32, plus 2 in the second pass (32 cells).
        static_assert(kBlock == 256, "lane spread 2 assumes 4 waves of 64");
        const int lane = tid & 63, wave = tid >> 6;
        const int n_it = a.lane_spread == 2 ? 2 * ((total + 2 * kBlock - 1) / (2 * kBlock))
                                            : (total + kBlock - 1) / kBlock;
        // the tile's point of this lane and iteration
        auto lane_point = [&](int it) {
            if (a.lane_spread == 2)
                return (it >> 1) * (2 * kBlock) + wave * 128 + ((lane & 31) << 2) + (lane >> 5) + 2 * (it & 1);
            if (a.lane_spread == 1) return it * kBlock + (wave << 6) + ((lane & 15) << 2) + (lane >> 4);
            return it * kBlock + tid;
        };
        // its SoA index; false past the end
        auto locate = [&](int it, long long &pt) -> bool {
            const int k = lane_point(it);
            if (k >= total) return false;
            pt = (unsigned)cursor.point(runs, k);
            return true;
        };
        // P2G of one point (kernels.cuh:59-121) into the LDS window, or into
        // global memory for the nodes outside it (a point that drifted since
        // the sort)
        auto p2g_emit = [&](double x, double y, const double v[2], const double B[4], const double F[4], double Jp,
                            long long ud, const StressTerms &terms) {
            P2GStencil st;
            const unsigned e = p2g_stencil(c, x, y, v, B, F, Jp, ud, terms, st);
            if (e) {
                err = max(err, e);
                return;
            }
            const int lx = st.bxc - wc0, ly = st.by - wr0;
            if (lx >= 0 && lx + 2 < win_w && ly >= 0 && ly + 2 < win_h) {
                lds_d *const p0 = acc_lane + 3 * (lx * WS + ly);
                st.nodes(c, [&](int i, int j, double dm, double dpx, double dpy) {
                    lds_d *const p = p0 + 3 * (i * WS + j);
                    lds_add(p, dm);
                    lds_add(p + 1, dpx);
                    lds_add(p + 2, dpy);
                });
            } else {
                st.nodes(c, [&](int i, int j, double dm, double dpx, double dpy) {
                    if (lx + i >= 0 && lx + i < win_w && ly + j >= 0 && ly + j < win_h) {
                        lds_d *const p = acc_lane + 3 * ((lx + i) * WS + ly + j);
                        lds_add(p, dm);
                        lds_add(p + 1, dpx);
                        lds_add(p + 2, dpy);
                    } else {
                        const long long gi = (long long)(st.bxc + i) * gridY + st.by + j;
                        glb_add(gw + gi, dm);
                        glb_add(gw + gp + gi, dpx);
                        glb_add(gw + 2 * gp + gi, dpy);
                        dflag[gi >> kSegShift] = 1;
                    }
                });
            }
        };
        // The state of the next point is loaded while the current one is
        // computed.  Its index is located one iteration earlier still: the
        // lookup reads LDS, and LDS reads wait for this wave's earlier LDS
        // atomics, so it is done after the loads are issued.
        long long pt_n = 0, ud_n = 0, pt_nn = 0;
        double x_n = 0, y_n = 0, F_n[4] = {0, 0, 0, 0}, Jp_n = 0;
        bool ok_n = lane_point(0) < total;
        if (ok_n) {
            pt_n = (unsigned)cursor.seek(runs, ncol, lane_point(0));
            ud_n = as_ll(R.at(kLineUtility, pt_n));
            load_state(R, pt_n, x_n, y_n, F_n, Jp_n);
        }

        // node velocities into LDS, accumulation windows cleared
        if (DO_G2P && FROM_M) {
#pragma unroll
            for (int u = 0; u < kU; u++) {
                const int i = tid + u * kBlock;
                if (u * kBlock >= WN) break;      // uniform
                if (i >= WN) break;
                const int qc = W.col_of(i), qr = i - qc * win_h;
                double vx = 0, vy = 0;
                if (m[u] != 0)
                    node_velocity(c, clk, nullptr, wc0 + qc - c.halo + c.xoff, wr0 + qr, m[u], px[u], py[u], vx, vy);
                const int li = qc * WS + qr;
                vw[2 * li] = vx;
                vw[2 * li + 1] = vy;
            }
        }
        if (DO_G2P && !FROM_M) {
            for (int i = tid; i < WN; i += kBlock) {
                const int qc = W.col_of(i), qr = i - qc * win_h, li = qc * WS + qr;
                const int col = wc0 + qc, row = wr0 + qr;
                double vx = 0, vy = 0;
                if (col >= 0 && col < c.ncols && row >= 0 && row < gridY) {
                    const long long gi = (long long)col * gridY + row;
                    vx = gr[gp + gi];
                    vy = gr[2 * gp + gi];
                }
                vw[2 * li] = vx;
                vw[2 * li + 1] = vy;
            }
        }
        if (DO_P2G) {
            // both windows, whole: 16 bytes per thread and store
            typedef double d2 __attribute__((ext_vector_type(2)));
            typedef __attribute__((address_space(3))) d2 lds_d2;
            lds_d2 *const z = (lds_d2 *)acc;
            for (int i = tid; i < 3 * WNmax; i += kBlock) z[i] = d2{0, 0};
        }
        bool ok_nn = n_it > 1 && locate(1, pt_nn);
        __syncthreads();
#pragma unroll 1
        for (int it = 0; it < n_it; it++) {
            const bool ok = ok_n;
            const long long pt = pt_n;
            long long ud = ud_n;
            double x = x_n, y = y_n, F[4] = {F_n[0], F_n[1], F_n[2], F_n[3]}, Jp = Jp_n;
            ok_n = ok_nn;
            pt_n = pt_nn;
            if (ok_n) {
                ud_n = as_ll(R.at(kLineUtility, pt_n));
                load_state(R, pt_n, x_n, y_n, F_n, Jp_n);
            }
            ok_nn = it + 2 < n_it && locate(it + 2, pt_nn);
            if (!ok) continue;
            if (ud & kDisabled) continue;
            double v[2], B[4];
            StressTerms terms;   // stress terms of F, passed from G2P to P2G
            terms.valid = false;
            if (DO_G2P) {
                double pp, qq;
                unsigned e;
                // With velocities formed from momenta, a point whose G2P
                // stencil leaves the LDS window (it drifted since the sort)
                // is set aside: its thread handles it after its tiles
                // (forming node velocities from global memory here would add
                // to the point loop's registers).
                if (!g2p_point(c, (const lds_d *)ftab, gr, gp, nullptr, vw, wc0, wr0, win_w, win_h, WS, FROM_M, x, y, v, B,
                               F, Jp, ud, pp, qq, e, terms)) {
                    if (e) {
                        err = max(err, e);
                    } else {
                        a.defer_next[pt] = aside;
                        a.defer_scene[pt] = ti.scene;
                        aside = (int)pt;
                    }
                    continue;
                }
                if (DO_P2G) store_state_fused(R, pt, x, y, F, Jp, ud, record, pp, qq);
                else store_state(R, pt, x, y, v, F, B, Jp, ud, record, pp, qq);
            } else {
                v[0] = R.at(kLineVelX, pt);
                v[1] = R.at(kLineVelX + 1, pt);
#pragma unroll
                for (int m = 0; m < 4; m++) B[m] = R.at(kLineBp00 + m, pt);
            }
            if (DO_P2G) p2g_emit(x, y, v, B, F, Jp, ud, terms);
        }
        if (err) atomicMax(&a.err[ti.scene], err);
        work.first += work.step;
        if (work.first < work.end) work.item = scalar_load(a.tile_list + work.first);
        __syncthreads();
        if (DO_P2G) {
            for (int i = tid; i < WN; i += kBlock) {
                const int qc = W.col_of(i), qr = i - qc * win_h, li = qc * WS + qr;
                const double m = acc[3 * li] + acc[3 * WNmax + 3 * li];
                if (m == 0) continue;
                const int col = wc0 + qc, row = wr0 + qr;
                if (col < 0 || col >= c.ncols || row < 0 || row >= gridY) continue;
                const long long gi = (long long)col * gridY + row;
                glb_add(gw + gi, m);
                glb_add(gw + gp + gi, acc[3 * li + 1] + acc[3 * WNmax + 3 * li + 1]);
                glb_add(gw + 2 * gp + gi, acc[3 * li + 2] + acc[3 * WNmax + 3 * li + 2]);
                dflag[gi >> kSegShift] = 1;
            }
        }
        if (!dyn && work.first >= work.end) break;   // before the next tile's loads
    }
    if (dyn && tid == 0) {
        if (atomicAdd(a.tile_queue + 8, 1) == n_blocks - 1)
            for (int k = 0; k < 9; k++) a.tile_queue[k] = 0;
    }
    if (FROM_M) {
        // The points this thread set aside.  Their G2P reads grid[rbuf], which
        // was complete before the launch, and their P2G adds into grid[wbuf]
        // with atomics, so nothing of the other threads' work is needed.
        while (aside >= 0) {
            const int pt = aside;
            aside = a.defer_next[pt];
            deferred_point(a, DO_P2G, rbuf, wbuf, pt);
        }
    } else {
        stamp_end(a);
    }
}

size_t tile_lds_bytes(const StepArgs &a, int mode)
{
    const size_t WN = (size_t)a.win_w * a.win_h;
    size_t n = 0;
    if (mode & kTileG2P) n += 2 * WN;
    if (mode & kTileP2G) n += 6 * WN;   // two accumulation windows
    return n * sizeof(double);
}

// window heights compiled in: ty = 16, 32, 64 with a drift margin of 1 or 0, and 8 with 1
template <int MODE, int WAVES>
static hipError_t launch_tiles_wh(const StepArgs &a, int rbuf, int wbuf, int zbuf, int record_mode, size_t lds,
                                  hipStream_t s)
{
    auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(tile_grid(a, MODE)), dim3(kBlock), lds, s, a, rbuf, wbuf, zbuf, record_mode);
    };
    switch (a.win_h) {
    case 12: run(k_tiles<MODE, 12, WAVES>); break;
    case 18: run(k_tiles<MODE, 18, WAVES>); break;
    case 20: run(k_tiles<MODE, 20, WAVES>); break;
    case 34: run(k_tiles<MODE, 34, WAVES>); break;
    case 36: run(k_tiles<MODE, 36, WAVES>); break;
    case 66: run(k_tiles<MODE, 66, WAVES>); break;
    case 68: run(k_tiles<MODE, 68, WAVES>); break;
    default: run(k_tiles<MODE, 0, WAVES>); break;
    }
    return hipGetLastError();
}

hipError_t launch_tiles(const StepArgs &a, int mode, int rbuf, int wbuf, int zbuf, int record_mode, hipStream_t s)
{
    if (a.tx > kMaxTX || a.n_work <= 0) return hipErrorInvalidValue;
    const size_t lds = tile_lds_bytes(a, mode);
    switch (mode) {
    case kTileG2P: return launch_tiles_wh<kTileG2P, kWaves>(a, rbuf, wbuf, zbuf, record_mode, lds, s);
    case kTileP2G: return launch_tiles_wh<kTileP2G, kWaves>(a, rbuf, wbuf, zbuf, record_mode, lds, s);
    case kTileTail: return launch_tiles_wh<kTileTail, kWaves>(a, rbuf, wbuf, zbuf, record_mode, lds, s);
    case kTileChain:
        return a.few ? launch_tiles_wh<kTileChain, kWavesFew>(a, rbuf, wbuf, zbuf, record_mode, lds, s)
                     : launch_tiles_wh<kTileChain, kWaves>(a, rbuf, wbuf, zbuf, record_mode, lds, s);
    default: return hipErrorInvalidValue;
    }
}

template <int MODE, int WAVES>
static int resident_wh(const StepArgs &a, size_t lds)
{
    auto ask = [&](auto kernel) {
        int n = 0;
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, kBlock, lds) == hipSuccess ? n : 0;
    };
    switch (a.win_h) {
    case 12: return ask(k_tiles<MODE, 12, WAVES>);
    case 18: return ask(k_tiles<MODE, 18, WAVES>);
    case 20: return ask(k_tiles<MODE, 20, WAVES>);
    case 34: return ask(k_tiles<MODE, 34, WAVES>);
    case 36: return ask(k_tiles<MODE, 36, WAVES>);
    case 66: return ask(k_tiles<MODE, 66, WAVES>);
    case 68: return ask(k_tiles<MODE, 68, WAVES>);
    default: return ask(k_tiles<MODE, 0, WAVES>);
    }
}

int tiles_resident_per_cu(const StepArgs &a, int mode)
{
    const size_t lds = tile_lds_bytes(a, mode);
    switch (mode) {
    case kTileG2P: return resident_wh<kTileG2P, kWaves>(a, lds);
    case kTileP2G: return resident_wh<kTileP2G, kWaves>(a, lds);
    case kTileTail: return resident_wh<kTileTail, kWaves>(a, lds);
    case kTileChain:
        return a.few ? resident_wh<kTileChain, kWavesFew>(a, lds) : resident_wh<kTileChain, kWaves>(a, lds);
    default: return 0;
    }
}

}  // namespace fp64
}  // namespace icempm
