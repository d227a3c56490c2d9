// tile_common.h -- parts of the binned tile kernels that both precision forms
// share: scalar copies of launch-invariant data, the clearing of the grid
// buffer two substeps back, the indenter force, and the runs of a tile's points.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

#include "kernels.h"
#include "point_fp64.h"

namespace icempm {

// Loads of workgroup-uniform data that no launch reading it writes (scene
// table, tile table, run table, the current clock slot) through the scalar
// cache into scalar registers.
template <class T>
__device__ __forceinline__ T scalar_load(const T *src)
{
    static_assert(sizeof(T) % 4 == 0, "scalar_load works on whole dwords");
    typedef const __attribute__((address_space(4))) unsigned cst_u;
    T out;
    cst_u *s = (cst_u *)reinterpret_cast<const unsigned *>(src);
    unsigned *d = reinterpret_cast<unsigned *>(&out);
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) / 4); i++) d[i] = s[i];
    return out;
}

// Moves loaded data into registers of its own, opaque to the compiler.  It
// would otherwise load the data again inside the point loop, where a scalar
// load waits for every LDS atomic in flight; and data left in the 8 or 16
// consecutive registers a wide load writes is spilled and restored as such a
// block (581 v_readlane in the FP64 point loop instead of 89).
// (The data is waited for here: issue all loads of a stage first.)
template <class T>
__device__ __forceinline__ void pin(T &t)
{
    unsigned *d = reinterpret_cast<unsigned *>(&t);
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) / 4); i++) {
        unsigned v;
        asm("s_mov_b32 %0, %1" : "=s"(v) : "s"(d[i]));
        d[i] = v;
    }
}

template <class T>
__device__ __forceinline__ T scalar_copy(const T *src)
{
    T out = scalar_load(src);
    pin(out);
    return out;
}

// The leading part of a scene's table entry (constants, grid place), held by a
// wave as one dword per lane and register: three loads, all in flight
// together.  Through the scalar cache the same 550 bytes took 1 us of a
// launch, its misses being served one after the other.  copy() moves fields
// to scalar registers of their own (the unused ones cost nothing).
struct SceneLanes {
    static constexpr int kRegs = 3;
    static_assert(offsetof(SceneDev, fail_tab) <= kRegs * 256 && sizeof(SceneDev) >= kRegs * 256,
                  "three registers hold the entry up to its table");
    unsigned v[kRegs];

    __device__ __forceinline__ void load(const SceneDev *S)
    {
        typedef const __attribute__((address_space(1))) unsigned glb_u;
        glb_u *p = (glb_u *)reinterpret_cast<const unsigned *>(S) + (threadIdx.x & 63);
#pragma unroll
        for (int r = 0; r < kRegs; r++) v[r] = p[64 * r];
    }
    __device__ __forceinline__ unsigned dword(int i) const { return __builtin_amdgcn_readlane(v[i >> 6], i & 63); }
    template <class T>
    __device__ __forceinline__ T copy(size_t offset) const
    {
        static_assert(sizeof(T) % 4 == 0, "whole dwords");
        T out;
        unsigned *d = reinterpret_cast<unsigned *>(&out);
#pragma unroll
        for (int i = 0; i < (int)(sizeof(T) / 4); i++) d[i] = dword((int)(offset / 4) + i);
        return out;
    }
};

// Clears the flagged node segments of grid buffer zb of every scene, and
// their flags.  zb is the buffer two substeps back: no launch reads it any
// more, and the next launch accumulates into it.  Wave `wave` of n_waves takes
// runs wave, wave + n_waves, ... of the run table (a run: up to 64 segments of
// 64 nodes; one flag per lane, a ballot picks the flagged ones).
__device__ __forceinline__ void clear_flagged(const StepArgs &a, int zb, int wave, int n_waves)
{
    const int lane = threadIdx.x & 63;
    for (int r = wave; r < a.n_chunks; r += n_waves) {
        const NodeChunk run = scalar_load(a.chunks + r);
        int *fl = a.dirty + zb * a.dirty_stride + run.flag0;
        const int f = lane < run.nseg ? fl[lane] : 0;
        unsigned long long mb = __ballot(f != 0);
        fp64::glb_d *g = (fp64::glb_d *)(a.grid_mem + zb * a.grid_buf_bytes + run.grid_off);
        const long long gp = run.gpitch, node0 = (long long)run.seg0 << kSegShift;
        while (mb) {
            const int sg = __builtin_ctzll(mb);
            mb &= mb - 1;
            const long long idx = node0 + ((long long)sg << kSegShift) + lane;
            g[idx] = 0;
            g[gp + idx] = 0;
            g[2 * gp + idx] = 0;
        }
        if (f) fl[lane] = 0;
    }
}

// The indenter's reaction of the substep (kernels.cuh:265-287): every node
// of scene sc inside the indenter circle that holds mass in grid rb adds its
// force to the scene's bins.  The tiles form the same node velocities again
// where they stage them (node_velocity without the force).  One workgroup
// visits the bounding box of the circle, clipped to the grid.
__device__ __forceinline__ void indenter_force_nodes(const StepArgs &a, int sc, int rb)
{
    const SceneDev &S = a.scenes[sc];
    const SceneConsts c = scalar_copy(&a.scenes[sc].c);
    if (!(c.ind_rsq > 0)) return;
    const SceneClock clk = next_clock(c, scalar_copy(a.clocks + sc));
    const double r = sqrt(c.ind_rsq);
    const int gx0 = max((int)floor((clk.ind_x - r) * c.hinv) - 1, c.xoff - c.halo);
    const int gx1 = min((int)ceil((clk.ind_x + r) * c.hinv) + 1, c.xoff - c.halo + c.ncols - 1);
    const int gy0 = max((int)floor((clk.ind_y - r) * c.hinv) - 1, 0);
    const int gy1 = min((int)ceil((clk.ind_y + r) * c.hinv) + 1, c.gridY - 1);
    if (gx1 < gx0 || gy1 < gy0) return;
    const int ny = gy1 - gy0 + 1;
    const long long nn = (long long)(gx1 - gx0 + 1) * ny;
    const fp64::glb_d *g = (const fp64::glb_d *)(a.grid_mem + S.grid_off[rb]);
    const long long gp = S.gpitch;
    double *force = a.force_mem + S.force_off;
    for (long long k = threadIdx.x; k < nn; k += blockDim.x) {
        const int gix = gx0 + (int)(k / ny), giy = gy0 + (int)(k % ny);
        const long long idx = (long long)(gix - c.xoff + c.halo) * c.gridY + giy;
        const double m = g[idx], px = g[gp + idx], py = g[2 * gp + idx];
        if (m == 0) continue;
        double vx, vy;
        fp64::node_velocity(c, clk, force, gix, giy, m, px, py, vx, vy);
    }
}

// The work of a kTileFromMomenta launch beside its tiles, in workgroups of its
// own: the indenter force (before the tile workgroups in the grid: it takes as
// long as a small tile) and the clearing (after them, so that it fills CUs as
// the tile workgroups of a full GPU end); the first clearing workgroup also
// writes the advanced clocks to the other slot, which nobody reads here.  In
// the tile workgroups this work lengthened every one of them: a 24 us substep
// of 69.6k points with an indenter by 6 us.
// Returns true for such a workgroup; else `block` is its place among the
// n_work tile workgroups.
__device__ __forceinline__ bool side_work(const StepArgs &a, int rb, int zb, int &block)
{
    block = blockIdx.x - a.n_service;
    if (block < 0) {
        // (A count, not a last entry that ends the list: the kernels of the mixed
        // form took 0.6% longer with that, by the registers around it.)
        const int n = a.scenes[0].n_ind;
        for (int k = blockIdx.x; k < n; k += a.n_service) indenter_force_nodes(a, a.scenes[k].ind_scene, rb);
        return true;
    }
    if (block < a.n_work) return false;
    const int k = block - a.n_work, per = blockDim.x / 64;
    clear_flagged(a, zb, k * per + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6),
                  (gridDim.x - a.n_service - a.n_work) * per);
    if (k == 0)
        for (int sc = threadIdx.x; sc < a.nscenes; sc += blockDim.x)
            a.clocks_next[sc] = next_clock(a.scenes[sc].c, a.clocks[sc]);
    return true;
}

// Workgroups of a tile launch.
inline unsigned tile_grid(const StepArgs &a, int mode)
{
    return (mode & kTileFromMomenta) ? a.n_service + a.n_work + a.n_clear : a.n_work;
}

// Point k of a tile's points is SoA point k + off of the run that holds it:
// the run of column c of the tile's box ends before point `end`.  The table
// has kMaxTX entries, those past the box's columns with the largest end.
typedef __attribute__((address_space(3))) TileRun lds_run;
constexpr int kRunEnd = 0x7fffffff;

struct RunCursor {
    int c;
    // The run of the tile's point k, from any place: the ends are compared
    // eight at a time, so that their reads are in flight together (walking
    // the runs one by one took up to 1 us of a small scene's launch).
    __device__ __forceinline__ int seek(const lds_run *runs, int ncol, int k)
    {
        c = 0;
        for (int b = 0; b < ncol; b += 8) {
#pragma unroll
            for (int j = 0; j < 8; j++) c += k >= runs[b + j].end;
        }
        return k + runs[c].off;
    }
    // The same by walking on from the last point's run: k must not decrease.
    __device__ __forceinline__ int point(const lds_run *runs, int k)
    {
        int off = runs[c].off, end = runs[c].end;
        while (k >= end) {
            c++;
            off = runs[c].off;
            end = runs[c].end;
        }
        return k + off;
    }
};

}  // namespace icempm
