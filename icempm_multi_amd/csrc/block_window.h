// block_window.h -- node window of the points of one workgroup, found from the
// points themselves: the unbinned P2G sums its contributions there.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.h"
#include "point_fp64.h"

namespace icempm {

// Points of a workgroup whose stencils' box has at most this many nodes are
// summed in LDS (24 bytes per node: 30 KiB, five workgroups per CU).  256
// points in cell order with 4 per cell fill 64 cells of a column, whose box is
// 3 to 5 columns high as the column, or 3 by 66: up to 250 occupied rows fit.
// Points in no order do not fit, and add into global memory one by one, as
// all points did before (102k points in cell order: 97 -> 7.1 us).
constexpr int kBlockWindowNodes = 1280;

struct BlockWindow {
    int c0, r0, w, h;   // nodes [c0, c0 + w) x [r0, r0 + h)
    bool fits;
};

// The box of the 3x3 stencils with base nodes (col, row) of the threads that
// have a point; called by all threads of a workgroup of 256.
__device__ __forceinline__ BlockWindow block_window(bool have, int col, int row)
{
    __shared__ int box[4][4];
    int v[4] = {have ? col : 0x7fffffff, have ? row : 0x7fffffff, have ? -col : 0x7fffffff, have ? -row : 0x7fffffff};
#pragma unroll
    for (int k = 32; k > 0; k >>= 1) {
#pragma unroll
        for (int q = 0; q < 4; q++) v[q] = min(v[q], __shfl_xor(v[q], k));
    }
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int q = 0; q < 4; q++) box[threadIdx.x >> 6][q] = v[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = min(min(box[0][q], box[1][q]), min(box[2][q], box[3][q]));
    BlockWindow b;
    b.c0 = v[0];
    b.r0 = v[1];
    // no point at all: an empty window
    b.w = v[0] == 0x7fffffff ? 0 : -v[2] - v[0] + 3;
    b.h = v[0] == 0x7fffffff ? 0 : -v[3] - v[1] + 3;
    b.fits = (long long)b.w * b.h <= kBlockWindowNodes;
    return b;
}

// Lane l of a wave takes point (l % 16) * 4 + l / 16 of its 64: in cell order,
// with 4 points per cell, adjacent lanes then hold points of different cells
// and their LDS atomics different addresses.
__device__ __forceinline__ int spread_point(int tid)
{
    return (tid & ~63) + ((tid & 15) << 2) + ((tid & 63) >> 4);
}

// The P2G of a workgroup's points: every thread with a point has its stencil
// in st; add_nodes(sink) calls sink(i, j, dm, dpx, dpy) for its 9 nodes.
template <class AddNodes>
__device__ __forceinline__ void block_p2g(const StepArgs &a, const SceneDev &S, int gridY, int wbuf, bool have, int col,
                                          int row, AddNodes &&add_nodes)
{
    using fp64::glb_add;
    using fp64::glb_d;
    using fp64::lds_add;
    using fp64::lds_d;
    __shared__ __attribute__((aligned(16))) double sums_raw[3 * kBlockWindowNodes];
    lds_d *const sums = (lds_d *)sums_raw;
    glb_d *const gw = (glb_d *)(a.grid_mem + S.grid_off[wbuf]);
    const long long gp = S.gpitch;
    int *const flags = a.dirty + wbuf * a.dirty_stride + S.seg_off;
    const BlockWindow b = block_window(have, col, row);
    if (!b.fits) {   // the same for all threads
        if (have)
            add_nodes([&](int i, int j, double dm, double dpx, double dpy) {
                const long long gi = (long long)(col + i) * gridY + row + j;
                glb_add(gw + gi, dm);
                glb_add(gw + gp + gi, dpx);
                glb_add(gw + 2 * gp + gi, dpy);
                flags[gi >> kSegShift] = 1;
            });
        return;
    }
    const int n = b.w * b.h;
    for (int k = threadIdx.x; k < 3 * n; k += blockDim.x) sums[k] = 0;
    __syncthreads();
    if (have) {
        lds_d *const p0 = sums + 3 * ((col - b.c0) * b.h + row - b.r0);
        const int stride = 3 * b.h;
        add_nodes([&](int i, int j, double dm, double dpx, double dpy) {
            lds_d *const p = p0 + i * stride + 3 * j;
            lds_add(p, dm);
            lds_add(p + 1, dpx);
            lds_add(p + 2, dpy);
        });
    }
    __syncthreads();
    const float inv_h = 1.0f / (float)b.h;   // node / h is exact, as in TileWindow (node < 1280, h <= 1280)
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
        const double m = sums[3 * k];
        if (m == 0) continue;
        const int c = (int)(((float)k + 0.5f) * inv_h);
        const long long gi = (long long)(b.c0 + c) * gridY + b.r0 + k - c * b.h;
        glb_add(gw + gi, m);
        glb_add(gw + gp + gi, sums[3 * k + 1]);
        glb_add(gw + 2 * gp + gi, sums[3 * k + 2]);
        flags[gi >> kSegShift] = 1;
    }
}

}  // namespace icempm
