// kernels_fp64_direct.hip -- unbinned FP64 kernels: one thread per point, in
// whatever order the points are (gpu_partition.cu:230-293).  Used before the
// first sort, on request, and by icempm_substeps_noalloc, whose caller keeps
// the points' order.
// Kept in its own translation unit: compiled together with the binned kernels
// it trips an inliner crash of the ROCm 7.2 device compiler.
#include <hip/hip_runtime.h>

#include "block_window.h"
#include "point_fp64.h"
#include "tile_common.h"

namespace icempm {
namespace fp64 {

// P2G: the contributions of a workgroup's 256 points are summed in the LDS
// window their stencils span, and each touched node gets one global atomic per
// line, instead of 27 per point, where the points lie in or near cell order
// (block_p2g).
__global__ void __launch_bounds__(kBlock) k_p2g_direct(StepArgs a, int scene, int wbuf)
{
    const SceneDev &S = a.scenes[scene];
    const SceneConsts c = uniform_copy(S.c);
    const int i = blockIdx.x * kBlock + spread_point(threadIdx.x);
    const long long pt = S.pt_off + i;
    const PtRef R{(double *)a.pts, a.pitch};
    long long ud = kDisabled;
    if (i < S.n_pts) ud = as_ll(R.at(kLineUtility, pt));
    bool have = !(ud & kDisabled);
    P2GStencil st;
    if (have) {
        double x, y, F[4], Jp, v[2], B[4];
        load_state(R, pt, x, y, F, Jp);
        v[0] = R.at(kLineVelX, pt);
        v[1] = R.at(kLineVelX + 1, pt);
#pragma unroll
        for (int m = 0; m < 4; m++) B[m] = R.at(kLineBp00 + m, pt);
        StressTerms none;
        none.valid = false;
        const unsigned e = p2g_stencil(c, x, y, v, B, F, Jp, ud, none, st);
        if (e) {
            atomicMax(&a.err[scene], e);
            have = false;
        }
    }
    block_p2g(a, S, c.gridY, wbuf, have, st.bxc, st.by, [&](auto &&sink) { st.nodes(c, sink); });
}

// One launch per substep (as k_tiles<kTileChain / kTileTail> for binned points):
// the grid update folded into the staging of the workgroup's velocity window,
// G2P, and (NEXT) P2G of the next substep into grid[wbuf]; the side work
// clears grid[zbuf], adds the indenter force and advances the clock.  The
// window is the box of the workgroup's 256 stencils and one node around it, so
// a point whose stencil moved by a cell still adds in LDS; workgroups whose
// points span too many nodes work on global memory, point by point.
// Measured on 102k points in cell order: one launch of 14.8 us per substep. The
// separate launches took 120 us, 97 of them in P2G's global atomics, and take
// 27 with the P2G above (fills 3, P2G 7.1, grid update 4.4, G2P 6.8, gaps 6).
constexpr int kChainNodes = 1280;   // 40 B per node, 50 KiB: three workgroups per CU, as its registers allow

template <bool NEXT>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(3)))
k_points(StepArgs a, int scene, int rbuf, int wbuf, int zbuf)
{
    __shared__ __attribute__((aligned(16))) double lds_raw[(NEXT ? 5 : 2) * kChainNodes];
    lds_d *const vw = (lds_d *)lds_raw;
    lds_d *const acc = vw + 2 * kChainNodes;
    int block = blockIdx.x;
    if (side_work(a, rbuf, zbuf, block)) return;
    const SceneDev &S = a.scenes[scene];
    const SceneConsts c = uniform_copy(S.c);
    const SceneClock clk = next_clock(c, uniform_copy(a.clocks[scene]));
    const bool record = (clk.step % c.update_every) == 0;
    const glb_d *const gr = (const glb_d *)(a.grid_mem + S.grid_off[rbuf]);
    glb_d *const gw = (glb_d *)(a.grid_mem + S.grid_off[wbuf]);
    int *const flags = a.dirty + wbuf * a.dirty_stride + S.seg_off;
    const long long gp = S.gpitch;
    const int gridY = c.gridY, tid = threadIdx.x;
    const int i = block * kBlock + spread_point(tid);
    const long long pt = S.pt_off + i;
    const PtRef R{(double *)a.pts, a.pitch};
    long long ud = kDisabled;
    double x = 0, y = 0, F[4] = {1, 0, 0, 1}, Jp = 1;
    if (i < S.n_pts) {
        ud = as_ll(R.at(kLineUtility, pt));
        load_state(R, pt, x, y, F, Jp);
    }
    bool have = !(ud & kDisabled);
    int bx, by;
    double f;
    base_fx(c, x, bx, f);
    base_fx(c, y, by, f);
    const int bxc = bx - c.xoff + c.halo;
    unsigned e = stencil_error(c, bxc, by);
    if (have && e) {
        atomicMax(&a.err[scene], e);
        have = false;
    }
    const BlockWindow b = block_window(have, bxc, by);
    const int wc0 = b.c0 - 1, wr0 = b.r0 - 1, win_h = b.h + 2;
    const bool fits = b.w > 0 && (long long)(b.w + 2) * win_h <= kChainNodes;   // the same for all threads
    const int win_w = fits ? b.w + 2 : 0, n = win_w * win_h;
    const float inv_h = 1.0f / (float)win_h;   // node / win_h is exact (see block_p2g)
    for (int k = tid; k < n; k += kBlock) {
        const int qc = (int)(((float)k + 0.5f) * inv_h), col = wc0 + qc, row = wr0 + k - qc * win_h;
        double vx = 0, vy = 0;
        if (col >= 0 && col < c.ncols && row >= 0 && row < gridY) {
            const long long gi = (long long)col * gridY + row;
            const double m = gr[gi], px = gr[gp + gi], py = gr[2 * gp + gi];
            if (m != 0) node_velocity(c, clk, nullptr, col - c.halo + c.xoff, row, m, px, py, vx, vy);
        }
        vw[2 * k] = vx;
        vw[2 * k + 1] = vy;
        if (NEXT) acc[3 * k] = acc[3 * k + 1] = acc[3 * k + 2] = 0;
    }
    __syncthreads();
    if (have) {
        double v[2], B[4], pp, qq;
        StressTerms terms;
        g2p_point(c, (const glb_d *)S.fail_tab, gr, gp, &clk, vw, wc0, wr0, win_w, win_h, win_h, false, x, y, v, B, F,
                  Jp, ud, pp, qq, e, terms);
        if (NEXT) store_state_fused(R, pt, x, y, F, Jp, ud, record, pp, qq);
        else store_state(R, pt, x, y, v, F, B, Jp, ud, record, pp, qq);
        if (NEXT) {
            P2GStencil st;
            e = p2g_stencil(c, x, y, v, B, F, Jp, ud, terms, st);
            const int lx = st.bxc - wc0, ly = st.by - wr0;
            if (e) {
                atomicMax(&a.err[scene], e);
            } else if (lx >= 0 && lx + 2 < win_w && ly >= 0 && ly + 2 < win_h) {
                lds_d *const p0 = acc + 3 * (lx * win_h + ly);
                const int stride = 3 * win_h;
                st.nodes(c, [&](int ni, int nj, double dm, double dpx, double dpy) {
                    lds_d *const p = p0 + ni * stride + 3 * nj;
                    lds_add(p, dm);
                    lds_add(p + 1, dpx);
                    lds_add(p + 2, dpy);
                });
            } else {
                st.nodes(c, [&](int ni, int nj, double dm, double dpx, double dpy) {
                    const long long gi = (long long)(st.bxc + ni) * gridY + st.by + nj;
                    glb_add(gw + gi, dm);
                    glb_add(gw + gp + gi, dpx);
                    glb_add(gw + 2 * gp + gi, dpy);
                    flags[gi >> kSegShift] = 1;
                });
            }
        }
    }
    if (!NEXT) return;
    __syncthreads();
    for (int k = tid; k < n; k += kBlock) {
        const double m = acc[3 * k];
        if (m == 0) continue;
        const int qc = (int)(((float)k + 0.5f) * inv_h), col = wc0 + qc, row = wr0 + k - qc * win_h;
        const long long gi = (long long)col * gridY + row;   // inside the grid: a stencil lies there
        glb_add(gw + gi, m);
        glb_add(gw + gp + gi, acc[3 * k + 1]);
        glb_add(gw + 2 * gp + gi, acc[3 * k + 2]);
        flags[gi >> kSegShift] = 1;
    }
}

hipError_t launch_points(const StepArgs &a, int scene, bool next, int rbuf, int wbuf, int zbuf, hipStream_t s)
{
    const unsigned grid = tile_grid(a, kTileChain);
    if (next) hipLaunchKernelGGL(k_points<true>, dim3(grid), dim3(kBlock), 0, s, a, scene, rbuf, wbuf, zbuf);
    else hipLaunchKernelGGL(k_points<false>, dim3(grid), dim3(kBlock), 0, s, a, scene, rbuf, wbuf, zbuf);
    return hipGetLastError();
}

__global__ void __launch_bounds__(kBlock) k_g2p_direct(StepArgs a, int scene, int rbuf, int record)
{
    const SceneDev &S = a.scenes[scene];
    const SceneConsts c = uniform_copy(S.c);
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= S.n_pts) return;
    const long long pt = S.pt_off + i;
    const PtRef R{(double *)a.pts, a.pitch};
    long long ud = as_ll(R.at(kLineUtility, pt));
    if (ud & kDisabled) return;
    double x, y, F[4], Jp, v[2], B[4], pp, qq;
    load_state(R, pt, x, y, F, Jp);
    unsigned e;
    StressTerms terms;
    if (!g2p_point(c, (const glb_d *)S.fail_tab, (const glb_d *)(a.grid_mem + S.grid_off[rbuf]), S.gpitch, nullptr,
                   nullptr, 0, 0, 0, 0, 0, false, x, y, v, B, F, Jp, ud, pp, qq, e, terms)) {
        atomicMax(&a.err[scene], e);
        return;
    }
    const bool rec = record >= 0 ? record != 0 : (a.clocks[scene].step % c.update_every) == 0;
    store_state(R, pt, x, y, v, F, B, Jp, ud, rec, pp, qq);
}

hipError_t launch_p2g_direct(const StepArgs &a, int scene, int n_pts, int wbuf, hipStream_t s)
{
    if (n_pts <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_p2g_direct, dim3((n_pts + kBlock - 1) / kBlock), dim3(kBlock), 0, s, a, scene, wbuf);
    return hipGetLastError();
}

hipError_t launch_g2p_direct(const StepArgs &a, int scene, int n_pts, int rbuf, int record_pq, hipStream_t s)
{
    if (n_pts <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_g2p_direct, dim3((n_pts + kBlock - 1) / kBlock), dim3(kBlock), 0, s, a, scene, rbuf,
                       record_pq);
    return hipGetLastError();
}

}  // namespace fp64
}  // namespace icempm
