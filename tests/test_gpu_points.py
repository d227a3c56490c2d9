"""The unbinned kernels in workgroup windows: points in cell order (the window
fits the LDS), in random order (it does not: global memory, point by point),
columns so high that it just fits or does not, counts around a workgroup, and
grids too large for three buffers in the allocation-free call's array.

icempm_substeps_noalloc and the partition's unbinned steps, against the FP64
oracle on the same order of points: every field to 1e-9 of its scale after 8
substeps, as for the binned kernels; the mixed form's positions to 1e-6 and
velocities to 1e-4, as in its other tests."""
import numpy as np
import pytest

import _oracle as O
import icempm_multi_amd as im
from icempm_multi_amd import scenes
from test_zz_no_alloc import noalloc, with_motion

pytestmark = pytest.mark.gpu

FIELDS = {"x": (4, 6), "v": (6, 8), "F": (8, 12), "C": (12, 16), "Jp": (3, 4), "PQ": (1, 3)}
NSUB = 8


def shuffled(h, n, seed):
    order = np.random.default_rng(seed).permutation(n)
    h[:, :n] = h[:, order]


def scene(nx, ny, grid, order, indenter):
    if indenter:
        P, h, n = scenes.sheet_scene(nx=nx, ny=ny, grid=grid, h=0.05, ind_diameter=0.5, ind_depth=0.15, n_grains=30,
                                     sampler="jittered")
        P.indenter_x = P.indenter_x_initial = 0.5 * grid[0] * 0.05      # on the ice
    else:
        P, h, n = scenes.block_scene(nx=nx, ny=ny, grid=grid, n_grains=30)
    P, h, n = with_motion(P, h, n, nx)
    if order == "random":
        shuffled(h, n, ny)
    elif order == "mixed":       # the second half in random order
        half = h[:, n // 2:n].copy()
        h[:, n // 2:n] = half[:, np.random.default_rng(ny).permutation(half.shape[1])]
    return P, h, n


def compare(out, P, h, n, force=None):
    ref = h.copy()
    _, _, fref, err = O.substeps(P, ref, n, NSUB, P.SimulationTime, P.SimulationStep)
    assert err == 0
    for name, (a, b) in FIELDS.items():
        scale = np.abs(ref[a:b, :n]).max() + 1e-300
        assert np.abs(out[a:b, :n] - ref[a:b, :n]).max() <= 1e-9 * scale, name
    assert np.array_equal(out[0, :n].view(np.int64), ref[0, :n].view(np.int64))
    if force is not None:
        assert np.allclose(force.reshape(-1, 2).sum(0), fref.reshape(-1, 2).sum(0), rtol=1e-8, atol=1e-6)


# 64 cells of a column per workgroup: 255 occupied rows give windows of 5 x 257
# nodes (more than 1280 with the margin), 200 rows 5 x 204 (they fit)
CASES = [(30, 8, (64, 32), "cells", False), (30, 8, (64, 32), "random", False), (30, 8, (64, 32), "mixed", False),
         (12, 200, (40, 224), "cells", False), (12, 255, (40, 280), "cells", False), (4, 1, (32, 16), "cells", False),
         (65, 1, (96, 16), "cells", False), (100, 16, (160, 48), "cells", True), (100, 16, (160, 48), "random", True),
         (40, 10, (1000, 420), "cells", False)]


@pytest.mark.parametrize("nx,ny,grid,order,indenter", CASES)
def test_noalloc_matches_oracle(nx, ny, grid, order, indenter):
    P, h, n = scene(nx, ny, grid, order, indenter)
    out, err, force = noalloc(P, h, n, NSUB)
    assert err == 0
    compare(out, P, h, n, force)


@pytest.mark.parametrize("precision", [im.PRECISION_FP64, im.PRECISION_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("nx,ny,grid,order,indenter", CASES[:5])
def test_unbinned_steps_match_oracle(nx, ny, grid, order, indenter, precision):
    P, h, n = scene(nx, ny, grid, order, indenter)
    part = im.Partition(0, 0, precision)
    part.allocate(h.shape[1], P.GridXTotal)
    part.update_constants(P)
    part.transfer_points_from_soa_to_device(h, 0, n)
    print(f"{n} points, {order}, precision {precision}", flush=True)
    part.step(NSUB, im.STEP_DIRECT_P2G)
    out = np.zeros_like(h)
    part.transfer_from_device(out, 0)
    assert part.error_code == 0
    part.close()
    if precision == im.PRECISION_FP64:
        compare(out, P, h, n)
        return
    ref = h.copy()
    O.substeps(P, ref, n, NSUB, 0.0, 0)
    for (a, b), tol in (((4, 6), 1e-6), ((6, 8), 1e-4)):
        assert np.linalg.norm(out[a:b, :n] - ref[a:b, :n]) <= tol * np.linalg.norm(ref[a:b, :n])
