"""The split of the tile table among the workgroups of a tile launch, and the
tile shape a partition takes by itself, against the FP64 oracle.

One block of 6,400 points stepped with shapes that give fewer tiles than
workgroups, several tiles per workgroup (the table cut by weight into one range
per XCD, taken in turn), and the smallest shape of the built-in rule; and blocks
of sizes around the rule's changes of shape with no shape set.  Every field to
1e-9 of its scale after 12 substeps, as for the other tile shapes."""
import numpy as np
import pytest

import _oracle as O
import icempm_multi_amd as im
from icempm_multi_amd import scenes

pytestmark = pytest.mark.gpu

FIELDS = {"x": (4, 6), "v": (6, 8), "F": (8, 12), "C": (12, 16), "Jp": (3, 4)}


def step_and_compare(P, h, n, shape, substeps=12):
    r = np.random.default_rng(n)
    h[6, :n] = 0.3 * np.sin(3 * h[4, :n])
    h[7, :n] = -0.2 * np.cos(2 * h[5, :n])
    h[8:12, :n] += 1e-5 * r.normal(size=(4, n))
    part = im.Partition(0, 0, im.PRECISION_FP64)
    part.allocate(h.shape[1], P.GridXTotal)
    part.update_constants(P)
    if shape:
        part.set_tile_shape(*shape)
    part.transfer_points_from_soa_to_device(h, 0, n)
    print(f"{n} points, tile {shape}", flush=True)
    part.step(substeps, im.STEP_GRAPH | im.STEP_RESORT)
    config = part.tile_config()
    out = np.zeros_like(h)
    part.transfer_from_device(out, 0)
    assert part.error_code == 0
    part.close()
    ref = h.copy()
    O.sort(P, ref, n)
    O.substeps(P, ref, n, substeps, 0.0, 0)
    for name, (a, b) in FIELDS.items():
        scale = np.abs(ref[a:b, :n]).max()
        assert np.abs(out[a:b, :n] - ref[a:b, :n]).max() <= 1e-9 * scale, name
    assert np.array_equal(out[0, :n].view(np.int64), ref[0, :n].view(np.int64))
    return config


@pytest.mark.parametrize("shape", [(1, 1, 1), (1, 2, 0), (2, 3, 1), (4, 8, 1), (32, 16, 0)])
def test_tile_split_matches_oracle(shape):
    P, h, n = scenes.block_scene(nx=80, ny=20, grid=(128, 64), n_grains=40)
    c = step_and_compare(P, h, n, shape)
    assert (c["tx"], c["ty"], c["margin"]) == shape


# the second case's tiles lie in columns whose last tile is one cell wide
@pytest.mark.parametrize("nx,ny", [(16, 4), (61, 33), (200, 128), (150, 400)])
def test_shape_by_rule_matches_oracle(nx, ny):
    P, h, n = scenes.block_scene(nx=nx, ny=ny, grid=(nx + 40, ny + 24), n_grains=40)
    c = step_and_compare(P, h, n, None)
    # no more cells per tile than the largest shape, and small scenes get the smallest
    assert c["tx"] * c["ty"] <= 16 * 32
    if n <= 4096:
        assert (c["tx"], c["ty"]) == (4, 8)


# tiles of one to all of their points: 2, 4 and 8 tiles per workgroup (assigned
# by weight, the last at the edge of that) and 16 and more (taken in turn)
@pytest.mark.parametrize("shape", [(3, 5, 1), (3, 3, 0), (2, 2, 1), (1, 2, 1)])
@pytest.mark.parametrize("nx,ny", [(200, 128), (230, 160)])
def test_uneven_tiles_match_oracle(nx, ny, shape):
    P, h, n = scenes.block_scene(nx=nx, ny=ny, grid=(nx + 40, ny + 24), n_grains=40)
    r = np.random.default_rng(nx)
    thin = 0.5 + 0.5 * np.sin(h[4, :n] * (7.0 / h[4, :n].max())) * np.cos(h[5, :n] * (9.0 / h[5, :n].max()))
    keep = np.flatnonzero(r.random(n) < thin)
    h[:, :keep.size] = h[:, keep]
    c = step_and_compare(P, h, keep.size, shape)
    assert (c["tx"], c["ty"], c["margin"]) == shape


# 400 to 1600 tiles: on both sides of the counts from which on the launch uses
# the kernel built for more waves per SIMD, changed between graph replays
@pytest.mark.parametrize("shapes", [[(4, 8, 1), (1, 2, 1), (4, 8, 1)], [(1, 3, 0), (2, 2, 1), (1, 4, 1), (1, 3, 0)]])
def test_few_and_many_tiles_in_turn_match_oracle(shapes):
    P, h, n = scenes.block_scene(nx=80, ny=20, grid=(128, 64), n_grains=40)
    h[6, :n] = 0.3 * np.sin(3 * h[4, :n])
    h[7, :n] = -0.2 * np.cos(2 * h[5, :n])
    part = im.Partition(0, 0, im.PRECISION_FP64)
    part.allocate(h.shape[1], P.GridXTotal)
    part.update_constants(P)
    part.transfer_points_from_soa_to_device(h, 0, n)
    ref = h.copy()
    t, step = 0.0, 0
    for shape in shapes:
        print(f"{n} points, tile {shape}", flush=True)
        part.set_tile_shape(*shape)
        part.step(20, im.STEP_GRAPH | im.STEP_RESORT)
        O.sort(P, ref, n)
        t, step, _, err = O.substeps(P, ref, n, 20, t, step)
        assert err == 0
    out = np.zeros_like(h)
    part.transfer_from_device(out, 0)
    assert part.error_code == 0
    part.close()
    for name, (a, b) in FIELDS.items():
        scale = np.abs(ref[a:b, :n]).max()
        assert np.abs(out[a:b, :n] - ref[a:b, :n]).max() <= 1e-9 * scale, name
    assert np.array_equal(out[0, :n].view(np.int64), ref[0, :n].view(np.int64))


# a table of 1.1M tiles, of which the builder's workgroups take 524,288 at once;
# the points' columns lie around the end of the first of these sweeps
def test_table_beyond_one_sweep_of_the_builder_matches_oracle():
    P, h, n = scenes.block_scene(nx=80, ny=20, grid=(1100, 1000), n_grains=40)
    c = step_and_compare(P, h, n, (1, 1, 1))
    first, last = (int(t(h[4, :n]) / P.cellsize) + P.GridHaloSize for t in (np.min, np.max))
    assert first * P.GridY < 524288 < last * P.GridY and (c["tx"], c["ty"]) == (1, 1)


# 102k points: the built-in rule takes 4x14 cells, which are no candidate of the
# autotuner and 14% faster than the best of them
def test_autotuner_keeps_a_faster_shape_in_force():
    P, h, n = scenes.block_scene(nx=320, ny=80, grid=(384, 112), h=0.1, n_grains=20)
    out = []
    for tune in (True, False):
        part = im.Partition(0, 0, im.PRECISION_FP64)
        part.allocate(h.shape[1], P.GridXTotal)
        part.update_constants(P)
        part.transfer_points_from_soa_to_device(h, 0, n)
        part.sort_points()
        before = part.tile_config()
        if tune:
            chosen, ms = part.autotune(20)
            assert chosen == len(ms) == 2 * len(im.capi.tile_candidates())
        assert part.tile_config() == before and (before["tx"], before["ty"]) == (4, 14)
        part.step(20, im.STEP_GRAPH | im.STEP_RESORT)
        out.append(np.zeros_like(h))
        part.transfer_from_device(out[-1], 0)
        assert part.error_code == 0
        part.close()
    for name, (a, b) in FIELDS.items():
        scale = np.abs(out[1][a:b, :n]).max()
        assert np.abs(out[0][a:b, :n] - out[1][a:b, :n]).max() <= 1e-9 * scale, name


# Pairs of points 0.6 cells apart, far from each other, fly a cell and a half: with
# tiles of one cell each pair fills one tile, then two, then one again, on both sides
# of the count from which on the launch uses the kernel built for more waves per SIMD
# (512 tiles in FP64, 768 in the mixed form).  The shape stays, so the captured graphs
# do: the frames with two tiles per pair capture graphs of their own, and those of the
# first kind serve again.
@pytest.mark.parametrize("precision,side", [(im.PRECISION_FP64, 20), (im.PRECISION_MIXED, 25)])
def test_few_and_many_tiles_by_motion_match_oracle(precision, side):
    gap, frames, substeps = 8, 49, 20
    grid = side * gap + 40
    P, _, _ = scenes.block_scene(nx=20, ny=8, grid=(grid, grid), n_grains=5)
    P.IndRSq = 0.0
    i, j = (a.ravel() for a in np.meshgrid(np.arange(side), np.arange(side)))
    x = np.concatenate([20 + gap * i + 0.52, 20 + gap * i + 1.12])      # 0.02 and 0.62 into cell 21 + 8 i
    n = x.size
    h = np.zeros((16, n))
    h[3], h[8], h[11] = 1, 1, 1
    h[4] = x * P.cellsize
    h[5] = np.tile(20 + gap * j + 0.1, 2) * P.cellsize
    h[6] = P.cellsize / (35 * substeps * P.InitialTimeStep)             # a cell in 35 frames
    part = im.Partition(0, 0, precision)
    part.allocate(n, P.GridXTotal)
    part.update_constants(P)
    part.set_tile_shape(1, 1, 1)
    part.transfer_points_from_soa_to_device(h, 0, n)
    ref = h.copy()
    t, step, captures = 0.0, 0, []
    print(precision, n, flush=True)
    for k in range(frames):
        part.step(substeps, im.STEP_GRAPH | im.STEP_RESORT)
        captures.append(part.graph_stats()[0])
        O.sort(P, ref, n)
        t, step, _, err = O.substeps(P, ref, n, substeps, t, step)
        assert err == 0
    out = np.zeros_like(h)
    part.transfer_from_device(out, 0)
    assert part.error_code == 0
    part.close()
    # frames 0 to 13 and 35 to 48: one tile per pair; 14 to 34: two
    assert captures[13] == captures[6] and captures[34] == 2 * captures[13] and captures[48] == captures[34]
    tol = dict(x=1e-9, v=1e-9, F=1e-9, C=1e-9, Jp=1e-9) if precision == im.PRECISION_FP64 else dict(x=1e-6, v=1e-4)
    for name, rtol in tol.items():
        a, b = FIELDS[name]
        scale = max(np.abs(ref[a:b]).max(), 1e-3 if name == "C" else 0)
        assert np.abs(out[a:b] - ref[a:b]).max() <= rtol * scale, name
    assert np.array_equal(out[0].view(np.int64), ref[0].view(np.int64))


# The tiles behind the built-in shape are counted by the cells on the first grid and by
# the points on the second, which has the same cells in its first columns and rows and
# more than 10 cells per point: the same counts, the same shape.
@pytest.mark.parametrize("precision", [im.PRECISION_FP64, im.PRECISION_MIXED])
@pytest.mark.parametrize("nx,ny,thin", [(16, 4, False), (61, 33, True), (320, 80, False), (375, 167, False),
                                        (300, 260, True), (633, 158, False), (633, 158, True)])
def test_shape_by_cells_and_by_points(nx, ny, thin, precision):
    P, h, n = scenes.block_scene(nx=nx, ny=ny, grid=(nx + 32, ny + 20), n_grains=40)
    r = np.random.default_rng(nx)
    if thin:
        keep = np.flatnonzero(r.random(n) < 0.5 + 0.5 * np.sin(0.9 * h[4, :n]) * np.cos(0.7 * h[5, :n]))
        n = keep.size
        h[:, :n] = h[:, keep]
    h[0, :n].view(np.int64)[r.random(n) < 0.05] |= 0x20000              # disabled: dropped by the sort
    side = int(np.sqrt(12.0 * h.shape[1])) + nx + ny
    Q, _, _ = scenes.block_scene(nx=16, ny=4, grid=(side, side), n_grains=4)
    assert Q.cellsize == P.cellsize
    got = []
    for prms in (P, Q):
        part = im.Partition(0, 0, precision)
        part.allocate(h.shape[1], prms.GridXTotal)
        part.update_constants(prms)
        part.transfer_points_from_soa_to_device(h, 0, n)
        part.sort_points()
        got.append((part.tile_config(), part.nPts_partition))
        part.close()
    assert got[0] == got[1] and got[0][1] < n
