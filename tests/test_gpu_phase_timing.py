"""The times of the phase calls, which their launches leave themselves (binned) or
events take: each phase's launches are counted, their times add up
to no more than the host's, and time in which the host does nothing between two
calls belongs to neither."""
import time

import numpy as np
import pytest

import icempm_multi_amd as im
from icempm_multi_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [im.PRECISION_FP64, im.PRECISION_MIXED])
@pytest.mark.parametrize("binned", [True, False])
@pytest.mark.parametrize("pause", [None, 0, 1, 2, 3])
def test_phase_times(precision, binned, pause):
    P, h, n = scenes.block_scene(nx=120, ny=80, grid=(200, 128), n_grains=20)
    part = im.Partition(0, 0, precision)
    part.allocate(h.shape[1], P.GridXTotal)
    part.update_constants(P)
    part.transfer_points_from_soa_to_device(h, 0, n)
    if binned:
        part.sort_points()
    calls = (part.reset_grid, part.p2g, lambda: part.update_nodes(P.SimulationTime, P.indenter_x, P.indenter_y),
             lambda: part.g2p(False))
    for f in calls:
        f()
    part.reset_indenter_force_accumulator()   # and the times
    print(precision, binned, pause, flush=True)
    rounds = 40
    t0 = time.perf_counter()
    for i in range(rounds):
        for k, f in enumerate(calls):
            f()
            if pause == k and i < 4:
                time.sleep(0.05)
    st = part.kernel_stats()
    wall = (time.perf_counter() - t0) * 1e3
    ms = {k: v[0] for k, v in st.items()}
    for k in ("zero", "p2g", "update", "g2p"):
        assert st[k][1] == rounds and ms[k] > 0, (k, st[k])
    total = sum(ms[k] for k in ("zero", "p2g", "update", "g2p"))
    assert total <= wall
    if pause is not None:
        assert total <= wall - 4 * 50 + 20    # the pauses, less 5 ms of scheduling each
    assert part.error_code == 0
    part.close()


def test_phase_time_lasts_to_the_last_wave():
    """A launch's time ends with its last wave, not with the first of each workgroup: a
    grid update whose workgroups have one wave without nodes (it takes every fourth grid
    column, a run of 64 segments) takes as long whichever wave that is."""
    P, _, _ = scenes.block_scene(nx=20, ny=8, grid=(2100, 4096), n_grains=5)
    ms = []
    for first in (2, 3):        # columns of points, which touch the one before and the one after
        x, y = np.meshgrid((np.arange(100, 500) * 4 + first) * P.cellsize, (np.arange(2, 126) * 32) * P.cellsize)
        n = x.size
        h = np.zeros((16, n))
        h[3], h[4], h[5], h[8], h[11] = 1, x.ravel(), y.ravel(), 1, 1
        part = im.Partition(0, 0, im.PRECISION_FP64)
        part.allocate(n, P.GridXTotal)
        part.update_constants(P)
        part.transfer_points_from_soa_to_device(h, 0, n)
        for i in range(13):
            if i == 3:
                part.reset_indenter_force_accumulator()   # and the times
            part.reset_grid()
            part.p2g()
            part.update_nodes(0.0, P.indenter_x, P.indenter_y)
        st = part.kernel_stats()
        assert st["update"][1] == 10 and part.error_code == 0
        ms.append(st["update"][0] / 10)
        part.close()
    print(ms, flush=True)
    assert ms[0] >= 0.75 * ms[1]
