"""Up- and download of point lines through the pinned staging, at sizes around
its chunks (4,096 to 32,768 points, three in flight; from 131,072 points on
other host threads help), odd counts, and offsets and capacities that leave the
caller's lines unaligned.

FP64 comes back bit for bit, NaN and infinities included, and the lines outside
the points stay untouched.  The mixed form comes back as its conversions give
it, each operation rounded on its own: the same values from numpy, bit for bit."""
import numpy as np
import pytest

import icempm_multi_amd as im
from icempm_multi_amd import scenes

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 255, 4095, 4096, 4097, 16385, 3 * 32768 + 1, 131073]


def state(n, capacity, offset, seed):
    r = np.random.default_rng(seed)
    h = r.normal(size=(16, capacity))
    h[4] = r.uniform(0.0, 60.0, capacity)
    h[5] = r.uniform(0.0, 30.0, capacity)
    h[0] = r.integers(0, 0x70000, capacity).astype(np.int64).view(np.float64)
    for k, v in enumerate((np.nan, np.inf, -np.inf, -0.0, 5e-324)):
        h[6 + k, offset + (k * 7) % n] = v
    return h


def partition(P, capacity, precision):
    part = im.Partition(0, 0, precision)
    part.allocate(capacity, P.GridXTotal)
    part.update_constants(P)
    return part


def as_mixed(h, P, part):
    """The FP64 lines after their way through the mixed form."""
    fb, ox, oy = part.position_map()
    out = h.copy()
    out[0] = (h[0].view(np.int64) & 0xFFFFFFFF).view(np.float64)
    for line, o in ((4, ox), (5, oy)):
        q = np.clip(np.rint((h[line] * P.cellsize_inv + o) * 2.0 ** fb), 0.0, 4294967295.0)
        out[line] = (q * 2.0 ** -fb - o) * P.cellsize
    with np.errstate(over="ignore"):
        for line in (1, 2, 6, 7, 9, 10, 12, 13, 14, 15):
            out[line] = h[line].astype(np.float32).astype(np.float64)
        for line in (3, 8, 11):
            out[line] = (h[line] - 1.0).astype(np.float32).astype(np.float64) + 1.0
    return out


@pytest.mark.parametrize("precision", [im.PRECISION_FP64, im.PRECISION_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("n", SIZES)
def test_points_come_back(n, precision):
    P = scenes.make_params(GridX=256, GridY=128, GridXDimension=64.0, nPartitions=1, GridHaloSize=8)
    capacity, offset = n + 7, 3
    h = state(n, capacity, offset, n)
    part = partition(P, n + 5, precision)
    print(f"{n} points, precision {precision}", flush=True)
    part.transfer_points_from_soa_to_device(h, offset, n)
    out = np.full((16, capacity + 2), -7.25)
    part.transfer_from_device(out, 5)
    want = h if precision == im.PRECISION_FP64 else as_mixed(h, P, part)
    part.close()
    assert np.array_equal(out[:, 5:5 + n].view(np.int64), want[:, offset:offset + n].view(np.int64))
    assert np.all(out[:, :5] == -7.25) and np.all(out[:, 5 + n:] == -7.25)


def test_batch_scenes_come_back():
    """Scenes of several sizes one after the other through the same staging."""
    P = scenes.make_params(GridX=256, GridY=128, GridXDimension=64.0, nPartitions=1, GridHaloSize=8)
    sizes = [40000, 3, 8191]
    b = im.Batch(0, im.PRECISION_FP64)
    hs = []
    for k, n in enumerate(sizes):
        h = state(n, n, 0, 100 + k)
        h[0] = np.arange(n, dtype=np.int64).view(np.float64)      # no point disabled
        h[4] = np.sort(h[4])                                       # and x in order: the sort keeps the columns
        h[5] = 4.0
        hs.append(h)
        b.add_scene(P, h, n)
    b.commit()
    for k, n in enumerate(sizes):
        out = np.zeros((16, n))
        b.transfer_from_device(k, out)
        assert np.array_equal(np.sort(out[0].view(np.int64)), np.arange(n))
        order = out[0].view(np.int64)
        assert np.array_equal(out.view(np.int64), hs[k][:, order].view(np.int64))
    b.close()
