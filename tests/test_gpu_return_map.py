"""The Drucker-Prager return of crushed points against the FP64 oracle, which
goes by way of the SVD, where the parts of F that the kernels scale vanish or
dominate: isotropic F, pure stretch and shear, rotated F, F almost a rotation,
and large strain.  Three substeps; every field to 1e-9 of its scale and the
flags exactly, as in the other comparisons."""
import numpy as np
import pytest

import _oracle as O
import icempm_multi_amd as im
from icempm_multi_amd import scenes

pytestmark = pytest.mark.gpu

CRUSHED = 0x10000
FIELDS = {"x": (4, 6), "v": (6, 8), "F": (8, 12), "C": (12, 16), "Jp": (3, 4)}


def deformation(kind, n, r):
    one = np.ones(n)
    s = 1e-4 * r.normal(size=n)
    if kind == "isotropic":
        return np.array([1 + s, 0 * one, 0 * one, 1 + s])
    if kind == "stretch":
        return np.array([1 + s, 0 * one, 0 * one, 1 - s])
    if kind == "shear":
        return np.array([one, s, s, one])
    if kind == "rotated":
        a = r.uniform(-np.pi, np.pi, n)
        return np.array([np.cos(a) * (1 + s), -np.sin(a) * (1 - s), np.sin(a) * (1 + s), np.cos(a) * (1 - s)])
    if kind == "rotation":
        a = r.uniform(-np.pi, np.pi, n)
        return np.array([np.cos(a), -np.sin(a), np.sin(a), np.cos(a)]) + 1e-13 * r.normal(size=(4, n))
    return np.array([one, 0 * one, 0 * one, one]) + 0.05 * r.uniform(-1, 1, (4, n))


@pytest.mark.parametrize("flags", [im.STEP_GRAPH, im.STEP_DIRECT_P2G])
@pytest.mark.parametrize("kind", ["isotropic", "stretch", "shear", "rotated", "rotation", "large"])
def test_crushed_points_match_oracle(kind, flags):
    P, h, n = scenes.block_scene(nx=40, ny=24, grid=(80, 64), n_grains=20)
    P.InitialTimeStep = 1e-6
    r = np.random.default_rng(3)
    h[0, :n].view(np.int64)[:] |= CRUSHED
    h[3, :n] = np.where(r.random(n) < 0.3, 0.999, 1.0)
    h[8:12, :n] = deformation(kind, n, r)
    ref = h.copy()
    part = im.Partition(0, 0, im.PRECISION_FP64)
    part.allocate(h.shape[1], P.GridXTotal)
    part.update_constants(P)
    part.transfer_points_from_soa_to_device(h, 0, n)
    if not flags & im.STEP_DIRECT_P2G:
        part.sort_points()
        O.sort(P, ref, n)
    print(kind, n, flush=True)
    part.step(3, flags)
    out = np.zeros_like(h)
    part.transfer_from_device(out, 0)
    assert part.error_code == 0
    part.close()
    O.substeps(P, ref, n, 3, 0.0, 0)
    assert np.isfinite(ref[:, :n]).all()
    for name, (a, b) in FIELDS.items():
        scale = np.abs(ref[a:b, :n]).max()
        assert np.abs(out[a:b, :n] - ref[a:b, :n]).max() <= 1e-9 * scale, name
    assert np.array_equal(out[0, :n].view(np.int64), ref[0, :n].view(np.int64))
