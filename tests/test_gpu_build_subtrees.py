"""Device build of meshes at the sizes where one wave builds a whole subtree: node sizes
around the rows of 16 lanes and the 64-lane wave, coordinates on a coarse grid (equal
centroids, zeros of both signs, leaves of several objects), against the CPU oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from rfmanta_amd import api, scenes  # noqa: E402


def check_build(oracle, v, i):
    on, oi, onn = oracle.build_bvh_approx(v, i)
    with api.Scene(v, i) as s:
        s.build(approximate=True)
        gi, gn = s.export_dynbvh()
    assert np.array_equal(gi, oi)
    a = gn.view(np.uint8).reshape(len(gn), 32)
    b = on.view(np.uint8).reshape(len(on), 32)
    bad = np.nonzero((a != b).any(1))[0]
    assert len(bad) == 0, (bad[:5], gn[bad[:3]], on[bad[:3]])


def _grid_mesh(n, seed, levels):
    rng = np.random.default_rng(seed)
    v = rng.integers(-levels, levels + 1, size=(3 * n, 3)).astype(np.float32)
    v[(v == 0) & (rng.random(v.shape) < 0.5)] = np.float32(-0.0)
    return v, np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)


SIZES = (4, 5, 15, 16, 17, 31, 32, 33, 47, 48, 49, 62, 63, 64, 65, 66, 200, 1000)


@pytest.mark.parametrize("levels", (1, 3, 40))
@pytest.mark.parametrize("n", SIZES)
def test_subtree_sizes(oracle, n, levels):
    check_build(oracle, *_grid_mesh(n, 100 * n + levels, levels))


@pytest.mark.parametrize("n", SIZES)
def test_subtree_sizes_soup(oracle, n):
    check_build(oracle, *scenes.soup(n, seed=n + 1000))


@pytest.mark.parametrize("scale", (1e-30, 1e18, 3e37))
def test_extreme_extents(oracle, scale):
    """Areas that underflow to zero or overflow to infinity."""
    v, i = scenes.soup(90, seed=4)
    m = np.abs(v).max()
    check_build(oracle, (v * np.float32(scale / m)).astype(np.float32), i)
