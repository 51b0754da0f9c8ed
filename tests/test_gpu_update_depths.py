"""Rotating updates of trees of every small depth: the update goes two depths at a time,
so trees of odd and even depth, entries with one or two inner children, and leaves split in
the same frame (their new records are not rotated) all occur. Checked against the CPU
oracle's update."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from rfmanta_amd import api, scenes  # noqa: E402
from test_gpu_update import canonical_equal  # noqa: E402


def _skewed(n):
    """Triangles at ever smaller distances from a corner: a deep one-sided tree."""
    t = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0.5]], np.float32)
    v = np.concatenate([(t + 2) * np.float32(0.7 ** k) for k in range(n)])
    return v.astype(np.float32), np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)


def _frames(oracle, v, i, amp):
    nodes, ids, nn = oracle.build_bvh(v, i)
    st = oracle.RotState(nodes, ids, nn)
    rng = np.random.default_rng(len(i))
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        for f in range(4):
            vd = (v + rng.normal(0, amp, v.shape)).astype(np.float32)
            st.update(vd, i)
            s.set_vertices(vd)
            s.update()
            api.sync()
            gi, gn = s.export_dynbvh()
            ok, msg, count = canonical_equal(gn, gi, st.nodes, st.ids)
            assert ok, (f, msg)
            assert count == st.next_free.value


@pytest.mark.parametrize("n", (2, 3, 4, 5, 6, 7, 9, 12, 17, 25, 40, 70, 129, 300, 1500))
def test_update_small_trees(oracle, n):
    _frames(oracle, *scenes.soup(n, seed=n), 0.2)


@pytest.mark.parametrize("n", (8, 21, 40, 60))
def test_update_skewed_trees(oracle, n):
    _frames(oracle, *_skewed(n), 0.05)
