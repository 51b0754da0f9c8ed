"""Packets over one-sided trees: the packet stack up to the deepest tree it takes (both of
its register pairs of 64 entries), whole and ragged packets, against the CPU oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from rfmanta_amd import api, scenes  # noqa: E402


def _chain(oracle, v, i, deep_left):
    """Leaves of one triangle, one per depth; the rest of the tree is the other child."""
    T = len(i)
    nodes = np.zeros(2 * T, oracle.NODE_DTYPE)
    rec, used = 0, 1
    for k in range(T - 1):
        nodes["child"][rec] = used
        leaf, rest = (used + 1, used) if deep_left else (used, used + 1)
        nodes["child"][leaf], nodes["children"][leaf] = k, 1
        rec, used = rest, used + 2
    nodes["child"][rec], nodes["children"][rec] = T - 1, 1
    ids = np.arange(T, dtype=np.int32)
    oracle.refit(v, i, nodes, ids)
    return nodes, ids


@pytest.mark.parametrize("deep_left", (False, True))
@pytest.mark.parametrize("n", (64, 65, 66, 127))
def test_packet_stack_depths(oracle, n, deep_left):
    v, i = scenes.soup(n, seed=n, sigma=0.4)
    nodes, ids = _chain(oracle, v, i, deep_left)
    rays = scenes.random_rays(1000, 5, (-1.3, -1.3, -1.3), (1.3, 1.3, 1.3))
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        _, tree = s.export_dynbvh()
        for packet in (2, 7, 63, 64):
            for any_hit in (False, True):
                g = s.trace_host(rays, any_hit=any_hit, packet_size=packet)
                o = oracle.trace(v, i, tree, ids, rays, any_hit=any_hit, packet_size=packet)
                assert np.array_equal(g["prim"], o["prim"]), (packet, any_hit)
                assert np.array_equal(g["t"].view(np.uint32), o["t"].view(np.uint32))
