"""The four-wide traversal against the oracle where it can go wrong: set sizes around the
waves' chunks, direction components of zero, rays outside its bounds, leaf sizes around the
two triangles of a step and the inline leaf count, trees whose boxes do not nest or whose
leaves overlap, and refits that meet or leave a vertex that is not a number. Results equal
the oracle's one-ray packets bit for bit (closest hit) or in flag and triangle (any hit)."""

import numpy as np
import pytest

from rfmanta_amd import _lib as L
from rfmanta_amd import api, scenes
from test_gpu_update import _tree_of_leaf_sizes

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


def _check(oracle, scene, v, i, nodes, ids, rays, what, **kw):
    for any_hit in (False, True):
        o = oracle.trace(v, i, nodes, ids, rays, packet_size=1, any_hit=any_hit, **kw)
        g = scene.trace_host(rays, any_hit=any_hit, packet_size=1)
        assert np.array_equal(g["prim"], o["prim"]), (what, any_hit)
        if any_hit:
            assert np.array_equal(g["occluded"], o["occluded"]), what
        else:
            for k in ("t", "u", "v"):
                assert np.array_equal(_bits(g[k]), _bits(o[k])), (what, k)


def _take(rays, n):
    return {k: np.ascontiguousarray(rays[k][:n]) for k in api.RAY_FIELDS}


@pytest.mark.parametrize("n", [1, 3, 4, 5, 63, 64, 65, 1023, 4097, 65537])
def test_set_sizes(oracle, n):
    v, i = scenes.heightfield(60, 40, seed=9)
    nodes, ids, _ = oracle.build_bvh(v, i)
    rays = scenes.random_rays(n, 5, (-1, -0.3, -0.7), (1, 0.6, 0.7))
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        _check(oracle, s, v, i, nodes, ids, rays, n)


def _odd_rays(n=640):
    """Rays with zero components of both signs, tiny and huge directions, origins on box
    planes, infinite and absent tmax, and components that are not finite."""
    r = scenes.random_rays(n, 11, (-1.2, -0.5, -1.2), (1.2, 0.5, 1.2))
    k = np.arange(n)
    f = np.float32
    for a, c in enumerate(("dx", "dy", "dz")):
        r[c][k % 16 == a] = f(0.0)
        r[c][k % 16 == 3 + a] = f(-0.0)
    for c in ("dx", "dy", "dz"):
        r[c][k % 16 == 6] *= f(1e-30)
        r[c][k % 16 == 7] *= f(1e25)
    r["dx"][k % 16 == 8] *= f(1e-20)
    two = k % 16 == 9
    r["dx"][two], r["dz"][two] = f(0.0), f(0.0)
    r["ox"][two] = np.round(r["ox"][two] * 8) / 8
    r["tmax"][k % 16 == 10] = np.inf
    r["dx"][k % 32 == 10] = f(0.0)
    r["tmax"][k % 16 == 11] = f(0.3)
    r["ox"][k % 16 == 12] = f(1e6)
    bad = k % 16 == 13
    r["oy"][bad] = np.where(k[bad] % 32 < 16, f(np.nan), f(np.inf))
    r["dy"][k % 16 == 14] = f(np.inf)
    r["tmax"][k % 16 == 15] = np.where(k[k % 16 == 15] % 32 < 16, f(np.nan), f(-1.0))
    return r


@pytest.mark.parametrize("mesh", ["soup", "heightfield", "grid"])
def test_odd_rays(oracle, mesh):
    if mesh == "soup":
        v, i = scenes.soup(700, seed=2, sigma=0.1)
    else:
        v, i = scenes.heightfield(17, 17, seed=2)
        if mesh == "grid":  # flat boxes, vertices on binary fractions
            v[:, 1] = 0
    nodes, ids, _ = oracle.build_bvh(v, i)
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        _check(oracle, s, v, i, nodes, ids, _odd_rays(), mesh)


def _chain_of_leaves(oracle, v, i, sizes):
    """A tree whose inner records each hold one leaf of the next size and the rest."""
    T = len(i)
    ids = np.arange(T, dtype=np.int32)
    tri = v[i.astype(np.int64)]
    lo, hi = tri.min(1), tri.max(1)
    off = np.concatenate([[0], np.cumsum(sizes)])
    m = len(sizes)
    nodes = np.zeros(2 * T, oracle.NODE_DTYPE)

    def leaf(r, k):
        a, b = off[k], off[k + 1]
        nodes[r]["lo"], nodes[r]["hi"] = lo[a:b].min(0), hi[a:b].max(0)
        nodes[r]["child"], nodes[r]["children"] = a, sizes[k]

    for k in range(m - 1):
        r = 2 * k
        nodes[r]["lo"], nodes[r]["hi"] = lo[off[k]:].min(0), hi[off[k]:].max(0)
        nodes[r]["child"], nodes[r]["axis"] = 2 * k + 1, k % 3
        leaf(2 * k + 1, k)
    leaf(2 * (m - 1), m - 1)
    return nodes, ids


def test_leaf_sizes(oracle):
    sizes = [1, 2, 3, 4, 5, 13, 14, 15, 16, 17, 31, 1, 2]
    v, i = scenes.soup(sum(sizes), seed=8, sigma=0.3)
    nodes, ids = _chain_of_leaves(oracle, v, i, sizes)
    rays = scenes.random_rays(3000, 4, (-1, -1, -1), (1, 1, 1))
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        _check(oracle, s, v, i, nodes, ids, rays, "chain")


@pytest.mark.parametrize("how", ["not nested", "overlapping"])
def test_trees_that_take_the_reference_steps(oracle, how):
    v, i = scenes.heightfield(24, 16, seed=6)
    nodes, ids, nn = oracle.build_bvh(v, i)
    nodes = nodes.copy()
    if how == "not nested":  # inner boxes shrunk: what they cut off is never visited
        inner = np.nonzero(nodes["children"][:nn] == 0)[0][1::3]
        nodes["hi"][inner, 0] -= np.float32(0.02)
    else:  # a leaf that also holds its neighbour's first triangle
        leaves = [r for r in range(nn) if nodes[r]["children"] > 0]
        a = next(r for r in leaves if nodes[r]["child"] + nodes[r]["children"] < len(i))
        nodes["children"][a] += 1
    rays = scenes.random_rays(4000, 3, (-1, 0.1, -0.7), (1, 0.6, 0.7))
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        _check(oracle, s, v, i, nodes, ids, rays, how)


@pytest.mark.parametrize("mesh", ["heightfield", "grid", "soup"])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_axis_parallel_rays_without_end(oracle, mesh, axis):
    """Infinite tmax and one or two zero components, origins on and off box planes."""
    if mesh == "soup":
        v, i = scenes.soup(700, seed=2, sigma=0.1)
    else:
        v, i = scenes.heightfield(17, 17, seed=2)
        if mesh == "grid":
            v[:, 1] = 0
    nodes, ids, _ = oracle.build_bvh(v, i)
    n = 1200
    rays = scenes.random_rays(n, 13 + axis, (-1.2, -1.2, -1.2), (1.2, 1.2, 1.2))
    k = np.arange(n)
    d = ["dx", "dy", "dz"]
    rays[d[axis]][:] = np.where(k % 2, 1, -1) * np.float32(1)
    rays[d[(axis + 1) % 3]][:] = np.where(k % 4 < 2, 0.0, -0.0)
    rays[d[(axis + 2) % 3]][k % 3 == 0] = 0.0
    for o in ("ox", "oy", "oz"):
        on = k % 5 < 2
        rays[o][on] = np.round(rays[o][on] * 8) / 8
    rays["tmax"][:] = np.inf
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        _check(oracle, s, v, i, nodes, ids, rays, mesh)


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_rays_through_vertices(oracle, axis):
    """Axis-parallel rays from the planes of their leaves' boxes, the other components zeros of
    both signs or tiny, so that whole waves hit leaves that the reference does not enter."""
    v, i = scenes.heightfield(33, 29, seed=4)
    v = np.ascontiguousarray(np.roll(v, axis - 1, axis=1))
    nodes, ids, _ = oracle.build_bvh(v, i)
    small = [0.0, -0.0, 6e-17, -6e-17, 1e-30, -1e-13]
    n, m = len(v), len(small)
    rays = {k: np.zeros(2 * m * n, np.float32) for k in api.RAY_FIELDS}
    for k, c in enumerate("xyz"):
        rays["o" + c][:] = np.tile(v[:, k], 2 * m)
        rays["d" + c][:] = np.repeat(np.array([small, small[1:] + small[:1]], np.float32).ravel(), n)
    sign = np.repeat([1.0, -1.0], m * n).astype(np.float32)
    rays["d" + "xyz"[axis]][:] = sign
    rays["o" + "xyz"[axis]][:] = -2 * sign
    rays["tmax"][:] = 1e19
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        _check(oracle, s, v, i, nodes, ids, rays, axis)
        _check_frames(oracle, s, v, i, nodes, ids, rays, axis)


def test_origin_in_the_plane_of_a_flat_leaf(oracle):
    """Rays without an x component in the plane of a leaf's flat box, which passes the
    reference's slab test while its parent's fails (a loaded tree whose leaf holds its
    triangle's box of another pose)."""
    v = np.array([[0.5, -1, 1], [0.5, 2, 1], [-1, 0, 1], [3, -1, 2], [3, 2, 2], [2, 0, 2]], np.float32)
    i = np.arange(6, dtype=np.uint32).reshape(2, 3)
    nodes = np.zeros(4, oracle.NODE_DTYPE)
    for r, (lo, hi) in enumerate([((0.25, -2, 0), (3, 2, 2)), ((0.25, -2, 0), (0.25, 2, 2)),
                                  ((2, -1, 2), (3, 2, 2))]):
        nodes["lo"][r], nodes["hi"][r] = lo, hi
    nodes["child"][0] = 1
    nodes["child"][1], nodes["children"][1] = 0, 1
    nodes["child"][2], nodes["children"][2] = 1, 1
    rays = {k: np.zeros(256, np.float32) for k in api.RAY_FIELDS}
    rays["ox"][:] = 0.25
    rays["dx"][1::2] = -0.0
    rays["oy"][:] = np.linspace(-0.9, 1.9, 256)
    rays["dz"][:] = 1
    rays["tmax"][:] = np.where(np.arange(256) % 4 < 2, 1e19, np.inf)
    ids = np.arange(2, dtype=np.int32)
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        _check(oracle, s, v, i, nodes, ids, rays, "flat")


def test_leaf_boxes_that_do_not_hold_their_triangles(oracle):
    """A loaded tree may hold boxes of another pose. Along the ray: a leaf whose box the ray
    misses by less than the inner boxes are widened, with a triangle on the ray at 10; a leaf
    whose box starts at 11, with a triangle at 3; a leaf with its triangle at 5. The reference
    never enters the first leaf, so it enters the second."""
    def wall(x):
        return [[x, -1, -1], [x, 1, -1], [x, 0, 2]]

    v = np.array(wall(10) + wall(3) + wall(5), np.float32)
    i = np.arange(9, dtype=np.uint32).reshape(3, 3)
    nodes = np.zeros(6, oracle.NODE_DTYPE)
    box = [((3, -1, -1), (12, 1, 2)), ((3, -1, -1), (12, 1, 2)), ((5, -1, -1), (5, 1, 2)),
           ((10, -1, -1), (10, -5e-6, 2)), ((11, -1, -1), (12, 1, 2))]
    for r, (lo, hi) in enumerate(box):
        nodes["lo"][r], nodes["hi"][r] = lo, hi
    nodes["child"][0], nodes["child"][1] = 1, 3
    for r, slot in ((2, 2), (3, 0), (4, 1)):
        nodes["child"][r], nodes["children"][r] = slot, 1
    ids = np.arange(3, dtype=np.int32)
    n = 70
    rays = {k: np.zeros(n, np.float32) for k in api.RAY_FIELDS}
    rays["dx"][:] = 1
    rays["tmax"][:] = 1e19
    rays["oz"][:] = np.linspace(-0.3, 0.3, n)
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        assert (oracle.trace(v, i, nodes, ids, rays, packet_size=1)["prim"] == 1).all()
        _check(oracle, s, v, i, nodes, ids, rays, "stale boxes")


def _check_frames(oracle, scene, v, i, nodes, ids, rays, what):
    sets = [(rays, False), (_take(rays, 777), True)]
    dev = [(api.DeviceRays.upload(r), api.DeviceHits.alloc(len(r["ox"]), any_hit=a), a)
           for r, a in sets]
    f = api.Frame(scene, dev)
    for refill, chunk in ((64, 0), (24, 64)):
        f.set_config(dict(layout=L.MH_LAYOUT_PAIR, stack_lds=8, block=64, blocks_per_cu=1,
                          refill=refill, chunk=chunk, reverse=0))
        f.launch()
        api.sync()
        for (_, dh, a), (r, _) in zip(dev, sets):
            o = oracle.trace(v, i, nodes, ids, r, packet_size=1, any_hit=a)
            g = dh.download()
            assert np.array_equal(g["prim"], o["prim"]), (what, refill, a)
            if not a:
                assert np.array_equal(_bits(g["t"]), _bits(o["t"])), (what, refill)
    f.close()


@pytest.mark.parametrize("how", ["not nested", "overlapping", "two large leaves at one slot"])
def test_trees_traversed_on_their_records(oracle, how):
    """Leaves around the inline leaf count in trees that the wide nodes do not serve, with odd
    rays among the others."""
    sizes = [1, 2, 3, 14, 15, 16, 17, 31, 1, 2, 5, 20]
    v, i = scenes.soup(sum(sizes), seed=8, sigma=0.3)
    nodes, ids = _chain_of_leaves(oracle, v, i, sizes)
    if how == "not nested":
        nodes["hi"][2:20:4, 0] -= np.float32(0.1)
    elif how == "overlapping":
        nodes["children"][3] += 1
    else:  # the leaf before starts with the next one's objects, four fewer
        r = 2 * sizes.index(20) - 1
        nodes["child"][r], nodes["children"][r] = sum(sizes) - 20, 16
    rays = scenes.random_rays(3000, 4, (-1, -1, -1), (1, 1, 1))
    odd = _odd_rays()
    rays = {k: np.concatenate([rays[k], odd[k]]) for k in api.RAY_FIELDS}
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        _check(oracle, s, v, i, nodes, ids, rays, how)
        _check_frames(oracle, s, v, i, nodes, ids, rays, how)


def test_refit_with_a_vertex_that_is_not_a_number(oracle):
    v, i = scenes.heightfield(40, 30, seed=3)
    nodes, ids, _ = oracle.build_bvh(v, i)
    rays = scenes.random_rays(5000, 7, (-1, -0.2, -0.7), (1, 0.6, 0.7))
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        for value in (np.nan, 0.05):
            vd = v.copy()
            vd[600, 1] = value
            s.set_vertices(vd)
            s.refit()
            api.sync()
            gi, gn = s.export_dynbvh()
            if not np.isnan(value):
                ref = nodes.copy()
                oracle.refit(vd, i, ref, ids)
                assert gn.tobytes() == ref.tobytes()
            # the tree as it stands on the device, box for box
            _check(oracle, s, vd, i, gn, gi, rays, value)


@pytest.mark.parametrize("seed", range(4))
def test_update_with_a_vertex_that_is_not_a_number(oracle, seed):
    rng = np.random.default_rng(seed)
    sizes = [int(x) for x in rng.integers(3, 9, 60)]
    v, i = scenes.soup(sum(sizes), seed=seed, sigma=0.3)
    ids = rng.permutation(sum(sizes)).astype(np.int32)
    nodes, _ = _tree_of_leaf_sizes(oracle, v, i, sizes, ids)
    starts = np.cumsum([0] + sizes[:-1])
    rays = scenes.random_rays(4000, 7 + seed, (-1, -1, -1), (1, 1, 1))
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        for bad in (True, False):
            vd = v.copy()
            if bad:  # the last corner of a leaf's first object, dropped from the leaf's box
                vd[i[ids[starts[::3]], 2], seed % 3] = np.nan
            s.set_vertices(vd)
            s.update()
            api.sync()
            gi, gn = s.export_dynbvh()
            _check(oracle, s, vd, i, gn, gi, rays, bad)
            g = s.trace_host(rays, packet_size=64)
            o = oracle.trace(vd, i, gn, gi, rays, packet_size=64)
            assert np.array_equal(g["prim"], o["prim"]), bad
            assert np.array_equal(_bits(g["t"]), _bits(o["t"])), bad


@pytest.mark.parametrize("n", [2, 4])
def test_single_leaf_with_a_vertex_that_is_not_a_number(oracle, n):
    v, i = scenes.soup(n, seed=n, sigma=0.5)
    bad = v.copy()
    bad[i[-1, 2], 1] = np.nan
    nodes = np.zeros(2 * n, oracle.NODE_DTYPE)
    nodes["children"][0] = n
    ids = np.arange(n, dtype=np.int32)
    oracle.refit(bad, i, nodes, ids)
    rays = scenes.random_rays(2000, n, (-1.5, -1.5, -1.5), (1.5, 1.5, 1.5))
    with api.Scene(bad, i) as s:
        s.load_dynbvh(ids, nodes)
        for k, step in enumerate([None, s.refit, s.update]):
            for vd in (bad, v) if step else (bad,):
                if step:
                    s.set_vertices(vd)
                    step()
                    api.sync()
                gi, gn = s.export_dynbvh()
                _check(oracle, s, vd, i, gn, gi, rays, k)
                g = s.trace_host(rays, packet_size=64)
                o = oracle.trace(vd, i, gn, gi, rays, packet_size=64)
                assert np.array_equal(g["prim"], o["prim"]), k
                assert np.array_equal(_bits(g["t"]), _bits(o["t"])), k


def test_frames_of_a_single_record(oracle):
    v, i = scenes.soup(3, seed=1, sigma=0.5)
    nodes = np.zeros(1, oracle.NODE_DTYPE)
    nodes["children"] = 3
    nodes["lo"], nodes["hi"] = v.min(0), v.max(0)
    ids = np.arange(3, dtype=np.int32)
    rays = scenes.random_rays(500, 2, (-1.5, -1.5, -1.5), (1.5, 1.5, 1.5))
    o = oracle.trace(v, i, nodes, ids, rays, packet_size=1)
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        dh = api.DeviceHits.alloc(500)
        f = api.Frame(s, [(api.DeviceRays.upload(rays), dh, False)])
        for layout in (L.MH_LAYOUT_PAIR, L.MH_LAYOUT_REF, L.MH_LAYOUT_SOA):
            f.set_config(dict(layout=layout, stack_lds=8, block=64, blocks_per_cu=1, refill=64,
                              chunk=64, reverse=0))
            dh.arrays["prim"].upload(np.full(500, 777, np.int32))
            f.launch()
            api.sync()
            assert np.array_equal(dh.download()["prim"], o["prim"]), layout
        f.close()


@pytest.mark.parametrize("batches", [1, 3])
def test_frames_of_zero_components_and_short_chunks(oracle, batches):
    v, i = scenes.heightfield(50, 30, seed=5)
    nodes, ids, _ = oracle.build_bvh(v, i)
    sets = [_odd_rays(640)] + [scenes.random_rays(n, n, (-1, -0.2, -0.7), (1, 0.5, 0.7))
                               for n in (1, 777)]
    kinds = [False, True, False]
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        dev = [(api.DeviceRays.upload(r), api.DeviceHits.alloc(len(r["ox"]), any_hit=a), a)
               for r, a in list(zip(sets, kinds))[:batches]]
        f = api.Frame(s, dev)
        for refill, chunk in ((64, 0), (64, 64), (64, 256), (24, 64)):
            for rev in (0, 1):
                f.set_config(dict(layout=L.MH_LAYOUT_PAIR, stack_lds=8, block=64, blocks_per_cu=1,
                                  refill=refill, chunk=chunk, reverse=rev))
                for _, dh, _ in dev:
                    dh.arrays["prim"].upload(np.full(dh.n, 777, np.int32))
                f.launch()
                api.sync()
                for (_, dh, a), r in zip(dev, sets):
                    o = oracle.trace(v, i, nodes, ids, r, packet_size=1, any_hit=a)
                    g = dh.download()
                    assert np.array_equal(g["prim"], o["prim"]), (refill, chunk, rev)
                    if not a:
                        assert np.array_equal(_bits(g["t"]), _bits(o["t"])), (refill, chunk, rev)
        f.close()

def _one_sided(oracle, v, i, deep_left=False):
    """A leaf of one triangle at every depth."""
    T = len(i)
    nodes = np.zeros(2 * T, oracle.NODE_DTYPE)
    rec = 0
    for k in range(T - 1):
        c = 2 * k + 1
        nodes["child"][rec], nodes["axis"][rec], nodes["bits"][rec] = c, k % 3, k % 2
        leaf, rec = (c + 1, c) if deep_left else (c, c + 1)
        nodes["child"][leaf], nodes["children"][leaf] = k, 1
    nodes["child"][rec], nodes["children"][rec] = T - 1, 1
    ids = np.arange(T, dtype=np.int32)
    oracle.refit(v, i, nodes, ids)
    return nodes, ids


@pytest.mark.parametrize("deep_left", [False, True])
@pytest.mark.parametrize("n", [20, 65, 130, 256])
def test_deep_trees_spill(oracle, n, deep_left):
    """One-sided trees: the stack beyond each ring size, of the wide nodes, of the records (a
    tree that does not nest) and of the reference's own steps (odd rays)."""
    v, i = scenes.soup(n, seed=n, sigma=0.4)
    nodes, ids = _one_sided(oracle, v, i, deep_left)
    rays = scenes.random_rays(1500, 5, (-1.3, -1.3, -1.3), (1.3, 1.3, 1.3))
    odd = _odd_rays()
    rays = {k: np.concatenate([rays[k], odd[k]]) for k in api.RAY_FIELDS}
    bad = nodes.copy()
    bad["hi"][1:2 * n - 1:5, 0] -= np.float32(0.05)
    with api.Scene(v, i) as s:
        for tree in (nodes, bad):
            s.load_dynbvh(ids, tree)
            dr, dh = api.DeviceRays.upload(rays), api.DeviceHits.alloc(len(rays["ox"]))
            o = oracle.trace(v, i, tree, ids, rays, packet_size=1)
            for ring in (8, 16, 32):
                dh.arrays["prim"].upload(np.full(dh.n, 777, np.int32))
                s.trace(dr, dh, False, api.trace_opts(stack_lds=ring))
                api.sync()
                g = dh.download()
                assert np.array_equal(g["prim"], o["prim"]), ring
                assert np.array_equal(_bits(g["t"]), _bits(o["t"])), ring
            _check_frames(oracle, s, v, i, tree, ids, rays, n)


@pytest.mark.parametrize("ring", [0, 8, 16])
def test_noalloc_on_deep_trees(oracle, ring):
    """Depths where the fixed area holds the records' stack but not the wide nodes'."""
    v, i = scenes.soup(72, seed=3, sigma=0.4)
    nodes, ids = _one_sided(oracle, v, i)
    n = 70_001
    rays = scenes.random_rays(n, 6, (-1.3, -1.3, -1.3), (1.3, 1.3, 1.3))
    with api.Scene(v, i) as s:
        s.load_dynbvh(ids, nodes)
        dr, dh = api.DeviceRays.upload(rays), api.DeviceHits.alloc(n)
        opts = api.trace_opts(stack_lds=ring)
        L.check(L.load().mh_trace_noalloc(s.h, dr.struct(), dh.struct(), n, 0, opts, None))
        api.sync()
        o = oracle.trace(v, i, nodes, ids, rays, packet_size=1)
        g = dh.download()
        assert np.array_equal(g["prim"], o["prim"])
        assert np.array_equal(_bits(g["t"]), _bits(o["t"]))
