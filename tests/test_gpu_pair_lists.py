"""One narrowphase launch takes the test lists of all pair types; a workgroup has 4 mesh pairs or 16 others of a
list (np_tiles), more in long lists.  Batches with one, almost, exactly and more than that of several types at once,
and with more such shares than workgroups, give every pair the contacts it has alone."""
import numpy as np
import pytest

from reactphysics3d_amd import scene as S

pytestmark = pytest.mark.gpu

SHAPES = {S.SPHERE: (0.5,), S.CAPSULE: (0.3, 0.8), S.BOX: (0.4, 0.5, 0.3), S.HULL: None}


def _pair(a, b, k):
    """Two overlapping bodies of shapes a and b, a little different for every k."""
    rng = np.random.default_rng(17 * k + 5)
    sc = S.Scene("pair", S.make_settings(gravity=(0.0, 0.0, 0.0)))
    for s, x in ((a, 0.0), (b, 0.55)):
        q = rng.normal(size=4)
        body = sc.add_body(S.DYNAMIC, (x, 0.0, 0.1 * rng.random()), tuple(q / np.linalg.norm(q)))
        if s == S.HULL:
            u = rng.normal(size=(20, 3))
            h = sc.add_hull_from_points((0.45 * u / np.linalg.norm(u, axis=1)[:, None]).astype(np.float32))
            sc.add_collider(body, S.HULL, (float(h), 0.0, 0.0))
        else:
            sc.add_collider(body, s, SHAPES[s])
    return sc


def _run(scenes, steps=3):
    from reactphysics3d_amd.lib import Batch
    dev = Batch(scenes)
    dev.step(1.0 / 60.0, steps)
    ct, state = dev.contacts(), dev.bodies()
    out = []
    for w, b0 in enumerate(dev.body_base[:len(scenes)]):
        m = ct["colliders"][:, 0] // 2 == w   # two colliders a world
        n = ct["nb_points"][m]
        out.append([n] + [ct[k][m][:, :n[0] if len(n) else 0] for k in ("normal_depth", "local1", "local2", "impulse")] +
                   [a[b0:b0 + 2] for a in state])
    return out


TYPES = [(S.SPHERE, S.SPHERE), (S.SPHERE, S.CAPSULE), (S.CAPSULE, S.CAPSULE), (S.BOX, S.SPHERE),
         (S.CAPSULE, S.BOX), (S.BOX, S.BOX), (S.HULL, S.BOX), (S.HULL, S.CAPSULE), (S.HULL, S.HULL)]


def _check(counts, steps):
    kinds = [(t, k % 5) for t, n in enumerate(counts) for k in range(n)]
    alone = {tk: _run([_pair(*TYPES[tk[0]], tk[1])], steps)[0] for tk in set(kinds)}
    assert all(len(a[0]) for a in alone.values())
    order = np.random.default_rng(3).permutation(len(kinds))
    for i, got in zip(order, _run([_pair(*TYPES[kinds[i][0]], kinds[i][1]) for i in order], steps)):
        for a, b in zip(alone[kinds[i]], got):
            assert np.array_equal(a, b), kinds[i]


@pytest.mark.parametrize("counts", [(1, 1, 1, 1, 1, 1, 1, 1), (127, 0, 129, 0, 1, 0, 128, 0), (0, 130, 0, 128, 0, 300, 0, 1),
                                    (15, 16, 17, 33, 31, 15, 3, 16, 4), (1, 0, 0, 0, 0, 17, 5, 0, 8)])
def test_every_pair_has_the_contacts_it_has_alone(counts):
    _check(counts, 3)


# The first step is launched for the counts of a step before it, of which there is none: 72 workgroups.  The mesh and
# box pairs are 150 and 253 workgroups' shares, so that workgroups go from mesh pairs to box pairs.
@pytest.mark.parametrize("counts", [(0, 0, 0, 0, 0, 800, 200, 0, 200), (100, 0, 0, 0, 100, 2000, 300, 40, 210)])
def test_workgroups_with_pairs_of_several_types(counts):
    _check(counts, 1)


# points: 12 (30 edges), 24 (66 edges, two chunks of the edge tables), 44 (the most a mesh may have: 126 edges, 84
# faces), 0: a box
@pytest.mark.parametrize("points", [(12, 12), (24, 12), (12, 24), (24, 24), (44, 24), (44, 44), (44, 0), (0, 44)])
def test_mesh_search_finds_the_smallest_penetration(points):
    from scipy.spatial import ConvexHull
    from scipy.spatial.transform import Rotation
    from reactphysics3d_amd.lib import Batch
    rng = np.random.default_rng(points[0] * 1000 + points[1])
    scenes, want = [], []
    for _ in range(24):
        sc = S.Scene("pair", S.make_settings(gravity=(0.0, 0.0, 0.0)))
        world = []
        for n, x in zip(points, (0.0, 0.85)):
            q = rng.normal(size=4)
            q /= np.linalg.norm(q)
            body = sc.add_body(S.DYNAMIC, (x, 0.0, 0.0), tuple(q))
            if n:
                u = rng.normal(size=(n, 3))
                v = (0.5 * u / np.linalg.norm(u, axis=1)[:, None]).astype(np.float32)
                sc.add_collider(body, S.HULL, (float(sc.add_hull_from_points(v)), 0.0, 0.0))
            else:
                v = np.float32([(i, j, k) for i in (-0.35, 0.35) for j in (-0.3, 0.3) for k in (-0.4, 0.4)])
                sc.add_collider(body, S.BOX, (0.35, 0.3, 0.4))
            world.append(Rotation.from_quat(q).apply(v.astype(np.float64)) + (x, 0.0, 0.0))
        d = ConvexHull((world[0][:, None] - world[1][None]).reshape(-1, 3))
        want.append(-d.equations[:, 3].max())   # > 0: the depth of the origin in the Minkowski difference
        scenes.append(sc)
    dev = Batch(scenes)
    dev.step(1e-6)
    ct = dev.contacts()
    depth = np.zeros(len(scenes))
    for c, n, nd in zip(ct["colliders"], ct["nb_points"], ct["normal_depth"]):
        depth[c[0] // 2] = nd[:n, 3].max()
    want = np.array(want)
    touch = want > 1e-4
    assert touch.sum() >= 6 and not depth[want < -1e-4].any()
    # a face is taken unless an edge pair is shallower by the test's bias (0.2 per cent and 0.5 mm, twice); the contact
    # points of a face may miss its deepest vertex, never exceed it
    assert (depth[touch] > 0.0).mean() > 0.9
    assert (depth[touch] <= 1.005 * want[touch] + 0.0015).all()
    hit = touch & (depth > 0.0)
    assert np.median(depth[hit] / want[hit]) > 0.9


class _Copies:
    """A batch of worlds that repeat a few built ones."""

    def __init__(self, scenes, which):
        import ctypes
        from reactphysics3d_amd import lib
        self.batch = lib.Batch.__new__(lib.Batch)
        worlds = [lib.world_from_scene(sc) for sc in scenes]
        handles = (ctypes.c_void_p * len(which))(*[worlds[w] for w in which])
        b = self.batch
        b.worlds, b.scenes, b.nb = worlds, [scenes[w] for w in which], 2 * len(which)
        b.body_base = b.collider_base = 2 * np.arange(len(which) + 1)
        b.joint_base = np.zeros(len(which) + 1, np.int64)
        b.h = lib.load().rp3dg_batch_create(handles, len(which))
        assert b.h, lib.last_error()


# 4,096 mesh pairs are the last with 2 a wavefront, 16,384 box pairs the last with 8 (np_wave_pairs)
@pytest.mark.parametrize("counts", [(4096, 16385), (4097, 16384), (8195, 17)])
def test_wider_shares_in_long_lists(counts):
    types = [(S.HULL, S.HULL), (S.HULL, S.BOX), (S.BOX, S.BOX)]
    kinds = [(t, k) for t in range(3) for k in range(5)]
    which = np.array([i % 10 for i in range(counts[0])] + [10 + i % 5 for i in range(counts[1])])
    which = which[np.random.default_rng(3).permutation(len(which))]
    scenes = [_pair(*types[t], k) for t, k in kinds]
    dev = _Copies(scenes, which).batch
    dev.step(1.0 / 60.0, 1)
    ct, state = dev.contacts(), dev.bodies()
    order = np.argsort(ct["colliders"][:, 0] // 2, kind="stable")
    assert np.array_equal(ct["colliders"][order, 0] // 2, np.arange(len(which)))   # one manifold a world
    for k, sc in enumerate(scenes):
        n, *want = _run([sc], 1)[0]
        at = order[which == k]
        assert (ct["nb_points"][at] == n[0]).all()
        for key, w in zip(("normal_depth", "local1", "local2", "impulse"), want):
            assert (ct[key][at][:, :n[0]] == w).all(), (kinds[k], key)
        for a, w in zip(state, want[4:]):
            assert (a.reshape(len(which), 2, -1)[which == k] == w).all(), kinds[k]
