"""Colouring of the per-colour layout (sv_color_round): every manifold takes the smallest colour that no
neighbour of higher priority has.  The device's colours equal greedy colouring in priority order, for worlds
of a single manifold to several thousand and for a body whose list is many chunks of neighbours long."""
import numpy as np
import pytest

from reactphysics3d_amd import scene as S
from tests.test_colouring_fixed_point import greedy

pytestmark = pytest.mark.gpu


def _plate(n):
    """n spheres resting on a dynamic plate on the ground."""
    sc = S.Scene("plate", S.make_settings(gravity=(0.0, 0.0, -9.81)))
    g = sc.add_body(S.STATIC, (0.0, 0.0, -0.5))
    sc.add_collider(g, S.BOX, (30.0, 30.0, 0.5))
    b = sc.add_body(S.DYNAMIC, (0.0, 0.0, 0.25))
    sc.add_collider(b, S.BOX, (8.0, 8.0, 0.25), density=50.0)
    for i in range(n):
        b = sc.add_body(S.DYNAMIC, (-7.0 + 0.95 * (i % 8), -7.0 + 0.95 * (i // 8), 1.0))
        sc.add_collider(b, S.SPHERE, (0.5,))   # neighbours touch
    return sc


def _prio(m):
    x = (np.arange(m, dtype=np.uint64) * 0x9E3779B1) & 0xFFFFFFFF
    x ^= x >> 16
    x = (x * 0x85EBCA6B) & 0xFFFFFFFF
    return x ^ (x >> 13)


@pytest.mark.parametrize("scene", [lambda: S.mixed_container(1, extent=(6.0, 6.0, 12.0), seed=8), lambda: _plate(7),
                                   lambda: _plate(48),
                                   lambda: S.mixed_container(700, extent=(20.0, 20.0, 12.0), seed=7),
                                   lambda: S.mixed_container(6000, extent=(60.0, 60.0, 12.0), seed=7)],
                         ids=["one", "plate_7", "plate_48", "heap_700", "heap_6000"])
def test_device_colours_are_greedy_by_priority(scene):
    from reactphysics3d_amd.lib import Batch
    sc = scene()
    dev = Batch(sc, solver="per_color")
    dev.step(1.0 / 60.0, 70)
    ct = dev.contacts()
    colour = {tuple(p): int(c) for p, c in zip(ct["colliders"].tolist(), ct["color"])}
    body = np.array([c[0] for c in sc.colliders])
    dynamic = np.array([b[0] == S.DYNAMIC for b in sc.bodies])
    pairs = [p for p in zip(*(a.tolist() for a in dev.pairs())) if p in colour]
    assert len(pairs) == len(colour) > 0
    mb = [tuple(int(body[c]) if dynamic[body[c]] else -1 for c in p) for p in pairs]
    prio = _prio(len(pairs))
    order = sorted(range(len(pairs)), key=lambda m: (-int(prio[m]), -m))
    want = greedy([mb[m] for m in order], len(dynamic))
    assert [colour[pairs[m]] for m in order] == want
