"""Colouring of a world group (sv_group_color in csrc/solver.hip): a manifold is coloured once it heads both its
bodies' lists of uncoloured manifolds.  On the CPU, the list schedule restated: its colours equal sequential
greedy colouring in manifold order, including the clamp when all 64 colours are used.  On the GPU, the
colours of a step's contacts equal greedy colouring of the pair table's colliding pairs in order."""
import random

import numpy as np
import pytest

from tests.test_colouring_fixed_point import greedy

NCOLORS = 64


def list_schedule(mb, nb):
    lists = [[m for m, bb in enumerate(mb) if b in bb] for b in range(nb)]
    head, mask = [0] * nb, [0] * nb
    left = [sum(b >= 0 for b in bb) for bb in mb]
    out = [0 if bb == (-1, -1) else None for bb in mb]
    ready = []

    def arrive(b):
        if head[b] < len(lists[b]):
            m = lists[b][head[b]]
            left[m] -= 1
            if left[m] == 0:
                ready.append(m)

    for b in range(nb):
        arrive(b)
    while ready:
        now, ready[:] = list(ready), []
        assert len({b for m in now for b in mb[m] if b >= 0}) == sum(b >= 0 for m in now for b in mb[m])
        random.shuffle(now)   # any order within a round
        for m in now:
            used = 0
            for b in mb[m]:
                used |= mask[b] if b >= 0 else 0
            c = next((k for k in range(NCOLORS) if not used >> k & 1), NCOLORS - 1)
            out[m] = c
            for b in mb[m]:
                if b >= 0:
                    mask[b] |= 1 << c
                    head[b] += 1
                    arrive(b)
    return out


@pytest.mark.parametrize("nb,nm,statics", [(1, 1, 0.9), (2, 40, 0.0), (3, 90, 0.3), (40, 300, 0.2), (300, 900, 0.1), (5, 400, 0.0)])
def test_list_schedule_equals_greedy(nb, nm, statics):
    rng = random.Random(nb * 1000 + nm)
    for _ in range(20):
        mb = []
        for _ in range(nm):
            x = rng.randrange(nb) if rng.random() >= statics else -1
            y = rng.randrange(nb) if rng.random() >= statics else -1
            mb.append((x, y if y != x else -1))
        assert list_schedule(mb, nb) == greedy(mb, nb)


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,groups", [((1,), 0), ((60, 3, 1), 0), ((260,), 0), ((700, 40), 512), ((3000,), 0), ((4000,), 0)])
def test_device_colours_are_greedy(sizes, groups):
    from reactphysics3d_amd import scene as S
    from reactphysics3d_amd.lib import Batch
    scenes = [S.mixed_container(n, extent=(max(6.0, (n * 0.6) ** 0.5),) * 2 + (12.0,), seed=7 + n) for n in sizes]
    dev = Batch(scenes, solver="fused", group_bodies=groups)
    for _ in range(12):
        dev.step(1.0 / 60.0)
    ct = dev.contacts()
    colour = {tuple(p): int(c) for p, c in zip(ct["colliders"].tolist(), ct["color"])}
    body = np.concatenate([[c[0] + b0 for c in sc.colliders] for sc, b0 in zip(scenes, dev.body_base)])
    dynamic = np.concatenate([[b[0] == S.DYNAMIC for b in sc.bodies] for sc in scenes])
    pairs = [p for p in zip(*(a.tolist() for a in dev.pairs())) if p in colour]
    assert len(pairs) == len(colour)
    mb = [tuple(int(body[c]) if dynamic[body[c]] else -1 for c in p) for p in pairs]
    assert [colour[p] for p in pairs] == greedy(mb, len(dynamic))
