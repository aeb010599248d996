"""Launch plans of the 2D register and life tiles over the sizes they take: every plan
advances the run, within the tile's halo, by an odd number of sweeps where there is no
spare buffer, and by an even one before another launch where there is one."""
import random

import pytest

import shapes

SHAPES = {shapes.J5: {(2, 16), (4, 8), (4, 16), (8, 8)}, shapes.BOX9: {(2, 8), (2, 16), (4, 8), (4, 16)},
          shapes.CLOUD: {(2, 8), (2, 16), (4, 8)}, shapes.LIFE8: {(2, 8), (2, 16), (4, 16), (8, 8), (8, 16)}}
DEEPEST = {shapes.LIFE8: 31}


@pytest.mark.parametrize("odd", [False, True])
@pytest.mark.parametrize("pattern", sorted(SHAPES))
def test_plans(pattern, odd):
    l = shapes.lib()
    rng = random.Random(pattern)
    seen = set()
    sizes = [(9, 3), (10, 16), (256, 32), (257, 33), (2048, 2048), (4096, 4096), (16000, 16000), (9, 20000), (60000, 3)]
    sizes += [(int(9 * 2 ** rng.uniform(0, 13)), int(3 * 2 ** rng.uniform(0, 14.5))) for _ in range(400)]
    for w, h in sizes:
        for rem in (1, 2, 3, 8, 17, 32, 33, 100, 12345):
            left, launches = rem, 0
            while left and launches < 40:
                r, nw, k = shapes.plan(l, pattern, w, h, left, odd)
                rows = r * nw
                assert (r, nw) in SHAPES[pattern] and 1 <= k <= min(left, DEEPEST.get(pattern, 32)), (w, h, left, k)
                assert h <= rows or 2 * k < rows, (w, h, rows, k)
                if pattern != shapes.LIFE8:
                    assert w <= 256 or 2 * (-(-k // 4) * 4) < 256, (w, k)
                if odd:
                    assert k % 2 == 1, (w, h, left, k)
                else:
                    assert k % 2 == 0 or k == left or k == 1, (w, h, left, k)
                seen.add((r, nw))
                left -= k
                launches += 1
    assert seen == SHAPES[pattern]  # every shape that is built is some grid's
