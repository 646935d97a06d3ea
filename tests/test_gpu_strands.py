"""Generation runs only the strands that may meet a column's segment: records,
their order, labels and enclosures equal the oracle's where the choice is
close -- vertical tangents on and beside column borders, strands that pass a
segment by less and more than its margins, coordinates past 2^20, lists that
fill several times -- in compact and general tiles, under both fill rules."""
import math

import numpy as np
import pytest

import gudni_amd as G
from gudni_amd import scenes as S
from tests.test_gpu_parity import dump_parity

pytestmark = pytest.mark.gpu


def circle(cx, cy, r, k):
    a = 2 * math.pi * np.arange(k) / k
    m = a + math.pi / k
    rc = r / math.cos(math.pi / k)
    return np.stack([cx + r * np.cos(a), cy + r * np.sin(a), cx + rc * np.cos(m), cy + rc * np.sin(m)], axis=1)


def tangents(n, size):
    """Circles whose left and right tangents lie on, and up to 1/4 px beside,
    column borders, of radii from a pixel to several canvases."""
    rng = np.random.default_rng(n)
    shapes = []
    for i in range(n):
        r = float(np.exp(rng.uniform(0.0, math.log(4.0 * size))))
        x = float(rng.integers(0, size)) + float(rng.choice([0.0, 1e-4, -1e-4, 0.01, -0.05, 0.2, -0.25]))
        y = float(rng.uniform(0, size)) if i % 3 else float(rng.integers(0, size))
        c = circle(x + r if i % 2 else x - r, y, r, int(rng.integers(4, 13)))
        tag = S.solid_tag(i)
        shapes.append((S.nonzero(tag) if i % 4 == 3 else tag, [c]))
    return S.build_scene(size, size, shapes, rng.uniform(0, 1, (n, 4)), name=f"tangents{n}")


def zigzag(n, size):
    """A closed zigzag of n teeth: 2 n strands in one shape, filling the
    strand list several times; the teeth end on pixel rows and beside them."""
    x = np.linspace(0.5, size - 0.5, 2 * n)
    y = np.where(np.arange(2 * n) % 2 == 0, 3.0, size - 3.0 + 0.25 * (np.arange(2 * n) % 8))
    pts = list(zip(np.where(np.arange(2 * n) % 2 == 0, x + 2.0, x - 2.0), y)) + [(size - 1.0, size + 5.0), (1.0, size + 5.0)]
    return S.build_scene(size, size, [(S.solid_tag(0), [S.straight_pairs(pts)]), (S.nonzero(S.solid_tag(1)), [
        S.straight_pairs(pts)])], [[1, 0, 0, 0.5], [0, 0, 1, 0.5]], name=f"zigzag{n}")


def far_points(size, reach):
    """Outlines with points out at +-reach."""
    rng = np.random.default_rng(5)
    shapes = []
    for i in range(24):
        p = rng.uniform(0, size, (5, 4))
        p[i % 5, i % 4] = reach if i % 2 else -reach
        shapes.append((S.solid_tag(i), [p]))
    return S.build_scene(size, size, shapes, rng.uniform(0, 1, (24, 4)), name=f"far{reach:g}")


@pytest.mark.parametrize("tile", [8, 16, 64, 256])
@pytest.mark.parametrize("make", [lambda: tangents(60, 48), lambda: tangents(300, 64), lambda: zigzag(40, 64),
                                  lambda: zigzag(97, 128), lambda: far_points(64, 1000.0),
                                  lambda: far_points(64, float(1 << 20)), lambda: far_points(64, 3.0e7),
                                  lambda: S.uniform_512(260, 64, 11)])
def test_strand_choice(make, tile):
    scene = make()
    spec = G.default_spec(max_tile_size=tile)
    r = G.Rasterizer(spec)
    try:
        dump_parity(r, scene, lambda n: sorted({0, n - 1}), cap=1024, spec=spec)
    finally:
        r.close()
