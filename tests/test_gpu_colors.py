"""Pictures and gradients at the edges of their cases equal the oracle's bit
for bit: texels inside, across and outside the picture's border, at its own
and other scales; gradients of 1 to 4 stops, with equal and descending
offsets, on and past their ends."""
import numpy as np
import pytest

import gudni_amd as G
from gudni_amd import scenes as S
from tests import helpers as H

pytestmark = pytest.mark.gpu


def check(scene, spec):
    want = H.oracle_render(scene, spec)
    assert want["rc"] == 0
    r = G.Rasterizer(spec)
    try:
        got, f32 = H.gpu_render_level2(r, scene, spec)
    finally:
        r.close()
    assert np.array_equal(got, want["out"]), H.first_mismatch(got, want["out"])
    assert np.array_equal(f32, want["f32"])


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("filt", [0, 1])
@pytest.mark.parametrize("w,h,scale", [(1, 1, 1.0), (2, 2, 1.0), (2, 1, 1.0), (7, 5, 1.0), (7, 5, 0.5), (7, 5, 3.7),
                                       (64, 64, 1.0), (3, 200, 0.3), (5, 5, 0.0)])
def test_picture_borders(w, h, scale, filt, mode):
    rng = np.random.default_rng(w * 1000 + h)
    data = rng.integers(0, 256, 4 * (3 + 2 * w * h), dtype=np.uint8)   # 12 bytes before the pictures
    uses = [(-3.5, -2.25, w, h, 12, scale), (0.0, 0.0, w, h, 12 + 4 * w * h, scale)]
    subs = [S.picture_substance(0), [0.2, 0.7, 0.1, 0.5], S.picture_substance(1)]
    shapes = [(S.picture_tag(0), [S.rectangle_pairs(-1.0, -1.0, 41.0, 30.0)]),
              (S.solid_tag(1), [S.straight_pairs([(2.3, 1.1), (30.2, 8.7), (6.5, 25.9)])]),
              (S.picture_tag(2), [S.rectangle_pairs(0.4, 0.3, 20.6, 33.0)])]
    check(S.build_scene(40, 33, shapes, subs, data, uses, name="pictures"),
          G.default_spec(max_tile_size=16, texture_filter=filt, coverage_mode=mode))


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("offsets", [(0.3,), (0.0, 1.0), (0.4, 0.4), (0.2, 0.5, 0.8), (0.7, 0.1, 0.5),
                                     (0.1, 0.3, 0.6, 0.9), (0.5, 0.5, 0.5, 0.5), (0.9, 0.6, 0.3, 0.0)])
def test_gradient_stops(offsets, kind, mode):
    rng = np.random.default_rng(len(offsets))
    cols = [rng.uniform(0, 1, (len(offsets), 4)) for _ in range(3)]
    ends = [((4.0, 3.0), (36.0, 21.0)), ((20.0, 16.0), (0.0 if kind else 20.0, 16.0)), ((50.0, -9.0), (30.0, 2.0))]
    grads = np.stack([S.gradient_record(kind, a, b, offsets, c) for (a, b), c in zip(ends, cols)])
    subs = [S.gradient_substance(0), S.gradient_substance(1), [0.9, 0.1, 0.3, 0.4], S.gradient_substance(2)]
    shapes = [(S.gradient_tag(0), [S.rectangle_pairs(-1.0, -1.0, 41.0, 34.0)]),
              (S.gradient_tag(1), [S.straight_pairs([(2.3, 1.1), (39.2, 8.7), (6.5, 30.9)])]),
              (S.solid_tag(2), [S.rectangle_pairs(10.5, 3.25, 31.0, 18.5)]),
              (S.gradient_tag(3), [S.straight_pairs([(38.0, 2.0), (35.0, 31.0), (12.0, 28.0)])])]
    check(S.build_scene(40, 33, shapes, subs, gradients=grads, name="gradients"),
          G.default_spec(max_tile_size=16, coverage_mode=mode))


@pytest.mark.parametrize("n", [1, 4, 5, 31, 32, 33, 64, 65, 100, 127])
def test_solids_among_gradients(n):
    """A tile of n shapes, every fifth a gradient: the tile's set of gradients
    reaches every bit of its words."""
    rng = np.random.default_rng(n)
    shapes, subs, grads = [], [], []
    for i in range(n):
        p = rng.uniform(-2, 34, (3, 2))
        if i % 5 == 4:
            grads.append(S.gradient_record(i % 2, p[0], p[1], (0.1, 0.8), rng.uniform(0, 1, (2, 4))))
            subs.append(S.gradient_substance(len(grads) - 1))
            shapes.append((S.gradient_tag(i), [S.straight_pairs(p)]))
        else:
            subs.append(rng.uniform(0, 1, 4).astype(np.float32))
            shapes.append((S.solid_tag(i), [S.straight_pairs(p)]))
    check(S.build_scene(32, 32, shapes, subs, gradients=np.stack(grads) if grads else None, name="solids"),
          G.default_spec(max_tile_size=32))
