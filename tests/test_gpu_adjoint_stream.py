"""Colour gradients of the adjoint where a lane sweeps far more sections than
it lists: the image equals the target in all but a few rows, or most sections
have no area.  Bars that do not overlap lie over an opaque background, so the
gradients have a closed form, evaluated here in FP64."""
import numpy as np
import pytest

import gudni_amd as G
from gudni_amd import scenes as S

pytestmark = pytest.mark.gpu

COLS = np.array([[0.9, 0.2, 0.1, 0.625], [0.1, 0.4, 0.8, 0.75]], np.float32)
GRADIENT = np.array([0.3, 0.6, 0.2, 0.5], np.float32)


def check(scene, cover, differs, spec):
    """cover: (n, H, W), how much of each pixel the n first substances cover;
    differs: (H, W), the pixels whose target is not the image.

    Tolerance: a term is some 64 roundings of values no larger than
    |dL/dC| x area (the composite below a layer is recovered by a division by
    1 - alpha >= 1/4), and N terms are added in FP32: 2^-24 (64 + N) of the sum
    of the terms' magnitudes."""
    rng = np.random.default_rng(scene.height)
    r = G.Rasterizer(spec)
    try:
        adj = G.Adjoint(r, [(scene, np.zeros((scene.height, scene.width, 4), np.float32))])
        adj.run()
        _, _, _, image = adj.result(0, image=True)
        adj.close()
        target = image.copy()
        target[differs] = rng.uniform(0, 1, (int(differs.sum()), 4)).astype(np.float32)
        adj = G.Adjoint(r, [(scene, target)])
        adj.run()
        loss, _, d_rgba, again = adj.result(0, image=True)
        adj.close()
    finally:
        r.close()
    assert np.array_equal(image, again)
    c = scene.substances.astype(np.float64)[:len(cover)]
    err = image.astype(np.float64) - target.astype(np.float64)
    assert abs(loss - (err ** 2).sum()) <= 1e-5 * loss
    g = 2.0 * err[..., :3]
    size = 2.0 * np.abs(err).sum(axis=-1)
    for i, w in enumerate(cover):
        sums = (w[..., None] * g).sum(axis=(0, 1))
        want = np.append(c[i, 3] * sums, ((c[i, :3] - 1.0) * sums).sum())
        bound = 2.0 ** -24 * (64 + differs.sum()) * (w * size).sum()
        assert np.abs(d_rgba[i] - want).max() <= bound, (i, d_rgba[i], want, bound)
    assert not d_rgba[len(cover):].any()


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("rows", [(0, 1), (0, 8), (20, 23)])
@pytest.mark.parametrize("height,tile", [(51, 64), (52, 64), (120, 256), (256, 256)])
def test_few_rows_differ(height, tile, rows, mixed):
    """Two bars in every column, 5 sections a pixel (7 with a gradient's bar),
    of which the rows that differ are listed."""
    w = 3
    bars = [[], [], []]
    for x in range(w):
        for b, (x0, x1) in zip(bars, ((0.125, 0.375), (0.5, 0.75), (0.8125, 0.9375))):
            b.append(S.rectangle_pairs(x + x0, -1.0, x + x1, height + 1.0))
    subs, grads = list(COLS), None
    shapes = [(S.solid_tag(0), bars[0]), (S.solid_tag(1), bars[1])]
    if mixed:
        grads = np.stack([S.gradient_record(0, (0.0, 0.0), (3.0, 9.0), (0.0, 1.0), [GRADIENT, GRADIENT])])
        subs.append(S.gradient_substance(0))
        shapes.append((S.gradient_tag(2), bars[2]))
    scene = S.build_scene(w, height, shapes, subs, gradients=grads, name="bars")
    differs = np.zeros((height, w), bool)
    differs[rows[0]:rows[1]] = True
    check(scene, np.ones((2, height, w)) * np.array([0.25, 0.25])[:, None, None], differs,
          G.default_spec(max_tile_size=tile))


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("copies,slivers,tile", [(101, 0, 8), (127, 0, 64), (301, 0, 8), (301, 0, 256), (301, 130, 8)])
def test_sections_without_area(copies, slivers, tile, mixed):
    """A bar drawn an odd number of times over itself: its edges coincide, so
    all but 5 of a pixel's sections have no area.  With 130 more shapes in the
    tile it is one that is not compact."""
    a = [S.rectangle_pairs(0.125, -1.0, 0.375, 9.0)]
    b = [S.rectangle_pairs(0.5, -1.0, 0.75, 9.0)] * copies
    shapes, subs = [(S.solid_tag(0), a), (S.solid_tag(1), b)], list(COLS)
    grads = None
    if mixed:
        grads = np.stack([S.gradient_record(1, (0.0, 0.0), (9.0, 0.0), (0.0, 1.0), [GRADIENT, GRADIENT])])
        subs.append(S.gradient_substance(0))
        shapes.append((S.gradient_tag(2), [S.rectangle_pairs(0.8125, -1.0, 0.9375, 9.0)]))
    for i in range(slivers):
        x = 5.0 + (i // 8 + 0.25) / 17.0
        shapes.append((S.solid_tag(len(subs)), [S.rectangle_pairs(x, i % 8, x + 0.5 / 17.0, i % 8 + 1.0)]))
        subs.append(np.array([0.5, 0.25, 0.75, 0.5], np.float32))
    scene = S.build_scene(8, 8, shapes, subs, gradients=grads, name="stacked")
    cover = np.zeros((2, 8, 8))
    cover[:, :, 0] = 0.25
    differs = np.zeros((8, 8), bool)
    differs[:, 0] = True
    check(scene, cover, differs, G.default_spec(max_tile_size=tile))
