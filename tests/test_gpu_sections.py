"""The sweep's section list: frames whose pixels hold fewer, exactly as many
and more sections than a list (192) equal the oracle's bit for bit, in one
column and in several, with colours grouped and walked."""
import numpy as np
import pytest

import gudni_amd as G
from gudni_amd import scenes as S
from tests import helpers as H

pytestmark = pytest.mark.gpu


def teeth(n, width, height):
    """One shape of n upright bars inside every pixel column, alternating
    between two colours' shapes: 2 n + 1 sections in every pixel."""
    bars = [[], []]
    for x in range(width):
        for i in range(n):
            x0 = x + (4 * i + 1) / (4.0 * n + 2)
            bars[i % 2].append(S.rectangle_pairs(x0, -1.0, x0 + 1.5 / (4.0 * n + 2), height + 1.0))
    shapes = [(S.solid_tag(i), b) for i, b in enumerate(bars) if b]
    return S.build_scene(width, height, shapes, [[0.9, 0.2, 0.1, 0.6], [0.1, 0.4, 0.8, 0.7]], name=f"teeth{n}")


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n,width,height", [(1, 1, 1), (95, 1, 3), (96, 1, 2), (31, 2, 2), (48, 2, 3), (97, 3, 2),
                                            (200, 1, 2), (1, 70, 9), (2, 64, 64)])
def test_section_lists(n, width, height, mode):
    scene = teeth(n, width, height)
    spec = G.default_spec(coverage_mode=mode)
    want = H.oracle_render(scene, spec)
    assert want["rc"] == 0
    r = G.Rasterizer(spec)
    try:
        got, f32 = H.gpu_render_level2(r, scene, spec)
    finally:
        r.close()
    assert np.array_equal(got, want["out"]), H.first_mismatch(got, want["out"])
    assert np.array_equal(f32, want["f32"])


@pytest.mark.parametrize("tile,width,height", [(32, 512, 768), (32, 300, 257), (64, 200, 130), (256, 40, 300), (16, 64, 33)])
def test_units_split_over_waves(tile, width, height):
    """Frames of few units run each unit in 1 to 64 waves, by their number and
    height; one pixel column holds more records than any of the small rings,
    so parts of units go through the retry pass."""
    bars = [S.rectangle_pairs(20 + (2 * i + 0.5) / 300, -1.0, 20 + (2 * i + 1.5) / 300, height + 1.0) for i in range(150)]
    rng = np.random.default_rng(width)
    shapes, cols = [(S.solid_tag(0), bars)], [[0.9, 0.2, 0.1, 0.6]]
    for i in range(1, 40):
        p = rng.uniform(0, 1, (int(rng.integers(3, 7)), 4)) * [width, height, width, height]
        shapes.append((S.nonzero(S.solid_tag(i)) if i % 3 == 0 else S.solid_tag(i), [p]))
        cols.append(rng.uniform(0, 1, 4))
    scene = S.build_scene(width, height, shapes, cols, name="split")
    spec = G.default_spec(max_tile_size=tile)
    want = H.oracle_render(scene, spec, want_f64=False)
    assert want["rc"] == 0
    r = G.Rasterizer(spec)
    try:
        got, f32 = H.gpu_render_level2(r, scene, spec)
        assert np.array_equal(got, want["out"]), H.first_mismatch(got, want["out"])
        assert np.array_equal(f32, want["f32"])
        assert np.array_equal(H.gpu_render_level1(r, scene, spec), want["out"])
    finally:
        r.close()


@pytest.mark.parametrize("copies,nonzero", [(1, False), (2, False), (5, True), (40, False)])
def test_records_that_tie(copies, nonzero):
    """Edges that several shapes share, edges that meet at one height and
    edges that cross: the lower parts of split records go back among records
    they tie with, in the reference's order."""
    w, h = 21, 19
    quads = [[(2.5, 1.0), (15.25, 4.0), (9.0, 17.5), (1.0, 12.0)], [(15.25, 4.0), (20.0, 4.0), (20.0, 12.0), (9.0, 17.5)],
             [(0.0, 4.0), (20.5, 4.0), (20.5, 8.0), (0.0, 8.0)], [(3.0, 2.0), (17.0, 16.0), (3.0, 16.0), (17.0, 2.0)],
             [(5.0, 0.5), (5.0, 18.5), (6.0, 18.5), (6.0, 0.5)]]
    rng = np.random.default_rng(copies)
    shapes, cols = [], []
    for k in range(copies):
        for i, p in enumerate(quads):
            tag = S.solid_tag(len(shapes))
            shapes.append((S.nonzero(tag) if nonzero and (i + k) % 2 else tag, [S.straight_pairs(p)]))
            cols.append(rng.uniform(0, 1, 4))
    scene = S.build_scene(w, h, shapes, cols, name="ties")
    for tile in (8, 256):
        for mode in (0, 1):
            spec = G.default_spec(max_tile_size=tile, coverage_mode=mode)
            want = H.oracle_render(scene, spec, want_f64=False)
            assert want["rc"] == 0
            r = G.Rasterizer(spec)
            try:
                got, f32 = H.gpu_render_level2(r, scene, spec)
            finally:
                r.close()
            assert np.array_equal(got, want["out"]), H.first_mismatch(got, want["out"])
            assert np.array_equal(f32, want["f32"])


@pytest.mark.parametrize("height,tile", [(1, 16), (51, 64), (52, 64), (120, 256), (256, 256)])
def test_adjoint_keeps_section_colours(height, tile):
    """Columns of fewer and more sections (5 a pixel) than the colours a lane
    keeps for the backward sweep (256): colour gradients of bars that do not
    overlap, over an opaque background, equal their closed form in FP64.
    Tolerance: 2 x 256 x 3 terms of either sign added in FP32, 2^-24 each."""
    w = 3
    a, b = [], []
    for x in range(w):
        a.append(S.rectangle_pairs(x + 0.125, -1.0, x + 0.375, height + 1.0))
        b.append(S.rectangle_pairs(x + 0.5, -1.0, x + 0.875, height + 1.0))
    cols = np.array([[0.9, 0.2, 0.1, 0.625], [0.1, 0.4, 0.8, 0.75]], np.float32)
    scene = S.build_scene(w, height, [(S.solid_tag(0), a), (S.solid_tag(1), b)], cols, name="bars")
    target = np.random.default_rng(height).uniform(0, 1, (height, w, 4)).astype(np.float32)
    r = G.Rasterizer(G.default_spec(max_tile_size=tile))
    try:
        adj = G.Adjoint(r, [(scene, target)])
        adj.run()
        loss, _, d_rgba, image = adj.result(0, image=True)
        adj.close()
    finally:
        r.close()
    c, cov, bg = cols.astype(np.float64), np.array([0.25, 0.375]), np.ones(3)
    over = c[:, :3] * c[:, 3:] + bg * (1.0 - c[:, 3:])
    rgb = cov @ over + (1.0 - cov.sum()) * bg
    assert np.abs(image[..., :3] - rgb).max() < 1e-6
    err = rgb - target[..., :3].astype(np.float64)
    g = 2.0 * err.sum(axis=(0, 1))
    want = np.concatenate([cov[:, None] * c[:, 3:] * g, (cov[:, None] * (c[:, :3] - bg) * g).sum(axis=1, keepdims=True)], axis=1)
    bound = 2.0 ** -24 * 2 * 256 * 3 * 2.0 * np.abs(err).sum()
    assert np.abs(d_rgba - want).max() <= max(bound, 1e-6)
    assert abs(loss - ((err ** 2).sum() + ((1.0 - target[..., 3].astype(np.float64)) ** 2).sum())) <= 1e-5 * loss
