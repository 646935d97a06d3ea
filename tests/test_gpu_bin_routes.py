"""A small scene's tree is tried by one block first; a scene that outgrows it is
built by level launches.  The tree is the host's wherever the block stops, and
what a context binned before costs the next scene nothing."""
import time

import numpy as np
import pytest

import gudni_amd as G
from gudni_amd import scenes as S
from tests.test_gpu_binning import compare_binning

pytestmark = pytest.mark.gpu


def clustered(n, size, part):
    """n outlines that all lie in a corner, 1 / part of the canvas wide."""
    rng = np.random.default_rng(n)
    shapes = [(S.solid_tag(i), [rng.uniform(0, size / part, (4, 4))]) for i in range(n)]
    return S.build_scene(size, size, shapes, rng.uniform(0, 1, (n, 4)), name="clustered")


@pytest.mark.parametrize("tile", [8, 64, 256])
@pytest.mark.parametrize("make", [lambda: S.uniform_512(1000, 512, 1), lambda: S.uniform_512(148, 363, 2),
                                  lambda: S.uniform_512(126, 388, 3), lambda: S.uniform_512(125, 256, 4),
                                  lambda: clustered(600, 1024, 4), lambda: clustered(300, 512, 16),
                                  lambda: S.build_scene(512, 512, [(S.solid_tag(0), [S.rectangle_pairs(1, 1, 500, 3)])],
                                                        [[1, 0, 0, 1]], name="one")])
def test_tree_wherever_the_block_stops(make, tile):
    spec = G.default_spec(max_tile_size=tile)
    r = G.Rasterizer(spec)
    try:
        scene = make()
        compare_binning(r, scene, spec)
        compare_binning(r, S.batch_scene(250, 120, 3), spec)
        compare_binning(r, scene, spec)
    finally:
        r.close()


def test_binning_does_not_depend_on_the_scene_before():
    """The median time of a large scene's scene_bin is the same after a small
    scene and after itself; 1.2 times allows for noise."""
    big, small = S.uniform_512(1000, 512, 1), S.batch_scene(250, 120, 3)
    r = G.Rasterizer(G.default_spec())
    try:
        def timed(scene):
            r.scene_upload_outlines(scene)
            t = time.perf_counter()
            r.scene_bin()
            return time.perf_counter() - t
        for scene in (big, small, big):
            timed(scene)
        after_small, after_big = [], []
        for _ in range(15):
            timed(small)
            after_small.append(timed(big))
            after_big.append(timed(big))
    finally:
        r.close()
    assert np.median(after_small) <= 1.2 * np.median(after_big)


@pytest.mark.parametrize("tile", [16, 32, 64, 256])
@pytest.mark.parametrize("make", [lambda: S.batch_scene(400, 4000, 4000), lambda: S.batch_scene(1000, 4000, 4000),
                                  lambda: S.batch_scene(1920, 1000, 1000), lambda: S.uniform_512(60, 700, 1),
                                  lambda: S.batch_scene(400, 4097, 4000), lambda: S.batch_scene(20, 4000, 1)])
def test_tree_goes_on_where_the_block_stops(make, tile):
    """Trees that the block builds whole, stops at early, stops at late, and does
    not begin (more than 4,096 shapes)."""
    spec = G.default_spec(max_tile_size=tile)
    r = G.Rasterizer(spec)
    try:
        compare_binning(r, make(), spec)
    finally:
        r.close()


def test_the_last_level_is_not_given_up():
    """4,000 shapes on 400^2 in 64-px tiles come to 66,304 pairs in a block's hands,
    2,982 of them in the last level; 4,097 are built by the level launches alone.
    The ratio of the medians is about 1, and was 2 where the block gave up there
    and the launches began anew."""
    rs, times = [], []
    for n in (4000, 4097):
        r = G.Rasterizer(G.default_spec(max_tile_size=64))
        r.scene_upload_outlines(S.batch_scene(400, n, 4000))
        rs.append(r)
        times.append([])
    try:
        for k in range(25):
            for r, t in zip(rs, times):
                start = time.perf_counter()
                r.scene_bin()
                if k >= 5:
                    t.append(time.perf_counter() - start)
    finally:
        for r in rs:
            r.close()
    assert np.median(times[0]) <= 1.35 * np.median(times[1]), [np.median(t) for t in times]
