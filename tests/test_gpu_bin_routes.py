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
