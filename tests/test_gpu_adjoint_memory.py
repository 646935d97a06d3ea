"""The adjoint's colour stream is sized by the work of its scenes: a small batch
does not hold a full chip's, and one whose work grows under an update has room."""
import dataclasses

import numpy as np
import pytest
import torch

import gudni_amd as G
from gudni_amd import scenes as S

pytestmark = pytest.mark.gpu


def target(scene):
    return np.random.default_rng(scene.width).uniform(0, 1, (scene.height, scene.width, 4)).astype(np.float32)


def test_a_small_batch_holds_a_small_stream():
    """A full chip's stream is 0.5 GB (256 KB for each of 2,048 wave slots)."""
    r = G.Rasterizer(G.default_spec(max_tile_size=16))
    try:
        scenes = [S.batch_scene(64, 10, 1, gradient_share=0), S.batch_scene(1024, 2000, 2, gradient_share=0)]
        warm = G.Adjoint(r, [(scenes[1], target(scenes[1]))])   # the context's own buffers
        used = []
        for scene in scenes:
            torch.cuda.synchronize()
            free = torch.cuda.mem_get_info()[0]
            a = G.Adjoint(r, [(scene, target(scene))])
            used.append(free - torch.cuda.mem_get_info()[0])
            a.close()
        warm.close()
    finally:
        r.close()
    assert used[0] <= used[1] - (400 << 20), used


@pytest.mark.parametrize("first,then", [(1, 40), (40, 1), (1, 8)])
def test_the_stream_follows_the_work(first, then):
    """Shapes gathered in a part of the canvas split its tiles: more work units
    than when they are spread (or fewer, the other way)."""
    scene = S.batch_scene(1024, 600, 3, gradient_share=0)
    offsets = scene.outline_pair_offsets
    centre = np.add.reduceat(scene.pairs[:, :2], offsets[:-1], axis=0) / np.diff(offsets)[:, None]
    centre = np.tile(np.repeat(centre, np.diff(offsets), axis=0), 2)
    def gathered(k):
        return (scene.pairs - centre + centre / np.float32(k) + np.float32(20)).astype(np.float32)
    spec = G.default_spec(max_tile_size=256)
    r = G.Rasterizer(spec)
    try:
        want_scene = dataclasses.replace(scene, pairs=gathered(then))
        a = G.Adjoint(r, [(want_scene, target(scene))])
        a.run()
        want = a.result(0, image=True)
        a.close()
        a = G.Adjoint(r, [(dataclasses.replace(scene, pairs=gathered(first)), target(scene))])
        a.run()
        a.update(0, pairs=gathered(then))
        a.run()
        got = a.result(0, image=True)
        a.close()
    finally:
        r.close()
    assert np.array_equal(got[3], want[3])
    assert abs(got[0] - want[0]) <= 1e-6 * want[0]
    for x, y in ((got[1], want[1]), (got[2], want[2])):
        np.testing.assert_allclose(x, y, rtol=1e-3, atol=1e-5 * np.abs(y).max())
