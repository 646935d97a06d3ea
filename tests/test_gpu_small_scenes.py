"""Trees of small scenes are built by one block, others by a launch a step:
both sides of the line, and a scene that outgrows the block's pairs between
small ones of the same context, equal the host build byte for byte."""
import pytest

import gudni_amd as G
from gudni_amd import scenes as S
from tests.test_gpu_binning import compare_binning

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [8, 16, 64, 256])
def test_block_and_launch_builds(tile):
    spec = G.default_spec(max_tile_size=tile)
    r = G.Rasterizer(spec)
    try:
        for scene in (S.build_scene(9, 5, [], [[0, 0, 0, 1]], name="empty"), S.batch_scene(250, 120, 3),
                      S.uniform_512(400, 256, 9),      # large shapes: past the block's pairs
                      S.batch_scene(250, 120, 4), S.batch_scene(64, 1, 5), S.batch_scene(512, 4096, 6),
                      S.batch_scene(512, 4200, 7), S.batch_scene(300, 1024, 8), S.uniform_512(125, 300, 2)):
            compare_binning(r, scene, spec)
    finally:
        r.close()
