"""A timed render counts every work unit once, however many waves run it."""
import dataclasses

import pytest
import torch

import gudni_amd as G
from gudni_amd import scenes as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,shapes,tile", [(64, 64, 12, 256), (8, 8, 1, 8), (512, 300, 100, 64),
                                                      (512, 512, 300, 32), (1024, 1024, 40, 8)])
def test_units_counted_once(width, height, shapes, tile):
    r = G.Rasterizer(G.default_spec(max_tile_size=tile))
    try:
        scene = dataclasses.replace(S.batch_scene(max(width, height), shapes, 5), width=width, height=height)
        out = torch.zeros(width * height, dtype=torch.int32, device="cuda")
        r.scene_upload_outlines(scene)
        r.scene_bin()
        r.enable_timing()
        r.frame_render(out.data_ptr())
        r.frame_check()
        assert int(r.last_stage_cycles()[3]) == r.scene_counts()[2]
    finally:
        r.close()
