"""How many waves run a work unit does not depend on what lies beside the canvas:
bars that reach far below it are held by the tile tree's nodes there, which have
no work units, and give the same frame in the same time as bars that end there."""
import time

import numpy as np
import pytest
import torch

import gudni_amd as G
from gudni_amd import scenes as S

pytestmark = pytest.mark.gpu


def bars(width, height, n, end):
    rng = np.random.default_rng(n)
    x = np.round(4 * rng.uniform(-32, width - 32, n)) / 4
    shapes = [(S.solid_tag(i), [S.rectangle_pairs(x[i], -5.0, x[i] + 64.0, end)]) for i in range(n)]
    return S.build_scene(width, height, shapes, rng.uniform(0, 1, (n, 4)).astype(np.float32), name="bars")


@pytest.mark.parametrize("upload", ["device", "host"])
@pytest.mark.parametrize("width,height,n,tile", [(4000, 37, 1200, 32), (2000, 20, 600, 32), (1000, 30, 300, 32),
                                                 (4000, 37, 1200, 64)])
def test_shapes_beside_the_canvas(width, height, n, tile, upload):
    """Medians of 15 renders in turn; 1.25 times allows for noise (the frames took
    1.5 to 4 times as long where the tiles beside the canvas were counted)."""
    spec = G.default_spec(max_tile_size=tile)
    frames, times, rasterizers = [], [], []
    for end in (height + 3.0, float(width)):
        scene = bars(width, height, n, end)
        r = G.Rasterizer(spec)
        r.set_stream(torch.cuda.current_stream().cuda_stream)
        if upload == "device":
            r.scene_upload_outlines(scene)
            r.scene_bin()
        else:
            _, geometry, jobs = G.prepare(scene, spec)
            r.upload_common(geometry.geo, scene)
            r.frame_upload(jobs, scene)
        rasterizers.append(r)
        frames.append(torch.zeros(width * height, dtype=torch.int32, device="cuda"))
        times.append([])
    try:
        for k in range(18):
            for r, out, t in zip(rasterizers, frames, times):
                torch.cuda.synchronize()
                start = time.perf_counter()
                r.frame_render(out.data_ptr())
                torch.cuda.synchronize()
                if k >= 3:
                    t.append(time.perf_counter() - start)
        for r in rasterizers:
            r.frame_check()
    finally:
        for r in rasterizers:
            r.close()
    assert torch.equal(frames[0], frames[1])
    assert np.median(times[1]) <= 1.25 * np.median(times[0]), [np.median(t) for t in times]
