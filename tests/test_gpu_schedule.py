"""Rasters whose waves are all resident take their tiles as they come, larger ones longest list first.

The order of the tiles changes no pixel: images and gradients have the same bits on both sides of the line (6144
waves, or 1024 under a cap of 4 waves a CU, which takes the other side), with one tile a wave.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)

from vkgs_amd import _lib  # noqa: E402
from vkgs_amd import diff as D  # noqa: E402
from vkgs_amd import pipeline as P  # noqa: E402
from vkgs_amd import scene as S  # noqa: E402

NEVER = 8


# 1, 6144 and 6240 tiles of 8x8; 1536 and 1584 of 16x16 (four waves each)
@pytest.mark.parametrize("tile,w,h,extra", [((8, 8), 8, 8, 0), ((8, 8), 768, 512, 0), ((8, 8), 777, 520, 0),
                                            ((8, 8), 768, 512, P.RASTER_TRIANGLES), ((16, 16), 768, 512, 0),
                                            ((16, 16), 777, 520, 0)])
def test_tile_order_changes_nothing(tile, w, h, extra):
    print("schedule", tile, w, h, extra, flush=True)
    sc = S.gaussian_cloud(3000, seed=w, pos_std=0.8, logscale=(-3.5, 0.5))
    cam = S.orbit_camera(w, h, 4.0)
    r = P.Renderer(sc.n)
    r.load_buffer(sc.ply_buffer(), sc.n)
    target = torch.rand(h, w, 4, device="cuda")
    images, grads = [], []
    for waves in (0, 4):
        cfg = _lib.RasterConfig()
        cfg.tile_w, cfg.tile_h, cfg.t_min, cfg.flags, cfg.waves_per_cu = *tile, 1.0 / 8192.0, NEVER | extra, waves
        r.set_config(config=cfg)
        for _ in range(3):  # a frame whose lists outgrow the storage sizes it for the next one
            out = r.render(cam)
            if r.frame_info()[0] == 0:
                break
        images.append(out.cpu().numpy())
        if tile == (8, 8) and not extra:
            p = D.scene_tensors(sc)
            img = D.render_batch([p], [(0, cam)], config=cfg)[0]
            (img * target).sum().backward()
            grads.append([img.detach().cpu().numpy()] + [p[k].grad.cpu().numpy() for k in D.PARAM_NAMES])
    r.close()
    np.testing.assert_array_equal(*images)
    for a, b in zip(*grads) if grads else ():
        np.testing.assert_array_equal(a, b)
