"""Triangle coverage with two tiles a wave: the image of one tile a wave.

Coverage is decided by the same integers in both forms and a tile stops after the same entry, so the images have
the same bits.  Quads with edges beyond 32768 pixels form their weights from 64-bit integers where the one-tile
form adds doubles: a rounding of 2^-53, at most one of alpha's 2^-24 steps, 1e-6 of the image.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)

from vkgs_amd import _lib  # noqa: E402
from vkgs_amd import pipeline as P  # noqa: E402
from vkgs_amd import scene as S  # noqa: E402

ALWAYS, NEVER = 4, 8


# (splats, log-scale, stretch of one axis): dust; round; slanted needles; one splat; lists around a batch of 32;
# quads of 10^4 and 10^5 pixels, on both sides of the edge limit; some past the million pixels that are drawn
@pytest.mark.parametrize("n,logscale,stretch", [
    (5000, -7.0, 0.0), (3000, -4.0, 0.5), (1500, -5.0, 3.5), (1, -1.0, 2.0), (31, 1.0, 0.0), (32, 1.0, 0.0),
    (33, 1.0, 0.0), (40, 3.0, 0.5), (40, 5.0, 0.5), (40, -2.0, 8.0), (60, 8.0, 0.0)])
@pytest.mark.parametrize("t_min", [0.0, 1.0 / 8192.0])
def test_two_tiles_a_wave_give_the_same_image(n, logscale, stretch, t_min):
    print("triangle pairs", n, logscale, stretch, t_min, flush=True)
    sc = S.gaussian_cloud(n, seed=n, pos_std=0.8, logscale=(logscale, 0.3))
    sc.rows[:, S.COL["scale_0"]] += stretch
    r = P.Renderer(n)
    r.load_buffer(sc.ply_buffer(), n)
    for w, h in ((333, 201), (8, 8), (1021, 37)):
        cam = S.orbit_camera(w, h, 4.0)
        img = {}
        for flags in (NEVER, ALWAYS):
            cfg = _lib.RasterConfig()
            cfg.tile_w, cfg.tile_h, cfg.t_min, cfg.flags = 8, 8, t_min, flags | P.RASTER_TRIANGLES
            r.set_config(config=cfg)
            for _ in range(3):  # a frame whose lists outgrow the storage sizes it for the next one
                out = r.render(cam)
                if r.frame_info()[0] == 0:
                    break
            img[flags] = out.cpu().numpy()
        if logscale + stretch < 3.0:
            np.testing.assert_array_equal(img[NEVER], img[ALWAYS])
        else:
            assert np.abs(img[NEVER] - img[ALWAYS]).max() <= 1e-6 * max(1.0, np.abs(img[NEVER]).max())
    r.close()
