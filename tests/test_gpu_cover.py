"""Records that cannot cover a tile are left out where two tiles share a wave: the results stay.

The tile lists hold every tile of a splat's rectangle; the pair rasters leave out the entries whose square misses
the tile's pixels.  A left-out entry changes no pixel, so the differentiable image and, with t_min = 0, the plain
one have the same bits as with one tile a wave (which steps every entry); with t_min > 0 the plain forms stop at
different entries and agree within 2 t_min.  Gradients: the same bits at every LDS batch depth; opacity's and
colour's 2e-3 relative between the two forms (each is held to 1e-3 of the 64-bit gradients).  The shape's are left
to the scenes of the other tests: the two forms add a lane's pixels in a different order, and a needle 400 times as
long as wide amplifies that rounding to 5%.
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

ALWAYS, NEVER = 4, 8


def scene_of(n, logscale, stretch, seed):
    """Splats of e^logscale with one axis e^stretch longer, at random angles."""
    sc = S.gaussian_cloud(n, seed=seed, pos_std=0.8, logscale=(logscale, 0.3))
    sc.rows[:, S.COL["scale_0"]] += stretch
    sc.rows[:, S.COL["opacity"]] = np.clip(sc.rows[:, S.COL["opacity"]], -6, 3)
    return sc


# (splats, log-scale, stretch): dust below a pixel; round; slanted needles over many tiles; needles wider than the
# view; one splat; lists of 31, 32 and 33 whole-screen entries, around a batch
CASES = [(5000, -7.0, 0.0), (3000, -4.0, 0.5), (1500, -5.0, 3.5), (150, -3.0, 6.0), (1, -1.0, 2.0), (31, 1.0, 0.0),
         (32, 1.0, 0.0), (33, 1.0, 0.0)]


def config(flags, lds_batch=0, t_min=1.0 / 8192.0):
    c = _lib.RasterConfig()
    c.tile_w, c.tile_h, c.t_min, c.flags, c.lds_batch = 8, 8, t_min, flags, lds_batch
    return c


@pytest.mark.parametrize("n,logscale,stretch", CASES)
def test_diff_pair_form_leaves_out_only_what_covers_nothing(n, logscale, stretch):
    print("diff cover", n, logscale, stretch, flush=True)
    sc = scene_of(n, logscale, stretch, n)
    views = [(0, S.orbit_camera(203, 131, 4.0)), (0, S.orbit_camera(88, 64, 3.0, theta=0.7))]
    rng = np.random.default_rng(n)
    weights = [torch.tensor(rng.uniform(0.5, 1.5, (c.screen_size[1], c.screen_size[0], 4)), dtype=torch.float32,
                            device="cuda") for _, c in views]
    images, grads = {}, {}
    for key in ((NEVER, 0), (ALWAYS, 0), (ALWAYS, 8), (ALWAYS, 16), (ALWAYS, 32)):
        p = D.scene_tensors(sc)
        imgs = D.render_batch([p], views, config=config(*key))
        sum((img * w).sum() for img, w in zip(imgs, weights)).backward()
        images[key] = [i.detach().cpu().numpy() for i in imgs]
        grads[key] = {k: p[k].grad.cpu().numpy() for k in D.PARAM_NAMES}
        for a, b in zip(images[(NEVER, 0)], images[key]):
            np.testing.assert_array_equal(a, b)
        for k in D.PARAM_NAMES:
            if key[0] == ALWAYS:
                np.testing.assert_array_equal(grads[(ALWAYS, 0)][k], grads[key][k], err_msg=k)
        for k in ("opacity_logits", "sh"):
            ref = np.linalg.norm(grads[(NEVER, 0)][k])
            assert np.linalg.norm(grads[key][k] - grads[(NEVER, 0)][k]) <= 2e-3 * ref, k


@pytest.mark.parametrize("n,logscale,stretch", CASES)
def test_plain_pair_form_leaves_out_only_what_covers_nothing(n, logscale, stretch):
    print("plain cover", n, logscale, stretch, flush=True)
    sc = scene_of(n, logscale, stretch, n)
    r = P.Renderer(n)
    r.load_buffer(sc.ply_buffer(), n)
    cam = S.orbit_camera(333, 201, 4.0)
    for t_min in (0.0, 1.0 / 8192.0):
        img = {}
        for flags in (NEVER, ALWAYS):
            r.set_config(config=config(flags, t_min=t_min))
            for _ in range(3):  # a frame whose lists outgrow the storage sizes it for the next one
                out = r.render(cam)
                if r.frame_info()[0] == 0:
                    break
            img[flags] = out.cpu().numpy()
        if t_min == 0.0:
            np.testing.assert_array_equal(img[NEVER], img[ALWAYS])
        else:
            assert np.abs(img[NEVER] - img[ALWAYS]).max() <= 2 * t_min * max(1.0, np.abs(img[NEVER]).max())


@pytest.mark.parametrize("n,logscale,stretch", CASES + [(64, 1.0, 0.0), (65, 1.0, 0.0)])
def test_plain_single_form_leaves_out_only_what_covers_nothing(n, logscale, stretch):
    """One 8x8 tile a wave (batches of 64) against 16x16 tiles, which step every entry of their lists: with t_min = 0
    each pixel composites the same splats in the same order with the same arithmetic, bit for bit."""
    print("single cover", n, logscale, stretch, flush=True)
    sc = scene_of(n, logscale, stretch, n)
    r = P.Renderer(n)
    r.load_buffer(sc.ply_buffer(), n)
    cam = S.orbit_camera(333, 201, 4.0)
    img = []
    for tile in (8, 16):
        cfg = config(NEVER, t_min=0.0)
        cfg.tile_w = cfg.tile_h = tile
        r.set_config(config=cfg)
        for _ in range(3):
            out = r.render(cam)
            if r.frame_info()[0] == 0:
                break
        img.append(out.cpu().numpy())
    r.close()
    np.testing.assert_array_equal(*img)
