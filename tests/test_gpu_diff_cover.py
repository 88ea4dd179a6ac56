"""The 8x8 rasters leave out the entries whose square misses a tile: against tiles of 16x16, which step every entry.

Training images: a pixel stops by itself there, so whatever the tile shape it composites the same splats in the same
order with the same arithmetic, bit for bit.  Gradients of opacity and colour agree within 2e-3 between the forms
(each is held to 1e-3 of the 64-bit gradients); the shape's are left to the scenes of the other tests, since the forms
add a tile's pixels in different orders and a needle amplifies that rounding.
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


def config(tile, flags=0):
    c = _lib.RasterConfig()
    c.tile_w, c.tile_h, c.t_min, c.flags = tile, tile, 1.0 / 8192.0, flags
    return c


# (splats, log-scale, stretch): dust below a pixel; round; slanted needles over many tiles; needles wider than the
# view; one splat; lists around the batches of 32 and 64 whole-screen entries
@pytest.mark.parametrize("n,logscale,stretch", [(5000, -7.0, 0.0), (3000, -4.0, 0.5), (1500, -5.0, 3.5),
                                                (150, -3.0, 6.0), (1, -1.0, 2.0)]
                         + [(n, 1.0, 0.0) for n in (31, 32, 33, 63, 64, 65)])
@pytest.mark.parametrize("flags", [ALWAYS, NEVER])
def test_training_forms_leave_out_only_what_covers_nothing(n, logscale, stretch, flags):
    print("training cover", n, logscale, stretch, flags, flush=True)
    sc = S.gaussian_cloud(n, seed=n, pos_std=0.8, logscale=(logscale, 0.3))
    sc.rows[:, S.COL["scale_0"]] += stretch
    sc.rows[:, S.COL["opacity"]] = np.clip(sc.rows[:, S.COL["opacity"]], -6, 3)
    views = [(0, S.orbit_camera(203, 131, 4.0)), (0, S.orbit_camera(88, 64, 3.0, theta=0.7))]
    rng = np.random.default_rng(n)
    weights = [torch.tensor(rng.uniform(0.5, 1.5, (c.screen_size[1], c.screen_size[0], 4)), dtype=torch.float32,
                            device="cuda") for _, c in views]
    images, grads = [], []
    for cfg in (config(16), config(8, flags)):
        p = D.scene_tensors(sc)
        imgs = D.render_batch([p], views, config=cfg)
        sum((img * w).sum() for img, w in zip(imgs, weights)).backward()
        images.append([i.detach().cpu().numpy() for i in imgs])
        grads.append({k: p[k].grad.cpu().numpy() for k in ("opacity_logits", "sh")})
    for a, b in zip(*images):
        np.testing.assert_array_equal(a, b)
    for k, want in grads[0].items():
        assert np.linalg.norm(grads[1][k] - want) <= 2e-3 * np.linalg.norm(want), k


@pytest.mark.parametrize("flags", [ALWAYS, NEVER])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_non_finite_colour_stays_in_the_tiles_its_square_may_cover(flags, bad):
    """A slanted needle of NaN or infinite colour: its tiles are not finite, the tiles of its rectangle that its
    square misses (by more than a pixel) are the frame's without it."""
    print("non-finite colour", flags, bad, flush=True)
    w, h = 256, 192
    rng = np.random.default_rng(1)
    inst = np.zeros((40, 12), np.float32)
    inst[:, 0:2] = rng.uniform(-1, 1, (40, 2))
    inst[:, 2], inst[:, 4], inst[:, 7] = 0.5, 0.1, 0.1
    inst[:, 8:12] = rng.uniform(0.1, 0.6, (40, 4))
    long, thin = 0.25, 0.004
    inst[20, 0:2] = 0.0
    inst[20, 4:8] = long, long, -thin, thin  # along the diagonal
    inst[20, 8:11] = bad
    di = torch.zeros(12, dtype=torch.int32, device="cuda")
    di[8] = 40
    cfg = config(8, flags)
    img = P.draw(torch.tensor(inst, device="cuda"), di, w, h, cfg=cfg)[0].cpu().numpy()
    without = inst.copy()
    without[20, 11] = 0.0
    without[20, 8:11] = 0.0
    ref = P.draw(torch.tensor(without, device="cuda"), di, w, h, cfg=cfg)[0].cpu().numpy()
    m = np.linalg.inv(np.array([[long * w / 2, -thin * w / 2], [long * h / 2, thin * h / 2]]))
    y, x = np.mgrid[0:h, 0:w] + 0.5
    u = np.abs(np.einsum("ij,jhw->ihw", m, np.stack([x - w / 2, y - h / 2])))  # in standard deviations
    covered = (u < 2.99).all(0)
    assert covered.sum() > 500 and not np.isfinite(img[covered][:, :3]).any()
    ty, tx = np.mgrid[4:h:8, 4:w:8]
    mid = np.abs(np.einsum("ij,jhw->ihw", m, np.stack([tx - w / 2, ty - h / 2])))
    reach = 4.5 * np.abs(m).sum(1)[:, None, None]  # the tile's pixels and one more
    missed = (mid > 3.0 + reach).any(0).repeat(8, 0).repeat(8, 1)
    box = 3.0 * np.array([long + thin, long + thin]) * [w / 2, h / 2]  # its rectangle
    inside = (np.abs(x - w / 2) < box[0]) & (np.abs(y - h / 2) < box[1])
    assert (missed & inside).sum() > 5000
    np.testing.assert_array_equal(img[missed & inside], ref[missed & inside])
