"""The plain rasters' exit test with opacities above 1.

A tile is done once all its pixels are below t_min, tested after every 4 entries of its list.  An instance drawn
with an opacity above 1 makes a pixel's transmittance negative and the next such one positive again, so where
that test falls decides the image: a tile whose pixels all end a group of 4 below t_min composites nothing more.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)

from vkgs_amd import _lib  # noqa: E402
from vkgs_amd import pipeline as P  # noqa: E402

ALWAYS, NEVER = 4, 8
T_MIN = 1.0 / 8192.0


def expected(opacity, colour):
    """One pixel under whole-frame splats, nearest first, in 64 bits."""
    t, out = 1.0, np.zeros(4)
    for i in range(0, len(opacity), 4):
        for o, c in zip(opacity[i:i + 4], colour[i:i + 4]):
            out += np.array([*c, o]) * t * o
            t -= t * o
        if t < T_MIN:
            break
    out[3] += t
    return out


# nearest first: below 0 after the first group of 4, above it again in the second; after the second, with the third
# in the same batch or (64 entries before them) past it; below 0 inside a group and above it at the group's end;
# opacities that keep the transmittance in range
@pytest.mark.parametrize("flags", [ALWAYS, NEVER])
@pytest.mark.parametrize("opacity", [
    [1.5, 0.1, 0.1, 0.1, 1.5, 0.1, 0.1, 0.1, 0.2],
    [0.1, 0.1, 0.1, 0.1, 0.1, 1.25, 0.1, 0.1, 1.5, 0.1, 0.1],
    [0.01] * 66 + [1.5, 0.1, 1.5, 0.1, 0.2],
    [0.01] * 64 + [1.5, 0.1, 0.1, 0.1, 1.5, 0.1, 0.2, 0.3],
    [1.5, 1.5, 0.1, 0.1, 0.3, 0.2, 1.0, 0.5],
    [0.1, 0.2, 0.3, 0.4, 0.5],
])
def test_a_tile_stops_where_every_group_of_four_is_tested(opacity, flags):
    n, w, h = len(opacity), 24, 24
    print("exit", n, flags, flush=True)
    rng = np.random.default_rng(n)
    inst = np.zeros((n, 12), np.float32)  # drawn last to first: the last instance is nearest
    inst[:, 2], inst[:, 4], inst[:, 7] = 0.5, 4000.0, 4000.0
    inst[::-1, 11] = opacity
    inst[:, 8:11] = rng.uniform(0, 1, (n, 3))
    cfg = _lib.RasterConfig()
    cfg.tile_w, cfg.tile_h, cfg.t_min, cfg.flags = 8, 8, T_MIN, flags
    di = torch.zeros(12, dtype=torch.int32, device="cuda")
    di[8] = n
    img, ds = P.draw(torch.tensor(inst, device="cuda"), di, w, h, cfg=cfg)
    assert ds.status() == (0, 9 * n)
    want = expected(inst[::-1, 11].astype(np.float64), inst[::-1, 8:11].astype(np.float64))
    # the falloff across the frame is below 1e-7; n steps of at most 1.5 in 32 bits, each a rounding or two
    np.testing.assert_allclose(img.cpu().numpy(), np.broadcast_to(want, (h, w, 4)), rtol=0, atol=n * 1e-6)
