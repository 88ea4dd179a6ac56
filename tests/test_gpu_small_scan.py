"""Scans at the sizes up to which one workgroup does them (8192 packed rectangles, 24,576 words), and above.

Splats behind the camera change nothing, so a training pass padded with them to sizes on both sides of the lines
has the same image and gradients bit for bit; the stage path's rank, whose scan has a word per 256 splats, is
compared with the oracle's.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)

import oracle  # noqa: E402
from vkgs_amd import diff as D  # noqa: E402
from vkgs_amd import pipeline as P  # noqa: E402
from vkgs_amd import scene as S  # noqa: E402


def padded(n, total):
    sc = S.gaussian_cloud(n, seed=3, pos_std=0.8, logscale=(-3.5, 0.5))
    rows = np.zeros((total, sc.rows.shape[1]), np.float32)
    rows[:n] = sc.rows
    rows[n:, S.COL["rot_0"]] = 1.0
    rows[n:, 1] = 1e4  # never in view
    sc.rows = rows
    return sc


def grads_of(total, cam, target):
    p = D.scene_tensors(padded(7000, total))
    img = D.render_batch([p], [(0, cam)])[0]
    (img * target).sum().backward()
    return img.detach().cpu().numpy(), {k: p[k].grad[:7000].cpu().numpy() for k in D.PARAM_NAMES}


# capacities in items are multiples of 256: up to 8192, above it, up to 24,576, above it
@pytest.mark.parametrize("total", [8192, 8193, 24_576, 24_577, 60_000])
def test_padding_changes_nothing(total):
    print("small scan", total, flush=True)
    cam = S.orbit_camera(200, 152, 4.0)
    target = torch.from_numpy(np.random.default_rng(1).random((152, 200, 4), dtype=np.float32)).cuda()
    img, g = grads_of(7000, cam, target)
    img2, g2 = grads_of(total, cam, target)
    np.testing.assert_array_equal(img, img2)
    for k in D.PARAM_NAMES:
        np.testing.assert_array_equal(g[k], g2[k], err_msg=k)


@pytest.mark.parametrize("n", [1, 256, 257, 8192 * 256, 8192 * 256 + 1])
def test_rank_counts(n):
    print("rank scan", n, flush=True)
    rng = np.random.default_rng(n)
    sc = padded(min(n, 7000), n)
    sc.rows[:, 0:3] = rng.normal(0.0, 3.0, (n, 3))
    st = P.parse_ply(sc.ply_buffer(), n)
    cam = S.orbit_camera(200, 152, 4.0)
    count, key, index = P.rank(cam, st)
    v, okey, oindex = oracle.rank(cam, np.ascontiguousarray(sc.rows[:, 0:3]))
    assert P.u32(count)[0] == v
    np.testing.assert_array_equal(P.u32(key)[:v], okey)
    np.testing.assert_array_equal(P.u32(index)[:v], oindex)
