"""The backward's per-slot sums in a launch of their own and inside the projection backward give the same bits.

The sums' launch takes calls of up to 2^25 (view, splat) items; a call padded past that with a view of a large
scene that is not in view keeps them inside.  Runs of 1 to 16 pairs, 17 to 32 (two in a wave), 33 to 64 and
beyond are in the scene; the tolerance is none (the same additions in the same order).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)

from vkgs_amd import diff as D  # noqa: E402
from vkgs_amd import scene as S  # noqa: E402


def far_scene(n):
    """n splats behind every camera used here."""
    p = {"means": torch.zeros(n, 3), "log_scales": torch.zeros(n, 3), "quats": torch.zeros(n, 4),
         "opacity_logits": torch.zeros(n), "sh": torch.zeros(n, 48)}
    p = {k: v.cuda() for k, v in p.items()}
    p["means"][:] = torch.tensor([0.0, 1e4, 0.0])
    p["quats"][:, 0] = 1.0
    return {k: v.requires_grad_() for k, v in p.items()}


@pytest.mark.parametrize("n,views", [(1, 1), (27, 1), (28, 1), (29, 2), (4001, 1), (4001, 3)])
def test_sums_in_their_own_launch_match(n, views):
    print("slot sums", n, views, flush=True)
    sc = S.gaussian_cloud(n, seed=n, pos_std=0.8, logscale=(-4.0, 1.0))
    sc.rows[: max(1, n // 50), S.COL["scale_0"]:S.COL["scale_0"] + 3] += 2.5
    cams = [S.orbit_camera(200 + 16 * i, 150, 4.0, theta=0.3 + i) for i in range(views)]
    rng = np.random.default_rng(n)
    grads = []
    for padded in (False, True):
        p = D.scene_tensors(sc)
        scenes, vs = [p], [(0, c) for c in cams]
        if padded:
            scenes.append(far_scene((1 << 25) // 8 + 1))
            vs += [(1, S.orbit_camera(8, 8, 4.0)) for _ in range(8)]
        imgs = D.render_batch(scenes, vs)
        w = [torch.from_numpy(rng.random(i.shape, dtype=np.float32)).cuda() for i in imgs[:views]] if not grads else w
        sum((i * k).sum() for i, k in zip(imgs, w)).backward()
        grads.append({k: p[k].grad.cpu().numpy() for k in D.PARAM_NAMES})
    for k in D.PARAM_NAMES:
        assert np.abs(grads[0][k]).max() > 0
        np.testing.assert_array_equal(grads[0][k], grads[1][k], err_msg=k)
