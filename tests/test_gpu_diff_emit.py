"""Training views of large splats, whose pairs the emit numbers across a wave and, past 2048 pairs a wave, queues as
segments.

Gradients against the float64 restatement with the bars of the other scenes (images: all but a handful of
coverage-edge pixels within 1e-4; gradients 1e-3 relative per parameter group), and, in a grid whose rectangles take
more than 32 bits, the plain renderer's image.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)

import oracle  # noqa: E402
from oracle import torch_ref  # noqa: E402
from vkgs_amd import diff as D  # noqa: E402
from vkgs_amd import pipeline as P  # noqa: E402
from vkgs_amd import scene as S  # noqa: E402

NAMES = D.PARAM_NAMES


def large_scene(n, seed, logscale, spread):
    sc = S.gaussian_cloud(n, seed=seed, pos_std=0.7, logscale=(logscale, spread))
    c = S.COL
    sc.rows[:, c["opacity"]] = np.clip(sc.rows[:, c["opacity"]] - 3.5, -6, -1.5)
    sc.rows[:, c["f_dc_0"]:c["f_rest_0"] + 45] = sc.rows[:, c["f_dc_0"]:c["f_rest_0"] + 45].astype(np.float16)
    return sc


# tiles a splat: about 170 (one segment), 625 (two), and a mix from one tile to the whole view
@pytest.mark.parametrize("n,size,logscale,spread", [(130, 104, 0.6, 0.1), (70, 200, 0.6, 0.1), (150, 160, -1.5, 1.0)])
def test_large_splats_gradients_match_float64(n, size, logscale, spread):
    print("large training splats", n, size, logscale, flush=True)
    sc, cam = large_scene(n, n, logscale, spread), S.orbit_camera(size, size, 4.0)
    pos = oracle.parse_ply(sc.rows, S.standard_offsets())[0]
    _, key, index = oracle.rank(cam, pos)
    order = oracle.sort_kv(key, index)[1].astype(np.int64)
    proj, view, eye = S.camera_arrays(cam)
    cam64 = [torch.tensor(proj.reshape(4, 4).T, dtype=torch.float64),
             torch.tensor(view.reshape(4, 4).T, dtype=torch.float64), torch.tensor(eye, dtype=torch.float64)]
    p64 = [torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, requires_grad=True)
           for a in (sc.means(), sc.log_scales(), sc.quats_wxyz(), sc.opacity_logits(), sc.sh_channel_major())]
    w = np.random.default_rng(n).uniform(0.5, 1.5, (size, size, 4))
    ref = torch_ref.render(*p64, *cam64, size, size, order)
    (ref * torch.tensor(w)).sum().backward()
    p = D.scene_tensors(sc)
    img = D.render(**p, camera=cam, t_min=0.0)
    (img * torch.tensor(w, dtype=torch.float32, device="cuda")).sum().backward()
    assert D.last_info["pairs"] > 64 * n
    d = np.abs(img.detach().cpu().numpy() - ref.detach().numpy()).max(-1)
    assert (d > 1e-4).mean() < 0.005 and d.max() < 0.02
    for name, t64 in zip(NAMES, p64):
        g, want = p[name].grad.cpu().double(), t64.grad
        assert float(torch.linalg.norm(g - want) / torch.linalg.norm(want)) <= 1e-3, name


def test_large_splats_in_a_wide_grid_match_the_plain_renderer():
    w, h, n = 4104, 1032, 40  # 513 x 129 tiles: 36 rectangle bits
    print("wide training view", w, h, flush=True)
    sc, cam = large_scene(n, 5, 0.8, 0.3), S.orbit_camera(w, h, 4.0)
    r = P.Renderer(n)
    r.load_buffer(sc.ply_buffer(), n)
    r.set_config(8, 8, 0.0)
    for _ in range(3):  # a frame whose lists outgrow the storage sizes it for the next one
        plain = r.render(cam)
        if r.frame_info()[0] == 0:
            break
    plain = plain.cpu().numpy()
    r.close()
    p = D.scene_tensors(sc, requires_grad=False)
    img = D.render(**p, camera=cam, t_min=0.0).cpu().numpy()
    d = np.abs(img - plain).max(-1)
    assert (d > 1e-5).mean() < 0.005 and d.max() < 0.02
