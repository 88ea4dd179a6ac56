"""Binning with large splats: pairs written by whole waves and, past kQueueWave pairs a wave, by queued segments.

The tile lists are integers: bit-exact against the CPU oracle's, in the renderer's packed and unpacked
(more than 32 rectangle bits) forms and in the draw stage, with pair storage that the first frame outgrows.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)

import oracle  # noqa: E402
from vkgs_amd import pipeline as P  # noqa: E402
from vkgs_amd import scene as S  # noqa: E402


def canonical(ranges):
    r = np.asarray(ranges).astype(np.int64)
    r[r[:, 1] == r[:, 0]] = 0
    return r


# (splats, log-scale, its spread, size): all small; 9-64 tiles; 65-512 (one segment); beyond 512 and
# whole-screen splats (several segments, up to 64 per splat); one splat, one pixel row of tiles
@pytest.mark.parametrize("n,logscale,spread,w,h", [
    (3000, -5.0, 0.3, 333, 201),
    (5000, -3.2, 0.3, 640, 480),
    (900, -1.6, 0.5, 1283, 721),
    (70, 1.5, 1.0, 1600, 900),
    (64, 2.0, 0.1, 2560, 1600),
    (1, 2.0, 0.0, 4096, 8),
])
def test_tile_lists_with_large_splats(n, logscale, spread, w, h):
    print("large splats", n, logscale, w, h, flush=True)
    sc = S.gaussian_cloud(n, seed=n, pos_std=1.0, logscale=(logscale, spread))
    cam = S.orbit_camera(w, h, 6.0)
    st = P.parse_ply(sc.ply_buffer(), sc.n)
    r = P.Renderer(n)
    r.load_buffer(sc.ply_buffer(), n)
    for _ in range(3):  # a frame whose lists outgrow the storage sizes it for the next one
        img = r.render(cam)
        status, v, k = r.frame_info()
        if status == 0:
            break
    assert status == 0 and v > 0 and k > 0
    ranges, lists = r.tile_lists()
    stage = P.reference_frame(cam, st, w, h)
    img2, ds = P.draw(stage["instances"], stage["draw_indirect"], w, h, max_pairs=k)
    assert ds.status() == (0, k)
    sranges, slist = ds.lists()
    inst = stage["instances"].cpu().numpy()[:v]
    oranges, olist = oracle.bin_tiles(inst, w, h, 8, 8)
    np.testing.assert_array_equal(sranges, canonical(oranges))
    np.testing.assert_array_equal(slist, olist)
    np.testing.assert_array_equal(ranges, canonical(oranges))
    np.testing.assert_array_equal(lists, P.u32(stage["index"])[:v][slist])
    np.testing.assert_array_equal(img.cpu().numpy(), img2.cpu().numpy())
    # too little room for the pairs: flagged, every list position written
    _, short = P.draw(stage["instances"], stage["draw_indirect"], w, h, max_pairs=max(1, k // 2))
    assert short.status() == (6, k)
    r.close()


# the two-level binning takes grids of at most 512 supertiles of 16 x 16 tiles and 128 columns and rows, with
# rows for twice as many counts; the pair sort takes the others.  Mixed sizes: most splats small, some of
# every size up to the whole frame.
@pytest.mark.parametrize("w,h,tw,th", [
    (1, 1, 8, 8),
    (128, 128, 8, 8),        # one supertile exactly
    (129, 127, 8, 8),
    (1000, 40, 64, 4),
    (777, 555, 16, 8),
    (4096, 2048, 8, 8),      # 512 supertiles
    (4104, 2048, 8, 8),      # 528: the pair sort
    (14336, 128, 8, 8),      # 112 columns
    (16384, 128, 8, 8),      # 128 columns and one row: the pair sort
    (2560, 1600, 16, 16),
])
@pytest.mark.parametrize("n", [700, 30_000])
def test_tile_lists_over_grids(w, h, tw, th, n):
    print("grid", w, h, tw, th, n, flush=True)
    from vkgs_amd import _lib
    sc = S.gaussian_cloud(n, seed=n + w, pos_std=1.0, logscale=(-5.0, 0.4))
    few = np.random.default_rng(w).integers(0, n, 60)
    sc.rows[few, S.COL["scale_0"]:S.COL["scale_0"] + 3] += np.linspace(0.0, 5.0, 60)[:, None].astype(np.float32)
    cam = S.orbit_camera(w, h, 5.0)
    st = P.parse_ply(sc.ply_buffer(), sc.n)
    count, key, index = P.rank(cam, st)
    P.sort_kv(count, key, index, 30)
    inst, di = P.projection(cam, st, P.inverse_index(count, index, n), count)
    v = int(P.u32(count)[0])
    host = inst.cpu().numpy()[:v]
    oranges, olist = oracle.bin_tiles(host, w, h, tw, th)
    k = olist.size
    cfg = _lib.default_raster_config()
    cfg.tile_w, cfg.tile_h = tw, th
    imgs = []
    for room in (max(k, 1), max(k, 1) + 3_000_000):  # exact room may be too little for the count rows: the pair sort
        img, ds = P.draw(inst, di, w, h, cfg=cfg, max_pairs=room)
        assert ds.status() == (0, k)
        ranges, lst = ds.lists()
        np.testing.assert_array_equal(ranges, canonical(oranges))
        np.testing.assert_array_equal(lst, olist)
        imgs.append(img.cpu().numpy())
    np.testing.assert_array_equal(imgs[0], imgs[1])
    r = P.Renderer(n)
    r.load_buffer(sc.ply_buffer(), n)
    r.set_config(tw, th)
    for _ in range(3):
        r.render(cam)
        if r.frame_info()[0] == 0:
            break
    ranges, lists = r.tile_lists()
    np.testing.assert_array_equal(ranges, canonical(oranges))
    np.testing.assert_array_equal(lists, P.u32(index)[:v][olist])
    r.close()
