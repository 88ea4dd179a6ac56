"""A frame whose (tile, splat) pairs outgrow their storage keeps the first max_pairs of the draw order, each splat's
in row-major tile order, and drops the rest: the lists are the oracle's cut there, every list position is written,
and two draws give the same image.

Whole-number lists, so equality is exact.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)

import ctypes as C  # noqa: E402

import oracle  # noqa: E402
from vkgs_amd import _lib  # noqa: E402
from vkgs_amd import pipeline as P  # noqa: E402
from vkgs_amd import scene as S  # noqa: E402

OVERFLOW = 6


def instances(n, sigma, spread, seed):
    """n splats of about sigma (of the frame's half width) anywhere in the frame, some outside it."""
    rng = np.random.default_rng(seed)
    inst = np.zeros((n, 12), np.float32)
    inst[:, 0:2] = rng.uniform(-1.2, 1.2, (n, 2))
    inst[:, 2] = 0.5
    s = sigma * np.exp(spread * rng.standard_normal((n, 2)))
    a = rng.uniform(0, 2 * np.pi, n)
    inst[:, 4], inst[:, 5] = s[:, 0] * np.cos(a), s[:, 0] * np.sin(a)
    inst[:, 6], inst[:, 7] = -s[:, 1] * np.sin(a), s[:, 1] * np.cos(a)
    inst[:, 8:11] = rng.uniform(0, 1, (n, 3))
    inst[:, 11] = rng.uniform(0.02, 0.6, n)
    return inst


def cut_lists(ranges, lst, room):
    """The lists of the first `room` pairs, pairs numbered by splat and then by tile."""
    ranges = np.asarray(ranges).astype(np.int64)
    tile = np.repeat(np.arange(len(ranges)), ranges[:, 1] - ranges[:, 0])
    keep = np.zeros(lst.size, bool)
    keep[np.lexsort((tile, lst))[:room]] = True
    count = np.bincount(tile[keep], minlength=len(ranges))
    end = np.cumsum(count)
    out = np.stack([end - count, end], 1)
    out[count == 0] = 0
    return out, lst[keep]


def whole_pairs(inst, w, h, tw, th):
    """Pairs of each splat, in draw order."""
    ranges, lst = oracle.bin_tiles(inst, w, h, tw, th)
    return ranges, lst, np.bincount(lst, minlength=len(inst))


def config(tw, th):
    cfg = _lib.default_raster_config()
    cfg.tile_w, cfg.tile_h = tw, th
    return cfg


def draw_short(inst, w, h, cfg, room):
    """(image, status, ranges, the list's `room` words) of a draw with room for that many pairs."""
    di = torch.zeros(12, dtype=torch.int32, device="cuda")
    di[8] = len(inst)
    img, ds = P.draw(torch.tensor(inst, device="cuda"), di, w, h, cfg=cfg, max_pairs=room)
    rp, lp, tx, ty = C.c_void_p(), C.c_void_p(), C.c_uint32(), C.c_uint32()
    _lib.check(_lib.lib().vkgs_draw_lists(P.ptr(ds.buf), ds.nbytes, C.byref(rp), C.byref(lp), C.byref(tx),
                                          C.byref(ty)), "vkgs_draw_lists")
    ranges = P._download_u32(rp.value, 2 * tx.value * ty.value).reshape(-1, 2).astype(np.int64)
    return img.cpu().numpy(), ds.status(), ranges, P._download_u32(lp.value, room)


# (splats, sigma, spread, size, tile): one chunk of splats; several; more than 256 chunks (whose rows a scan sums);
# 2, 5 x 4 and 510 supertiles, one of 64 x 4 tiles; and grids that the two-level binning refuses (528 supertiles; 129
# columns and rows), whose pairs are emitted and sorted: splats of up to 8 tiles, of some, and of thousands, which a
# wave with more than 2048 pairs queues as segments
@pytest.mark.parametrize("n,sigma,spread,w,h,tw,th", [
    (400, 0.2, 0.6, 640, 480, 8, 8),
    (20_000, 0.02, 0.8, 640, 480, 8, 8),
    (300, 0.5, 0.3, 200, 120, 8, 8),
    (9_000, 0.05, 1.0, 777, 555, 16, 16),
    (3_000, 0.3, 0.5, 1000, 60, 64, 4),
    (2_000, 0.03, 0.8, 3839, 2159, 8, 8),
    (700_000, 0.004, 0.6, 640, 480, 8, 8),
    (60, 0.3, 0.3, 4104, 2048, 8, 8),
    (5_000, 0.006, 1.3, 4104, 2048, 8, 8),
    (300, 0.3, 0.3, 16384, 128, 8, 8),
    (5_000, 0.01, 1.3, 16384, 128, 8, 8),
])
def test_short_storage_keeps_the_first_pairs_of_the_draw_order(n, sigma, spread, w, h, tw, th):
    inst = instances(n, sigma, spread, n)
    ranges, lst, per = whole_pairs(inst, w, h, tw, th)
    k, ends = lst.size, np.cumsum(per)
    some = int(np.searchsorted(ends, k // 3))
    # half; all but one; whole splats exactly; one pair more; and inside the largest splat of the last two thirds
    big = int(np.argmax(np.where(ends - per > k // 3, per, 0)))
    rooms = [k, k // 2, k - 1, int(ends[some]), int(ends[some]) + 1, int(ends[big] - per[big] + per[big] // 2 + 1)]
    for room in rooms:
        print("short draw", n, w, h, tw, th, "pairs", k, "room", room, flush=True)
        want_ranges, want = cut_lists(ranges, lst, room)
        images = []
        for _ in range(2):
            img, status, got_ranges, got = draw_short(inst, w, h, config(tw, th), room)
            assert status == (OVERFLOW if room < k else 0, k)
            np.testing.assert_array_equal(got, want)
            np.testing.assert_array_equal(got_ranges, want_ranges)
            images.append(img)
        np.testing.assert_array_equal(*images)


# whole-frame splats, the renderer's own first storage (4 pairs a splat and 2^20); rectangles of 30 bits and of more
# than 32; the same in grids that the two-level binning refuses
@pytest.mark.parametrize("n,w,h", [(200, 1600, 900), (40, 4096, 2048), (900, 16384, 128), (40, 4104, 2048)])
def test_renderers_first_frame_of_large_splats(n, w, h):
    print("first frame", n, w, h, flush=True)
    sc = S.gaussian_cloud(n, seed=n, pos_std=0.5, logscale=(2.0, 0.2))
    cam = S.orbit_camera(w, h, 6.0)
    st = P.parse_ply(sc.ply_buffer(), sc.n)
    stage = P.reference_frame(cam, st, w, h)
    v = int(P.u32(stage["count"])[0])
    ranges, lst, _ = whole_pairs(stage["instances"].cpu().numpy()[:v], w, h, 8, 8)
    room = 4 * n + (1 << 20)
    assert lst.size > room
    want_ranges, want = cut_lists(ranges, lst, room)
    r = P.Renderer(n)
    r.load_buffer(sc.ply_buffer(), n)
    first = r.render(cam).cpu().numpy()
    rp, lp, tx, ty = C.c_void_p(), C.c_void_p(), C.c_uint32(), C.c_uint32()
    _lib.check(_lib.lib().vkgs_renderer_tile_lists(r._h, C.byref(rp), C.byref(lp), C.byref(tx), C.byref(ty)), "lists")
    got_ranges = P._download_u32(rp.value, 2 * len(ranges)).reshape(-1, 2).astype(np.int64)
    np.testing.assert_array_equal(got_ranges, want_ranges)
    np.testing.assert_array_equal(P._download_u32(lp.value, room), P.u32(stage["index"])[:v][want])
    np.testing.assert_array_equal(r.render(cam).cpu().numpy(), first)
    assert r.frame_info() == (OVERFLOW, v, lst.size)
    r.render(cam)  # with room for the whole list
    assert r.frame_info() == (0, v, lst.size)
    got_ranges, got = r.tile_lists()
    full = np.asarray(ranges).astype(np.int64)
    full[full[:, 0] == full[:, 1]] = 0
    np.testing.assert_array_equal(got_ranges, full)
    np.testing.assert_array_equal(got, P.u32(stage["index"])[:v][lst])
    r.close()


def test_pair_total_past_32_bits_is_flagged():
    """32,776 whole-frame splats of 131,072 tiles are 2^32 + 2^20 pairs: the total's low 32 bits would fit."""
    n, w, h, tiles, room = (1 << 15) + 8, 4096, 2048, 1 << 17, (1 << 21) + 77
    print("past 32 bits", n, w, h, "room", room, flush=True)
    inst = np.zeros((n, 12), np.float32)
    inst[:, 2], inst[:, 4], inst[:, 7], inst[:, 11] = 0.5, 10.0, 10.0, 0.01
    _, status, ranges, lst = draw_short(inst, w, h, config(8, 8), room)
    assert status == (OVERFLOW, (n * tiles) & 0xffffffff)
    # splats 0-15 in every tile, 16 in the first 77
    count = np.where(np.arange(tiles) < room - 16 * tiles, 17, 16)
    end = np.cumsum(count)
    np.testing.assert_array_equal(ranges, np.stack([end - count, end], 1))
    np.testing.assert_array_equal(lst, np.arange(room) - np.repeat(end - count, count))
