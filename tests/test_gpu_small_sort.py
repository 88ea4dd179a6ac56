"""Sorts of up to 8192 pairs, which one workgroup does in one kernel, and the passes just above.

Integers: bit-exact against numpy's stable argsort on the sorted bits; bits above them stay with their pair.  The
depth order of small scenes (64-bit and 32-bit values, in place and from the alternate buffers) is the stable
order of its keys.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)

from vkgs_amd import pipeline as P  # noqa: E402
from vkgs_amd import scene as S  # noqa: E402


# (capacity, live count): none; one; around a wave, a round of 1024 and the limit; few of many; above the limit
@pytest.mark.parametrize("capacity,count", [(5, 0), (1, 1), (65, 64), (65, 65), (1024, 1024), (1025, 1025),
                                            (8192, 1023), (8191, 8191), (8192, 8192), (8193, 8193)])
@pytest.mark.parametrize("bits", [1, 9, 10, 25, 30, 32])
def test_small_sorts(capacity, count, bits):
    print("small sort", capacity, count, bits, flush=True)
    rng = np.random.default_rng(capacity * 64 + bits)
    key = rng.integers(0, 1 << 32, capacity, dtype=np.uint64).astype(np.uint32)
    key[: capacity // 3] &= np.uint32(0x00FF0F03)  # crowded digits
    key[capacity // 3: capacity // 2] = 0xFFFFFFFF
    value = rng.permutation(capacity).astype(np.uint32)
    k = torch.from_numpy(key.view(np.int32)).cuda()
    v = torch.from_numpy(value.view(np.int32)).cuda()
    P.sort_kv(torch.tensor([count], dtype=torch.int32, device="cuda"), k, v, bits)
    order = np.argsort(key[:count].astype(np.uint64) & ((1 << bits) - 1), kind="stable")
    np.testing.assert_array_equal(P.u32(k)[:count], key[:count][order])
    np.testing.assert_array_equal(P.u32(v)[:count], value[:count][order])
    np.testing.assert_array_equal(P.u32(k)[count:], key[count:])
    np.testing.assert_array_equal(P.u32(v)[count:], value[count:])


@pytest.mark.parametrize("n", [3, 1000, 8192, 8193])
@pytest.mark.parametrize("width,height", [(256, 200), (2560, 1600)])  # packed rectangles, and too wide for them
def test_small_scenes_depth_order(n, width, height):
    print("small depth order", n, width, height, flush=True)
    sc = S.gaussian_cloud(n, seed=n, pos_std=1.5, logscale=(-5.0, 0.3))
    sc.rows[n // 2:, 0:3] = sc.rows[: n - n // 2, 0:3]  # equal depths
    cam = S.orbit_camera(width, height, 6.0)
    r = P.Renderer(n)
    r.load_buffer(sc.ply_buffer(), n)
    for _ in range(3):  # a frame whose lists outgrow the storage sizes it for the next one
        r.render(cam)
        status, visible, _ = r.frame_info()
        if status == 0:
            break
    ids, keys = r.sorted_ids()
    r.close()
    st = P.parse_ply(sc.ply_buffer(), n)
    stage = P.reference_frame(cam, st, width, height)
    assert status == 0 and visible == len(ids) > 0
    np.testing.assert_array_equal(ids, P.u32(stage["index"])[:visible])
    same = keys[1:] == keys[:-1]
    assert (keys[1:] >= keys[:-1]).all() and (ids[1:][same] > ids[:-1][same]).all()
