"""The sort at the edges of its launch rules: one to many chunks, the grid from which the row scan runs, live
counts of a few chunks in large storage, and the depth sort's three-pass form on small scenes.

Sorted keys and values are integers: bit-exact against numpy's stable argsort and the CPU oracle.
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

# (capacity, live count): sub-tiles of 2048; 256 blocks = 524,288; 64 live chunks; 1024 blocks and beyond
SIZES = [(1, 1), (2047, 2047), (2049, 2049), (16_385, 16_385), (524_288, 524_288), (524_289, 524_289),
         (524_289, 131_072), (524_289, 131_073), (2_097_152, 5), (2_097_152, 131_073), (2_097_153, 2_097_153),
         (3_000_000, 2_500_001)]


@pytest.mark.parametrize("capacity,count", SIZES)
@pytest.mark.parametrize("bits", [3, 8, 17, 32])
def test_sort_sizes(capacity, count, bits):
    print("sort", capacity, count, bits, flush=True)
    rng = np.random.default_rng(capacity + bits)
    key = rng.integers(0, 1 << bits, capacity, dtype=np.uint64).astype(np.uint32)
    key[: capacity // 2] &= np.uint32(0xFFFFFFF3)  # crowded digits
    value = np.arange(capacity, dtype=np.uint32)
    k = torch.from_numpy(key.view(np.int32)).cuda()
    v = torch.from_numpy(value.view(np.int32)).cuda()
    c = torch.tensor([count], dtype=torch.int32, device="cuda")
    P.sort_kv(c, k, v, bits)
    order = np.argsort(key[:count], kind="stable")
    np.testing.assert_array_equal(P.u32(k)[:count], key[:count][order])
    np.testing.assert_array_equal(P.u32(v)[:count], value[:count][order])
    np.testing.assert_array_equal(P.u32(v)[count:], value[count:])


@pytest.mark.parametrize("n", [1, 63, 2048, 20_001, 524_288, 524_289])
@pytest.mark.parametrize("width,height", [(256, 200), (2560, 1600)])
def test_depth_order_of_small_and_larger_scenes(n, width, height):
    """Packed and unpacked values, below and above the three-pass limit (524,288 splats of capacity)."""
    print("depth order", n, width, height, flush=True)
    sc = S.gaussian_cloud(n, seed=n, pos_std=1.5, logscale=(-6.0, 0.3))
    cam = S.orbit_camera(width, height, 3.0)
    r = P.Renderer(n)
    r.load_buffer(sc.ply_buffer(), n)
    for _ in range(3):
        r.render(cam)
        status, v, _ = r.frame_info()
        if status == 0:
            break
    assert status == 0
    ids, keys = r.sorted_ids()
    r.close()
    pos = np.ascontiguousarray(sc.rows[:, 0:3], np.float32)
    ov, okey, oindex = oracle.rank(cam, pos)
    skey, sidx = oracle.sort_kv(okey, oindex)
    assert v == ov
    np.testing.assert_array_equal(keys, skey)
    np.testing.assert_array_equal(ids, sidx)
