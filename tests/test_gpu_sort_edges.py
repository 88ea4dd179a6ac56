"""The sort on both sides of its launch rules' lines: one kernel or passes of short keys (6144 pairs), two or three
launches a pass (192 blocks: 393,216 pairs), 512 or 256 threads and three or four passes (524,288), and the sizes
where chunks are dealt to the dies (512 and 928 single sub-tiles of 2048, chunks of three and four).

Integers: bit-exact against numpy's stable argsort on the sorted bits, and the CPU oracle's depth order.
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


@pytest.mark.parametrize("capacity,count", [
    (6144, 6144), (6145, 6145), (393_216, 393_216), (393_216, 131_073), (393_217, 393_217), (393_217, 131_073),
    (393_217, 131_072), (524_288, 400_000), (1_048_576, 1_048_576), (1_048_577, 1_048_577), (1_900_544, 1_900_544),
    (1_900_545, 1_900_545), (6_291_456, 6_291_456), (6_291_457, 6_291_457)])
@pytest.mark.parametrize("bits", [2, 13, 18, 19, 30])
def test_sorts_at_the_lines(capacity, count, bits):
    print("sort line", capacity, count, bits, flush=True)
    rng = np.random.default_rng(capacity + bits)
    key = rng.integers(0, 1 << 32, capacity, dtype=np.uint64).astype(np.uint32)
    key[: capacity // 2] &= np.uint32(0xFFFFF0F3)  # crowded digits
    value = np.arange(capacity, dtype=np.uint32)
    k = torch.from_numpy(key.view(np.int32)).cuda()
    v = torch.from_numpy(value.view(np.int32)).cuda()
    P.sort_kv(torch.tensor([count], dtype=torch.int32, device="cuda"), k, v, bits)
    order = np.argsort(key[:count] & np.uint32((1 << bits) - 1), kind="stable")
    np.testing.assert_array_equal(P.u32(k)[:count], key[:count][order])
    np.testing.assert_array_equal(P.u32(v)[:count], value[:count][order])
    np.testing.assert_array_equal(P.u32(v)[count:], value[count:])


@pytest.mark.parametrize("n", [393_216, 393_217, 524_288])
@pytest.mark.parametrize("width,height", [(256, 200), (2560, 1600)])  # packed rectangles, and too wide for them
def test_three_wide_passes_with_and_without_the_row_scan(n, width, height):
    print("wide depth order", n, width, height, flush=True)
    sc = S.gaussian_cloud(n, seed=n, pos_std=1.5, logscale=(-6.0, 0.3))
    cam = S.orbit_camera(width, height, 9.0)
    r = P.Renderer(n)
    r.load_buffer(sc.ply_buffer(), n)
    for _ in range(3):  # a frame whose lists outgrow the storage sizes it for the next one
        r.render(cam)
        status, v, _ = r.frame_info()
        if status == 0:
            break
    ids, keys = r.sorted_ids()
    r.close()
    ov, okey, oindex = oracle.rank(cam, np.ascontiguousarray(sc.rows[:, 0:3], np.float32))
    skey, sidx = oracle.sort_kv(okey, oindex)
    assert v == ov > 64 * 2048
    np.testing.assert_array_equal(keys, skey)
    np.testing.assert_array_equal(ids, sidx)


@pytest.mark.parametrize("n", [5000, 8193, 300_000, 600_000])
def test_storage_aligned_to_a_word_only(n):
    """Storage that starts one word into an allocation sorts as any other."""
    print("word-aligned storage", n, flush=True)
    from vkgs_amd._lib import check, lib
    key = np.random.default_rng(n).integers(0, 1 << 30, n, dtype=np.uint64).astype(np.uint32)
    k = torch.from_numpy(key.view(np.int32)).cuda()
    v = torch.arange(n, dtype=torch.int32, device="cuda")
    c = torch.tensor([n], dtype=torch.int32, device="cuda")
    nbytes = lib().vkgs_sort_kv_storage_bytes(n)
    storage = torch.empty(nbytes + 4, dtype=torch.uint8, device="cuda")
    check(lib().vkgs_sort_kv(n, c.data_ptr(), k.data_ptr(), v.data_ptr(), 30, storage.data_ptr() + 4, nbytes,
                             torch.cuda.current_stream().cuda_stream), "vkgs_sort_kv")
    order = np.argsort(key, kind="stable")
    np.testing.assert_array_equal(P.u32(k), key[order])
    np.testing.assert_array_equal(P.u32(v), order)
