"""Node boxes and leaf decisions are formed bottom-up by chunks of 1024
positions, then by 32 chunks at a time: every primitive count around those
edges, and trees whose nodes span many chunks, answer as the oracle's brute
force and hold every primitive once."""
import numpy as np
import pytest

from conftest import mismatches

pytestmark = pytest.mark.gpu


def check(rtc, oracle, device, mesh, quality, n_rays=400):
    sc = rtc.Scene(device, [mesh], quality=quality).commit()
    _, tris = sc.read_bvh()
    rec = tris.view(np.uint32).reshape(-1, 12)
    assert np.array_equal(np.sort(rec[:, 3]), np.arange(len(mesh[1])))
    rays = rtc.gen_random_rays(n_rays, seed=3)
    ref = rays.copy()
    sc.intersect1M(rays)
    oracle.BVH([mesh]).intersect(ref)
    assert len(mismatches(rays, ref)) == 0
    sc.release()


@pytest.mark.parametrize("quality", [0, 1])
@pytest.mark.parametrize("n", [2, 3, 1023, 1024, 1025, 1026, 2049, 32767, 32768, 32769, 33793])
def test_sizes_around_the_chunks(rtc, oracle, device, n, quality):
    check(rtc, oracle, device, rtc.gen_soup(n, seed=n, h=0.02), quality)


@pytest.mark.parametrize("quality", [0, 1])
def test_three_levels_of_chunks(rtc, oracle, device, quality):
    check(rtc, oracle, device, rtc.gen_soup((1 << 20) + 1, seed=8), quality)


@pytest.mark.parametrize("quality", [0, 1])
def test_skewed_and_equal_primitives(rtc, oracle, device, quality):
    # sizes and positions in geometric steps (deep, one-sided splits), and 3000
    # copies of one triangle (equal Morton codes, no spatial split)
    v, ix = rtc.gen_soup(40000, seed=9, h=0.01)
    v = v.reshape(-1, 3, 3)
    v *= (0.9995 ** np.arange(len(v), dtype=np.float64)).astype(np.float32)[:, None, None]
    v[5000:8000] = v[5000]
    check(rtc, oracle, device, (v.reshape(-1, 3), ix), quality)


@pytest.mark.parametrize("width", [2, 3, 8])
@pytest.mark.parametrize("n", [1, 9, 511, 513, 2048, 2049, 4097, 70001])
def test_widths_and_subtrees(rtc, oracle, n, width):
    # the wide nodes are numbered by subtrees of at most 2048 primitives or 1/256 of them
    dev = rtc.Device(f"bvh_width={width}")
    check(rtc, oracle, dev, rtc.gen_soup(n, seed=n + 1, h=0.03), 1)
    dev.release()


def test_more_scenes_than_top_nodes(rtc, oracle, device):
    # 2300 scenes of one build: empty ones, single triangles, small meshes and a large one
    meshes = [rtc.gen_soup(k % 7, seed=k + 1, h=0.2) if k % 500 else rtc.gen_soup(20000, seed=k + 1, h=0.02)
              for k in range(2300)]
    scs = [rtc.Scene(device, [m]) for m in meshes]
    rtc.commit_scenes(scs)
    for k in (0, 1, 2, 6, 7, 500, 501, 1999, 2000, 2299):
        rays = rtc.gen_random_rays(200, seed=k)
        ref = rays.copy()
        scs[k].intersect1M(rays)
        oracle.BVH([meshes[k]]).intersect(ref)
        assert len(mismatches(rays, ref)) == 0, k
    for s in scs:
        s.release()
