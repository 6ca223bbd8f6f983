"""Segments of more than 4096 references are split by chunks of 1024
positions, each meeting at most two of them: counts around those edges,
segments that begin anywhere in a chunk, and segments no bin separates
answer as the oracle's brute force and hold every primitive once."""
import numpy as np
import pytest

from conftest import mismatches

pytestmark = pytest.mark.gpu


def prims(sc):
    _, tris = sc.read_bvh()
    return np.sort(tris.view(np.uint32).reshape(-1, 12)[:, 3])


def check(rtc, oracle, sc, mesh, n_rays=300):
    rays = rtc.gen_random_rays(n_rays, seed=4)
    ref = rays.copy()
    sc.intersect1M(rays)
    oracle.BVH([mesh]).intersect(ref)
    assert len(mismatches(rays, ref)) == 0


@pytest.mark.parametrize("quality", [1, 2])
@pytest.mark.parametrize("n", [4096, 4097, 5119, 5120, 5121, 8193, 9217, 66561])
def test_sizes_around_the_classes(rtc, oracle, device, n, quality):
    mesh = rtc.gen_soup(n, seed=n, h=0.02)
    sc = rtc.Scene(device, [mesh], quality=quality).commit()
    assert np.array_equal(prims(sc), np.arange(n))
    check(rtc, oracle, sc, mesh)
    sc.release()


def test_segments_that_begin_inside_a_chunk(rtc, oracle, device):
    # one build of 40 trees, large and small in turn
    sizes = [(4097 + 389 * k) if k % 3 else 1 + 97 * k for k in range(40)]
    meshes = [rtc.gen_soup(n, seed=n, h=0.03) for n in sizes]
    scs = [rtc.Scene(device, [m]) for m in meshes]
    rtc.commit_scenes(scs)
    # the scenes of a build share its records
    assert np.array_equal(prims(scs[0]), np.sort(np.concatenate([np.arange(n) for n in sizes])))
    for s, m in zip(scs, meshes):
        check(rtc, oracle, s, m, 60)
        s.release()


@pytest.mark.parametrize("copies", [4097, 13000])
def test_references_no_bin_separates(rtc, oracle, device, copies):
    # copies of one triangle among others: object medians of large segments
    v, ix = rtc.gen_soup(copies + 9000, seed=5, h=0.02)
    v = v.reshape(-1, 3, 3)
    v[3000:3000 + copies] = v[3000]
    mesh = (v.reshape(-1, 3), ix)
    sc = rtc.Scene(device, [mesh]).commit()
    assert np.array_equal(prims(sc), np.arange(copies + 9000))
    check(rtc, oracle, sc, mesh)
    sc.release()
