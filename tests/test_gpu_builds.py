"""Builds that share a device's scratch memory with other threads' builds."""
import threading

import numpy as np
import pytest

from conftest import mismatches

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quality", ["LOW", "MEDIUM"])
def test_builds_beside_builds_without_a_valid_primitive(rtc, device, oracle, quality):
    q = getattr(rtc, f"RTC_BUILD_QUALITY_{quality}")
    v, ix = rtc.gen_soup(60000, seed=3, h=0.01)
    rays = rtc.gen_random_rays(20000, seed=4)
    want = rays.copy()
    oracle.BVH([(v, ix)]).intersect(want)
    bad = []
    stop = threading.Event()

    def invalid():
        w, jx = rtc.gen_soup(400000, seed=5)
        w[::3] = np.nan  # a corner of every triangle
        sc = rtc.Scene(device, [(w, jx)], quality=q)
        while not stop.is_set():
            sc.commit()
            if sc.stats()["num_prims"] != 0:
                bad.append("a primitive of the invalid mesh")
        sc.release()

    other = threading.Thread(target=invalid)
    other.start()
    try:
        for _ in range(40):
            sc = rtc.Scene(device, [(v, ix)], quality=q).commit()
            _, tris = sc.read_bvh()
            prims = tris.view(np.uint32).reshape(-1, 12)[:, 3]  # primID, the fourth word of a record
            if len(np.unique(prims)) != len(ix) or len(prims) != len(ix):
                bad.append("lost or doubled primitives")
            out = rays.copy()
            sc.intersect1M(out)
            if len(mismatches(out, want)):
                bad.append("wrong hits")
            sc.release()
    finally:
        stop.set()
        other.join()
    assert not bad
