"""Hits whose distance overflows to infinity or NaN (inf / inf, with an interval
that begins behind the origin) are recorded as the oracle records them, by the
kernel of one lane a ray and that of eight, and in two-level scenes."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def case(rtc, oracle):
    s = 1e18
    mesh = np.array([[-s, -s, s], [s, -s, s], [0, s, s]], np.float32), np.array([[0, 1, 2]], np.uint32)
    rays = rtc.new_rayhits(70001)  # more than eight lanes a ray take
    rng = np.random.default_rng(3)
    rays["org_z"] = -s
    rays["dir_x"] = rng.random(len(rays)) * 1e-3
    rays["dir_z"] = np.where(np.arange(len(rays)) % 3 == 0, 1.0, 10.0 ** rng.uniform(2.5, 6.0, len(rays)))
    rays["tnear"] = -1.0
    want = rays.copy()
    oracle.BVH([mesh]).intersect(want)
    assert np.isnan(want["tfar"]).sum() > 40000 and np.isinf(want["tfar"]).sum() > 20000
    assert (want["geomID"] == 0).all()
    return mesh, rays, want


@pytest.mark.parametrize("two_level", [False, True])
@pytest.mark.parametrize("n", [1, 1000, 70001])
def test_distances_that_overflow(rtc, device, case, n, two_level):
    mesh, rays, want = case
    sc = top = rtc.Scene(device, [mesh]).commit()
    if two_level:
        top = rtc.Scene(device)
        top.add_instance(sc, np.array([1, 0, 0, 0, 1, 0, 0, 0, 1, 0, 0, 0], np.float32))
        top.commit()
    out = rays[:n].copy()
    d = device.malloc(out.nbytes)
    device.memcpy(d, out.ctypes.data, out.nbytes)
    rtc.lib().rtcIntersect1M(top.h, ctypes.byref(rtc.init_context()), d, n, 80)
    device.check("query")
    device.memcpy(out.ctypes.data, d, out.nbytes)
    device.free(d)
    for k in out.dtype.names:
        if k != "instID":
            assert np.array_equal(out[k], want[:n][k], equal_nan=out[k].dtype.kind == "f"), k
    assert (out["instID"] == (0 if two_level else 0xFFFFFFFF)).all()
    if two_level:
        top.release()
    sc.release()
