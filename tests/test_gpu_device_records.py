"""Streams in device memory that are large enough for the kernels of one lane a
ray (records in host memory go through in pieces that eight lanes a ray take),
and two-level scenes queried in host memory: every record identical to the
oracle's, or to that of the same query over device records."""
import ctypes

import numpy as np
import pytest

from conftest import mismatches

pytestmark = pytest.mark.gpu


def on_device(rtc, dev, sc, recs):
    call = rtc.lib().rtcOccluded1M if recs.itemsize == 48 else rtc.lib().rtcIntersect1M
    d = dev.malloc(recs.nbytes)
    dev.memcpy(d, recs.ctypes.data, recs.nbytes)
    call(sc.h, ctypes.byref(rtc.init_context()), d, len(recs), recs.itemsize)
    dev.check("query")
    out = np.empty_like(recs)
    dev.memcpy(out.ctypes.data, d, recs.nbytes)
    dev.free(d)
    return out


def shadow_of(rtc, rays, tfar):
    out = np.zeros(len(rays), rtc.RTCRay)
    for k in rtc.RTCRay.names:
        out[k] = rays[k]
    out["tfar"] = tfar
    return out


@pytest.mark.slow
def test_soup_full_size(rtc, device, oracle):
    mesh = rtc.gen_soup(1 << 20, seed=1, h=0.005)
    sc = rtc.Scene(device, [mesh]).commit()
    bvh = oracle.BVH([mesh])
    rays = rtc.gen_random_rays(1 << 24, seed=2)
    shadow = shadow_of(rtc, rays[:1 << 23], 0.1)
    out = on_device(rtc, device, sc, rays)
    bvh.intersect(rays)
    assert len(mismatches(out, rays)) == 0
    out = on_device(rtc, device, sc, shadow)
    bvh.occluded(shadow)
    assert len(mismatches(out, shadow)) == 0
    sc.release()


@pytest.mark.parametrize("robust", [False, True])
@pytest.mark.parametrize("config", ["", "refill_min=1,refill_min_occ=1", "refill_min=64,refill_min_occ=64,blocks_per_cu=1",
                                    "trace_stack=0", "trace_stack=8", "trace_stack=16", "persistent=0", "ray_sort=1"])
def test_one_lane_kernels(rtc, oracle, config, robust):
    dev = rtc.Device(config)
    mesh = rtc.gen_soup(20000, seed=17, h=0.02)
    sc = rtc.Scene(dev, [mesh], flags=rtc.RTC_SCENE_FLAG_ROBUST if robust else 0).commit()
    bvh = oracle.BVH([mesh])
    rays = rtc.gen_random_rays(500001, seed=18)
    shadow = shadow_of(rtc, rays, 0.1)
    for recs, check in ((rays, bvh.intersect), (shadow, bvh.occluded)):
        want = recs.copy()
        check(want, robust=robust)
        assert len(mismatches(on_device(rtc, dev, sc, recs), want)) == 0
    sc.release()
    dev.release()


@pytest.mark.parametrize("n", [1, 1000, 8192, 8193, 100001])
def test_two_level_queries_in_host_memory(rtc, device, n):
    obj = rtc.Scene(device, [rtc.gen_soup(5000, seed=3, h=0.05)]).commit()
    top = rtc.Scene(device)
    for m in rtc.random_transforms(80, seed=4, scale=(0.5, 2.0), extent=4.0):
        top.add_instance(obj, m)
    top.commit()
    rays = rtc.gen_random_rays(n, seed=5, lo=-4.0, hi=4.0)
    shadow = shadow_of(rtc, rays, 2.0)
    for recs, call in ((rays, rtc.lib().rtcIntersect1M), (shadow, rtc.lib().rtcOccluded1M)):
        step = recs.itemsize + 12
        wide = np.full((n, step), 0xA5, np.uint8)
        wide[:, :recs.itemsize] = recs.view(np.uint8).reshape(n, -1)
        call(top.h, ctypes.byref(rtc.init_context()), wide.ctypes.data, n, step)
        device.check("query")
        got = np.ascontiguousarray(wide[:, :recs.itemsize]).reshape(-1).view(recs.dtype)
        assert len(mismatches(got, on_device(rtc, device, top, recs))) == 0
        assert (wide[:, recs.itemsize:] == 0xA5).all()
    top.release()
    obj.release()
