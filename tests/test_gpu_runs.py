"""Small streams are traced with eight lanes a ray, larger ones with one, whose
rays are shared out in runs of 64 to waves and queues: every record of every
stream length around the edges of a block, of the change between the two, of
the eight queues and the waves' first runs is traced once, byte-identical to
the oracle."""
import ctypes
import threading

import numpy as np
import pytest

from conftest import mismatches

pytestmark = pytest.mark.gpu

# one ray, a block of eight, the last sizes with eight lanes a ray (occlusion,
# closest hit) and the first with one, all resident waves' first runs at 5, 6
# and 7 blocks on 256 compute units, and past them (the counters start)
SIZES = [1, 7, 8, 9, 1021, 32767, 32769, 65535, 65537, 327679, 327681, 393215, 393217, 458753, 600001]


@pytest.fixture(scope="module")
def scene(rtc, device, oracle):
    mesh = rtc.gen_sphere(8)
    sc = rtc.Scene(device, [mesh]).commit()
    rays = rtc.gen_random_rays(max(SIZES), seed=31, lo=-2.0, hi=2.0)
    rays["tnear"][::17] = 1.0
    rays["tfar"][::17] = 0.5  # skipped records
    hits = rays.copy()
    bvh = oracle.BVH([mesh])
    bvh.intersect(hits)
    shadow = np.zeros(len(rays), rtc.RTCRay)
    for k in rtc.RTCRay.names:
        shadow[k] = rays[k]
    dark = shadow.copy()
    bvh.occluded(dark)
    yield sc, rays, hits, shadow, dark
    sc.release()


def on_device(rtc, device, sc, recs, call):
    d = device.malloc(recs.nbytes)
    device.memcpy(d, recs.ctypes.data, recs.nbytes)
    call(sc.h, ctypes.byref(rtc.init_context()), d, len(recs), recs.itemsize)
    device.check("query")
    device.memcpy(recs.ctypes.data, d, recs.nbytes)
    device.free(d)
    return recs


@pytest.mark.parametrize("n", SIZES)
def test_every_record_of_a_stream(rtc, device, scene, n):
    sc, rays, hits, shadow, dark = scene
    L = rtc.lib()
    assert len(mismatches(on_device(rtc, device, sc, rays[:n].copy(), L.rtcIntersect1M), hits[:n])) == 0
    assert len(mismatches(on_device(rtc, device, sc, shadow[:n].copy(), L.rtcOccluded1M), dark[:n])) == 0


# in place in pinned memory up to 8192 records, then chunks of 16384 to 65536 on up to eight threads
@pytest.mark.parametrize("stride", [0, 12])
@pytest.mark.parametrize("n", [1, 2, 8191, 8192, 8193, 16384, 16385, 50001, 300001, 600001])
def test_every_record_in_host_memory(rtc, device, scene, n, stride):
    sc, rays, hits, shadow, dark = scene
    L = rtc.lib()
    for src, ref, call in ((rays, hits, L.rtcIntersect1M), (shadow, dark, L.rtcOccluded1M)):
        step = src.itemsize + stride
        buf = np.full((n, step), 0xA5, np.uint8)
        buf[:, :src.itemsize] = src[:n].view(np.uint8).reshape(n, -1)
        call(sc.h, ctypes.byref(rtc.init_context()), buf.ctypes.data, n, step)
        device.check("query")
        got = np.ascontiguousarray(buf[:, :src.itemsize]).reshape(-1).view(src.dtype)
        assert len(mismatches(got, ref[:n])) == 0
        assert (buf[:, src.itemsize:] == 0xA5).all()


def test_host_queries_of_several_threads(rtc, device, scene):
    sc, rays, hits, _, _ = scene
    bad = []

    def one(n, first):
        out = rays[first:first + n].copy()
        sc.intersect1M(out)
        bad.append(len(mismatches(out, hits[first:first + n])))

    th = [threading.Thread(target=one, args=(100000 + 7 * k, 20000 * k)) for k in range(6)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert bad == [0] * 6


def test_geometry_uploads_in_pieces_and_again(rtc, oracle):
    # buffers above and below the size that several threads copy, with a vertex
    # stride, in one geometry that changes size from commit to commit
    dev = rtc.Device("")
    L = rtc.lib()
    sc = rtc.Scene(dev)
    g = L.rtcNewGeometry(dev.h, rtc.RTC_GEOMETRY_TYPE_TRIANGLE)
    L.rtcAttachGeometry(sc.h, g)
    rays = rtc.gen_random_rays(2000, seed=8)
    for n in (500, 400000, 399000, 900000, 40, 400000):
        v, ix = rtc.gen_soup(n, seed=n, h=0.02)
        wide = np.full((len(v) + 1, 5), np.nan, np.float32)
        wide[:-1, :3] = v
        ix = np.ascontiguousarray(ix)
        L.rtcSetSharedGeometryBuffer(g, rtc.RTC_BUFFER_TYPE_VERTEX, 0, rtc.RTC_FORMAT_FLOAT3, wide.ctypes.data, 0, 20, len(v))
        L.rtcSetSharedGeometryBuffer(g, rtc.RTC_BUFFER_TYPE_INDEX, 0, rtc.RTC_FORMAT_UINT3, ix.ctypes.data, 0, 12, n)
        L.rtcCommitGeometry(g)
        sc.commit()
        out, ref = rays.copy(), rays.copy()
        sc.intersect1M(out)
        oracle.BVH([(v, ix)]).intersect(ref)
        assert len(mismatches(out, ref)) == 0, n
    L.rtcReleaseGeometry(g)
    sc.release()
    dev.release()


@pytest.mark.parametrize("n", [1, 65, 2049, 327681, 600001])
def test_every_record_through_an_instance(rtc, device, oracle, scene, n):
    sc, rays, _, _, _ = scene
    l2w = np.eye(4, 3, dtype=np.float32).reshape(12)
    l2w[9:12] = 0.5, 0.0, -0.25
    top = rtc.Scene(device)
    top.add_instance(sc, l2w)
    top.commit()
    out = on_device(rtc, device, top, rays[:n].copy(), rtc.lib().rtcIntersect1M)
    ref = rays[:n].copy()
    o = oracle.Instances()
    o.add_instance(o.add_object([rtc.gen_sphere(8)]), l2w, 0)
    o.intersect_bvh(ref)
    assert len(mismatches(out, ref)) == 0
    top.release()


@pytest.mark.parametrize("config,robust", [("", False), ("", True), ("bvh_leaf=15,cost_tri=0.02", False),
                                           ("bvh_leaf=15,cost_tri=0.02", True), ("bvh_width=2", False)])
@pytest.mark.parametrize("n,stride", [(999, 80), (999, 84), (70001, 80), (70001, 84)])
def test_both_kernels_on_other_trees(rtc, oracle, config, robust, n, stride):
    # leaves of more than eight triangles, binary trees, robust scenes, records
    # that are not 16-byte aligned, intervals that start behind the origin
    dev = rtc.Device(config)
    soup = rtc.gen_soup(3000, seed=5, h=0.06)
    sc = rtc.Scene(dev, [soup, rtc.gen_sphere(9, center=(0.5, 0.5, 0.5), radius=0.3)],
                   flags=rtc.RTC_SCENE_FLAG_ROBUST if robust else 0).commit()
    bvh = oracle.BVH([soup, rtc.gen_sphere(9, center=(0.5, 0.5, 0.5), radius=0.3)])
    rays = rtc.gen_random_rays(n, seed=6)
    rays["tnear"][::3] = -0.5
    rays["tfar"][1::5] = 0.2
    ref = rays.copy()
    bvh.intersect(ref, robust=robust)
    wide = np.zeros((n, stride), np.uint8)
    wide[:, :80] = rays.view(np.uint8).reshape(n, 80)
    d = dev.malloc(wide.nbytes)
    dev.memcpy(d, wide.ctypes.data, wide.nbytes)
    rtc.lib().rtcIntersect1M(sc.h, ctypes.byref(rtc.init_context()), d, n, stride)
    dev.check("rtcIntersect1M")
    dev.memcpy(wide.ctypes.data, d, wide.nbytes)
    dev.free(d)
    assert len(mismatches(np.ascontiguousarray(wide[:, :80]).reshape(-1).view(rtc.RTCRayHit), ref)) == 0
    occ = np.zeros(n, rtc.RTCRay)
    for k in rtc.RTCRay.names:
        occ[k] = rays[k]
    dark = occ.copy()
    sc.occluded1M(occ)
    bvh.occluded(dark, robust=robust)
    assert len(mismatches(occ, dark)) == 0
    sc.release()
    dev.release()


@pytest.mark.parametrize("n", [65, 32771, 65539, 393217, 600001])
def test_every_record_of_a_batch(rtc, device, scene, n):
    _, rays, hits, _, _ = scene
    mesh = rtc.gen_sphere(8)
    scs = [rtc.Scene(device, [mesh]) for _ in range(3)]
    rtc.commit_scenes(scs)
    first = [0, n // 3, n // 3 + 1, n]
    d = device.malloc(80 * n)
    items = rtc.batch_items([(s, d + 80 * a, b - a, 80) for s, a, b in zip(scs, first, first[1:])])
    graph = rtc.lib().rtcgNewBatchGraph(items.ctypes.data, 3, 0)
    device.check("rtcgNewBatchGraph")
    for _ in range(2):
        out = rays[:n].copy()
        device.memcpy(d, out.ctypes.data, out.nbytes)
        rtc.lib().rtcgLaunchBatchGraph(graph, None)
        device.check("rtcgLaunchBatchGraph")
        device.memcpy(out.ctypes.data, d, out.nbytes)
        assert len(mismatches(out, hits[:n])) == 0
    rtc.lib().rtcgReleaseBatchGraph(graph)
    device.free(d)
    for s in scs:
        s.release()


def test_queries_that_overlap_on_several_streams(rtc, device, scene):
    # one thread, more streams than keep ray counters of their own, each with a
    # closest-hit and an occlusion query too large for the waves' first runs
    sc, rays, hits, shadow, dark = scene
    hip = ctypes.CDLL("libamdhip64.so")
    L, ctx, made = rtc.lib(), rtc.init_context(), []
    for k in range(20):
        s = ctypes.c_void_p()
        assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
        bufs = []
        for src in (rays, shadow):
            d = device.malloc(src.nbytes)
            device.memcpy(d, src.ctypes.data, src.nbytes)
            bufs.append(d)
        made.append((s, bufs))
    for s, (a, b) in made:
        L.rtcgIntersect1MAsync(sc.h, ctypes.byref(ctx), a, len(rays), 80, s)
        L.rtcgOccluded1MAsync(sc.h, ctypes.byref(ctx), b, len(shadow), 48, s)
    device.check("queries")
    for s, bufs in made:
        assert hip.hipStreamSynchronize(s) == 0
        for d, ref in zip(bufs, (hits, dark)):
            out = np.empty_like(ref)
            device.memcpy(out.ctypes.data, d, out.nbytes)
            assert len(mismatches(out, ref)) == 0
            device.free(d)
        assert hip.hipStreamDestroy(s) == 0


def test_captured_query(rtc, device, scene):
    # captured on a stream of its own after a query on another one, replayed
    # with eager queries between
    sc, rays, hits, _, _ = scene
    hip = ctypes.CDLL("libamdhip64.so")
    L, ctx = rtc.lib(), rtc.init_context()
    d, src = device.malloc(rays.nbytes), device.malloc(rays.nbytes)
    device.memcpy(src, rays.ctypes.data, rays.nbytes)
    s, graph, run = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
    assert hip.hipStreamBeginCapture(s, 2) == 0  # hipStreamCaptureModeRelaxed
    L.rtcgIntersect1MAsync(sc.h, ctypes.byref(ctx), d, len(rays), 80, s)
    assert hip.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
    device.check("capture")
    assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        device.memcpy(d, src, rays.nbytes)
        assert hip.hipGraphLaunch(run, s) == 0
        assert hip.hipStreamSynchronize(s) == 0
        out = np.empty_like(rays)
        device.memcpy(out.ctypes.data, d, out.nbytes)
        assert len(mismatches(out, hits)) == 0
        eager = rays[:100000].copy()
        sc.intersect1M(eager)
        assert len(mismatches(eager, hits[:100000])) == 0
    assert hip.hipGraphExecDestroy(run) == 0
    assert hip.hipGraphDestroy(graph) == 0
    assert hip.hipStreamDestroy(s) == 0
    device.free(d)
    device.free(src)
