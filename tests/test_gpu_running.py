"""A commit right after an asynchronous query that has not run yet: the query
still sees the mesh that was committed when it was queued (records identical to
the oracle's on it), and the next one sees the new mesh."""
import ctypes

import numpy as np
import pytest

from conftest import mismatches

pytestmark = pytest.mark.gpu

NOT_READY = 600  # hipErrorNotReady
N = 50000


def hip():
    h = ctypes.CDLL("libamdhip64.so")
    for f in ("hipStreamSynchronize", "hipStreamDestroy", "hipStreamQuery"):
        getattr(h, f).argtypes = [ctypes.c_void_p]
    h.hipStreamCreateWithFlags.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_uint]
    return h


@pytest.fixture(scope="module")
def queue(rtc, device):
    """A caller's stream, and what keeps it busy for tens of milliseconds."""
    h, s = hip(), ctypes.c_void_p()
    assert h.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
    sc = rtc.Scene(device, [rtc.gen_soup(1 << 20, seed=1)]).commit()
    recs = rtc.gen_random_rays(1 << 22, seed=2)
    d = device.malloc(recs.nbytes)
    device.memcpy(d, recs.ctypes.data, recs.nbytes)

    def fill():
        for _ in range(20):  # (the closest hit lies within the distance that the one before wrote)
            rtc.lib().rtcgIntersect1MAsync(sc.h, ctypes.byref(rtc.init_context()), d, len(recs), 80, s)

    yield h, s, fill
    assert h.hipStreamSynchronize(s) == 0
    device.free(d)
    sc.release()
    h.hipStreamDestroy(s)


class Records:
    def __init__(self, rtc, device, lo, hi):
        self.src, self.device = rtc.gen_random_rays(N, seed=5, lo=lo, hi=hi), device
        self.d = device.malloc(self.src.nbytes)
        device.memcpy(self.d, self.src.ctypes.data, self.src.nbytes)

    def get(self):
        out = np.empty_like(self.src)
        self.device.memcpy(out.ctypes.data, self.d, out.nbytes)
        return out

    def expect(self, oracle, mesh):
        ref = self.src.copy()
        oracle.BVH([mesh]).intersect(ref)
        return ref


def shared_scene(rtc, device, mesh, quality):
    """A scene over the caller's own vertices (padded), which it may rewrite."""
    v, ix = mesh
    verts = np.zeros((len(v) + 1, 3), np.float32)
    verts[:-1] = v
    ix = np.ascontiguousarray(ix)
    L = rtc.lib()
    sc = rtc.Scene(device, quality=quality)
    sc.keep = [verts, ix]
    g = L.rtcNewGeometry(device.h, rtc.RTC_GEOMETRY_TYPE_TRIANGLE)
    L.rtcSetSharedGeometryBuffer(g, rtc.RTC_BUFFER_TYPE_VERTEX, 0, rtc.RTC_FORMAT_FLOAT3, verts.ctypes.data, 0, 12, len(v))
    L.rtcSetSharedGeometryBuffer(g, rtc.RTC_BUFFER_TYPE_INDEX, 0, rtc.RTC_FORMAT_UINT3, ix.ctypes.data, 0, 12, len(ix))
    L.rtcCommitGeometry(g)
    L.rtcAttachGeometry(sc.h, g)
    L.rtcReleaseGeometry(g)
    sc.commit()

    def change(new):
        verts[:-1] = new
        L.rtcUpdateGeometryBuffer(g, rtc.RTC_BUFFER_TYPE_VERTEX, 0)
        L.rtcCommitGeometry(g)
        sc.commit()

    return sc, change


# a scene committed once is only noted, one committed again gets an event
@pytest.mark.parametrize("commits", [1, 2])
@pytest.mark.parametrize("call", ["async", "no_alloc"])
@pytest.mark.parametrize("quality,size", [("LOW", 300), ("MEDIUM", 20000), ("HIGH", 20000)])
def test_commit_after_a_queued_query(rtc, device, oracle, queue, quality, size, call, commits):
    h, s, fill = queue
    v, ix = rtc.gen_soup(size, seed=7, h=0.05)
    sc, change = shared_scene(rtc, device, (v, ix), getattr(rtc, f"RTC_BUILD_QUALITY_{quality}"))
    first, second = (Records(rtc, device, 0.0, 1.0) for _ in range(2))
    want = first.expect(oracle, (v, ix))
    for _ in range(commits - 1):
        change(v)
    w = np.ascontiguousarray(v[::-1]) * np.float32(0.75)
    after = second.expect(oracle, (w, ix))
    L, ctx = rtc.lib(), rtc.init_context()
    fill()
    if call == "async":
        L.rtcgIntersect1MAsync(sc.h, ctypes.byref(ctx), first.d, N, 80, s)
    else:
        L.rtcgQuery1MNoAlloc(sc.h, ctypes.byref(ctx), first.d, N, 80, 0, s)
    device.check("query")
    assert h.hipStreamQuery(s) == NOT_READY
    change(w)
    L.rtcgIntersect1MAsync(sc.h, ctypes.byref(ctx), second.d, N, 80, s)
    assert h.hipStreamSynchronize(s) == 0
    device.check("query")
    assert len(mismatches(first.get(), want)) == 0
    assert len(mismatches(second.get(), after)) == 0
    for r in (first, second):
        device.free(r.d)
    sc.release()


@pytest.mark.parametrize("commits", [1, 2])
def test_commit_of_a_two_level_scene_after_a_queued_query(rtc, device, oracle, queue, commits):
    h, s, fill = queue
    v, ix = rtc.gen_sphere(24)
    obj = rtc.Scene(device, [(v, ix)]).commit()
    moves = rtc.random_transforms(60, seed=6, scale=(0.3, 0.6), extent=3.0)

    def place(a):
        top = rtc.Scene(device)
        for m in moves[a:a + 30]:
            top.add_instance(obj, m)
        return top.commit()

    def traced(sc, r):
        out = r.src.copy()
        sc.intersect1M(out)
        return out

    first, second = (Records(rtc, device, -3.0, 3.0) for _ in range(2))
    other = place(30)
    after = traced(other, second)
    other.release()
    top = place(0)
    for _ in range(commits - 1):
        top.commit()
    want = traced(top, first)
    assert len(mismatches(want, after)) > 100
    L, ctx = rtc.lib(), rtc.init_context()
    fill()
    L.rtcgIntersect1MAsync(top.h, ctypes.byref(ctx), first.d, N, 80, s)
    assert h.hipStreamQuery(s) == NOT_READY
    for k, m in enumerate(moves[30:]):
        g = L.rtcGetGeometry(top.h, k)
        m = np.ascontiguousarray(m, np.float32).reshape(-1)
        L.rtcSetGeometryTransform(g, 0, rtc.RTC_FORMAT_FLOAT3X4_COLUMN_MAJOR, m.ctypes.data)
        L.rtcCommitGeometry(g)
    top.commit()
    L.rtcgIntersect1MAsync(top.h, ctypes.byref(ctx), second.d, N, 80, s)
    assert h.hipStreamSynchronize(s) == 0
    device.check("query")
    assert len(mismatches(first.get(), want)) == 0
    assert len(mismatches(second.get(), after)) == 0
    for r in (first, second):
        device.free(r.d)
    top.release()
    obj.release()


@pytest.mark.parametrize("commits", [1, 2])
def test_queries_of_many_scenes(rtc, device, oracle, queue, commits):
    """More scenes with queued queries than the library has events for, or
    keeps apart."""
    h, s, fill = queue
    v, ix = rtc.gen_soup(2000, seed=8, h=0.05)
    w = np.ascontiguousarray(v[::-1])
    scenes = [shared_scene(rtc, device, (v, ix), rtc.RTC_BUILD_QUALITY_LOW) for _ in range(70)]
    for _, change in scenes * (commits - 1):
        change(v)
    recs = [Records(rtc, device, 0.0, 1.0) for _ in scenes]
    want = recs[0].expect(oracle, (v, ix))
    L, ctx = rtc.lib(), rtc.init_context()
    fill()
    for (sc, _), r in zip(scenes, recs):
        L.rtcgIntersect1MAsync(sc.h, ctypes.byref(ctx), r.d, N, 80, s)
    assert h.hipStreamQuery(s) == NOT_READY
    for _, change in scenes:
        change(w)
    assert h.hipStreamSynchronize(s) == 0
    device.check("query")
    for r in recs:
        assert len(mismatches(r.get(), want)) == 0
        device.free(r.d)
    for sc, _ in scenes:
        sc.release()


def test_commit_after_a_replayed_query(rtc, oracle, queue):
    h, s, fill = queue
    device = rtc.Device("")
    v, ix = rtc.gen_soup(20000, seed=9, h=0.05)
    sc, change = shared_scene(rtc, device, (v, ix), rtc.RTC_BUILD_QUALITY_LOW)
    r = Records(rtc, device, 0.0, 1.0)
    want = r.expect(oracle, (v, ix))
    graph, run = ctypes.c_void_p(), ctypes.c_void_p()
    assert h.hipStreamBeginCapture(s, 2) == 0  # hipStreamCaptureModeRelaxed
    rtc.lib().rtcgIntersect1MAsync(sc.h, ctypes.byref(rtc.init_context()), r.d, N, 80, s)
    assert h.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
    device.check("capture")
    assert h.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
    fill()
    assert h.hipGraphLaunch(run, s) == 0
    assert h.hipStreamQuery(s) == NOT_READY
    change(np.ascontiguousarray(v[::-1]))
    assert h.hipStreamSynchronize(s) == 0
    assert len(mismatches(r.get(), want)) == 0
    assert h.hipGraphExecDestroy(run) == 0
    assert h.hipGraphDestroy(graph) == 0
    device.free(r.d)
    sc.release()
    device.release()
