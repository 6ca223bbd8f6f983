"""The rays of a launch are shared out in runs of 64 to waves and queues:
every record of every stream length around the edges of a run, a block, the
eight queues and the waves' first runs is traced once, byte-identical to the
oracle."""
import numpy as np
import pytest

from conftest import mismatches

pytestmark = pytest.mark.gpu

# one lane, a run, a block of four, eight blocks (the queues start), all
# resident waves' first runs at 5, 6 and 7 blocks on 256 compute units, and
# past them (the counters start)
SIZES = [1, 63, 64, 65, 255, 257, 1792, 1793, 2049, 327679, 327681, 393215, 393217, 458753, 600001]


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


@pytest.mark.parametrize("n", SIZES)
def test_every_record_of_a_stream(rtc, device, scene, n):
    sc, rays, hits, shadow, dark = scene
    out = rays[:n].copy()
    sc.intersect1M(out)
    assert len(mismatches(out, hits[:n])) == 0
    occ = shadow[:n].copy()
    sc.occluded1M(occ)
    assert len(mismatches(occ, dark[:n])) == 0


@pytest.mark.parametrize("n", [1, 65, 2049, 327681, 600001])
def test_every_record_through_an_instance(rtc, device, oracle, scene, n):
    sc, rays, _, _, _ = scene
    l2w = np.eye(4, 3, dtype=np.float32).reshape(12)
    l2w[9:12] = 0.5, 0.0, -0.25
    top = rtc.Scene(device)
    top.add_instance(sc, l2w)
    top.commit()
    out = rays[:n].copy()
    top.intersect1M(out)
    ref = rays[:n].copy()
    o = oracle.Instances()
    o.add_instance(o.add_object([rtc.gen_sphere(8)]), l2w, 0)
    o.intersect_bvh(ref)
    assert len(mismatches(out, ref)) == 0
    top.release()


@pytest.mark.parametrize("n", [65, 2049, 393217, 600001])
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
