"""Builds that share a device's scratch memory with other threads' builds,
the walk of a tree whose top has nearly as many subtrees as there is room for,
commits that the memory monitor refuses, and what HIGH commits keep."""
import ctypes
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


def clusters():
    """The centres of 250 clusters on a grid, and a mesh of them: dense ones, each
    with three small groups beside it that a split takes off first."""
    rng = np.random.default_rng(9)
    x = np.array([0, 1, 3, 4, 9, 10, 12, 13])  # (pairs, pairs of pairs, ...: every split lies between clusters)
    at = np.stack(np.meshgrid(x, x, x[:4], indexing="ij"), -1).reshape(-1, 3)[:250]
    beside = np.array([[0.25, 0.0, 0.0], [0.0, 0.25, 0.0], [-0.2, 0.0, 0.2]])
    parts = []
    for c in at:
        parts.append(c + (rng.random((2380, 3)) - 0.5) * 0.01)
        for b in beside:
            parts.append(c + b + (rng.random((12, 3)) - 0.5) * 0.005)
    p = np.concatenate(parts)
    v = p[:, None, :] + (rng.random((len(p), 3, 3)) - 0.5) * 0.002
    return at, v.reshape(-1, 3).astype(np.float32), np.arange(3 * len(p), dtype=np.uint32).reshape(-1, 3)


def walk(nodes, tris):
    """The level sizes of the tree's top and the subtrees there are before each,
    as the collapse walks it (nodes of more than a 256th of the primitives, and
    of more than 2048, are walked; the others are subtrees)."""
    N = nodes.reshape(-1, 80)
    base = N[:, 16:24].copy().view(np.uint32)
    flags = tris.view(np.uint32).reshape(-1, 12)[:, 11]
    ends = np.nonzero(flags & 1)[0]
    n = len(flags)
    size = np.zeros(len(N), np.int64)
    kids = []
    for i in range(len(N) - 1, -1, -1):  # (children follow their parents)
        k = []
        for m in N[i, 24:32]:
            if m & 0x80:
                k.append(int(base[i, 0]) + int(m & 0x7f))
                size[i] += size[k[-1]]
            elif m:
                first = int(base[i, 1]) + int(m) - 1
                size[i] += ends[np.searchsorted(ends, first)] - first + 1
        kids.append(k)
    kids.reverse()
    assert size[0] == n
    share = max(n // 256, 2048)
    level, subs, out = [0], 0, []
    while level:
        out.append((len(level), subs))
        children = [c for i in level for c in kids[i]]
        level = [c for c in children if size[c] > share]
        subs += len(children) - len(level)
    return out + [(0, subs)]


def test_top_walk_near_its_room_for_subtrees(rtc, oracle):
    room = 2047  # subtrees of a build of one scene
    dev = rtc.Device("bvh_width=2")
    at, v, ix = clusters()
    sc = rtc.Scene(dev, [(v, ix)]).commit()
    nodes, tris = sc.read_bvh()
    levels = walk(nodes, tris)
    # a level that is walked, while its own subtrees leave too little room for as many again
    assert any(subs + 8 * count <= room < then + 8 * count for (count, subs), (_, then) in zip(levels, levels[1:])), levels
    # and one that is left as subtrees
    assert any(count and subs + 8 * count > room for count, subs in levels), levels
    prims = tris.view(np.uint32).reshape(-1, 12)[:, 3]
    assert np.array_equal(np.sort(prims), np.arange(len(ix)))
    rays = rtc.gen_random_rays(50000, seed=6, lo=0.0, hi=13.0)
    rng = np.random.default_rng(10)
    to = at[rng.integers(len(at), size=len(rays))] + (rng.random((len(rays), 3)) - 0.5) * 0.01
    for k, axis in enumerate("xyz"):
        rays[f"dir_{axis}"] = to[:, k] - rays[f"org_{axis}"]
    want, out = rays.copy(), rays.copy()
    oracle.BVH([(v, ix)]).intersect(want)
    sc.intersect1M(out)
    assert (want["geomID"] == 0).sum() > 10000
    assert len(mismatches(out, want)) == 0
    sc.release()
    dev.release()


def test_refused_commits_keep_no_memory(rtc):
    # the memory monitor refuses every other commit at its first, second, ... call
    dev = rtc.Device("")
    L = rtc.lib()
    hip = ctypes.CDLL("libamdhip64.so")
    left = [0]

    @ctypes.CFUNCTYPE(ctypes.c_bool, ctypes.c_void_p, ctypes.c_ssize_t, ctypes.c_bool)
    def monitor(_, size, post):
        left[0] -= 1
        return left[0] != 0

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    L.rtcSetDeviceMemoryMonitorFunction(dev.h, monitor, None)
    sc = rtc.Scene(dev, [rtc.gen_soup(200000, seed=k) for k in range(3)]).commit()
    start = None
    for refused in (1, 2, 3, 1, 2, 3, 1, 2, 3):
        left[0] = refused
        L.rtcCommitScene(sc.h)
        assert L.rtcGetDeviceError(dev.h) == rtc.RTC_ERROR_OUT_OF_MEMORY
        left[0] = 0
        sc.commit()
        start = start or free()
    assert start - free() < 8 << 20  # (a mesh's buffers are 10 MB)
    sc.release()
    dev.release()


def test_high_commits_give_the_other_tree_back(rtc):
    # what a device keeps after a HIGH commit of a large mesh is what a MEDIUM
    # commit of as many references keeps, and the split's own scratch
    hip = ctypes.CDLL("libamdhip64.so")

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    def kept(n, quality):
        dev = rtc.Device("")
        sc = rtc.Scene(dev, [rtc.gen_soup(n, seed=1, h=0.02)], quality=quality).commit()
        sc.release()
        before = free()
        dev.release()
        return free() - before

    n = 3000000
    high = kept(n, rtc.RTC_BUILD_QUALITY_HIGH)
    # (at most 1.3 n references are built over, and 48 bytes a triangle are the split's)
    medium = kept(int(1.3 * n), rtc.RTC_BUILD_QUALITY_MEDIUM)
    assert high < medium + 48 * n + (200 << 20)  # (a second tree has 208 bytes a triangle, 620 MB)
