"""The packet gather (gather mode 7) at the sizes where its stages, windows,
groups and tie handling change, on caller-given photon maps, against the
8-byte heap gather (mode 1), which keeps exact (d^2, index) keys and shares
none of the search with it (both use the FP64 sums and the phase function).
Both sum a query's neighbours in FP64, so a query's FP32
sum differs by at most its last bit between them, and a pixel's radiance (a
sum of non-negative terms, each off by at most 2^-23 of itself, and the
rounding of the sums) by less than 5e-7 of itself.
"""
import ctypes
import sys

import numpy as np
import pytest

import pmamd

pytestmark = pytest.mark.gpu

RTOL = 5e-7


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def volume_points(rng, layout, n):
    if layout == "uniform":
        return rng.random((n, 3), dtype=np.float32)
    if layout == "coincident":  # 50 photons at each place: counters wrap, ties go by index
        return np.repeat(rng.random((n // 50, 3), dtype=np.float32), 50, axis=0)
    if layout == "lattice":  # many equal distances
        m = int(round(n ** (1.0 / 3.0)))
        g = (np.indices((m, m, m)).reshape(3, -1).T + 0.5) / m
        return g.astype(np.float32)
    # nine in ten inside a small ball in view: stages overflow, groups split
    p = rng.random((n, 3), dtype=np.float32)
    d = rng.normal(size=(n, 3))
    ball = 0.5 + 0.02 * d / np.linalg.norm(d, axis=1, keepdims=True) * rng.random((n, 1)) ** (1.0 / 3.0)
    inside = np.arange(n) % 10 != 0
    p[inside] = ball[inside].astype(np.float32)
    return p


def wall_points(rng, layout, n):
    p = volume_points(rng, layout, n)
    w = np.arange(len(p)) % 5
    p[np.arange(len(p)), np.array([0, 0, 1, 1, 2])[w]] = np.array([0, 1, 0, 1, 1], np.float32)[w]
    return p


CASES = [
    # layout, photons, leaf, k, cap, spp, width, height, spheres
    ("uniform", 1, 32, 32, 0.05, 1, 33, 17, 2),
    ("uniform", 64, 64, 64, 3.0, 1, 9, 7, 2),  # exactly k points, one leaf, all in reach
    ("uniform", 65, 64, 64, 3.0, 1, 9, 7, 2),
    ("uniform", 5000, 1, 1, 0.05, 1, 40, 24, 2),
    ("uniform", 5001, 7, 33, 0.2, 3, 24, 16, 2),
    ("uniform", 40000, 52, 64, 0.5, 4, 24, 16, 2),
    ("uniform", 40000, 64, 64, 0.03, 16, 7, 5, 2),
    ("uniform", 200000, 32, 32, 0.05, 2, 19, 11, 200),  # queries far apart: many groups
    ("coincident", 20000, 32, 32, 0.2, 1, 24, 16, 2),
    ("coincident", 20000, 16, 64, 0.2, 4, 12, 8, 2),
    ("lattice", 27000, 32, 64, 0.2, 1, 24, 16, 2),
    ("dense", 200000, 52, 64, 0.1, 4, 24, 16, 2),
    ("dense", 200000, 8, 64, 0.5, 1, 24, 16, 2),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c[:7]))
def test_packet_equals_heap_gather(case):
    layout, n, leaf, k, cap, spp, w, h, spheres = case
    say("case: packet gather, %s, n=%d, leaf=%d, k=%d, r<=%g, %dx%dx%d" % (layout, n, leaf, k, cap, w, h, spp))
    c = pmamd.batch_scene(3, 5) if spheres > 2 else pmamd.preset(1)
    c.leaf_size = leaf
    c.k_surface = c.k_volume = k
    c.rcap_surface = c.rcap_volume = cap
    c.width, c.height, c.spp = w, h, spp
    c.medium, c.sigma_s, c.sigma_a, c.hg_g = pmamd.PM_MEDIUM_HOMOGENEOUS, 0.1, 0.01, 0.6
    rng = np.random.default_rng(11)
    g = pmamd.PhotonMapper(c)
    for which, pos in ((pmamd.PM_MAP_SURFACE, wall_points(rng, layout, n)),
                       (pmamd.PM_MAP_VOLUME, volume_points(rng, layout, n))):
        d = rng.normal(size=pos.shape)
        d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
        g.set_records(which, pos, rng.uniform(0.5, 1.5, pos.shape).astype(np.float32), d, 2 * n)
    g.build()
    g.set_option(pmamd.PM_OPT_GATHER_MODE, 1)
    ref = g.render()
    rq = g.stats()
    g.set_option(pmamd.PM_OPT_GATHER_MODE, 7)
    img = g.render()
    q = g.stats()
    assert (q.surface_queries, q.volume_queries) == (rq.surface_queries, rq.volume_queries)
    assert q.volume_queries > 0 and (n < 100 or ref.max() > 0)
    np.testing.assert_allclose(img, ref, rtol=RTOL, atol=0)
    g.close()


@pytest.mark.parametrize("storage", [pmamd.PM_STORE_FP32, pmamd.PM_STORE_BF16])
@pytest.mark.parametrize("mode", [0, 1, 2, 4, 7])
def test_directions_longer_than_one_have_no_weight(mode, storage):
    """At g = 0.99 a photon that travels 1.05 long along the view direction has
    1 + g^2 - 2 g cos = -0.1: no phase function, and no weight in the sum.  A
    view that meets no other photons is black."""
    say("case: directions of length 1.05, g = 0.99, gather mode %d, storage %d" % (mode, storage))
    c = pmamd.preset(1)
    c.n_spheres = 0
    c.width, c.height, c.focal, c.storage = 8, 8, 50.0, storage
    c.medium, c.sigma_s, c.sigma_a, c.hg_g = pmamd.PM_MEDIUM_HOMOGENEOUS, 0.1, 0.01, 0.99
    rng = np.random.default_rng(3)
    pos = rng.random((20000, 3), dtype=np.float32)
    none = np.zeros((0, 3), np.float32)
    g = pmamd.PhotonMapper(c)
    g.set_records(pmamd.PM_MAP_SURFACE, none, none, none, 1)
    g.set_records(pmamd.PM_MAP_VOLUME, pos, np.ones_like(pos), np.tile(np.float32([0, 0, -1.05]), (len(pos), 1)), 1)
    g.build()
    g.set_option(pmamd.PM_OPT_GATHER_MODE, mode)
    img = g.render()
    assert g.stats().volume_queries > 0
    assert np.array_equal(img, np.zeros_like(img)), img.max()
    g.close()


# photons, k, cap, width, height, spp, march; the faster gather is 2 to 12 times the other
AUTO_CASES = [
    (1000, 32, 0.005, 256, 256, 1, 1),    # balls below a march step in an empty map: heap
    (20000, 8, 0.004, 440, 220, 1, 1),
    (20000, 32, 0.05, 64, 48, 1, 1),      # few waves: packet, march steps in lanes
    (100000, 32, 0.05, 256, 256, 1, 1),
    (20000, 4, 0.15, 640, 360, 4, 1),
    (20000, 32, 0.05, 640, 360, 1, 0),    # surface hits: a search per wave and no seed
    (100000, 32, 0.02, 960, 540, 1, 0),   # full balls, the cap close to them
    (100000, 16, 0.4, 200, 150, 1, 0),
    (100000, 1, 0.1, 256, 256, 1, 0),
    (100000, 64, 0.03, 640, 360, 4, 0),   # samples in lanes
]


@pytest.mark.parametrize("case", AUTO_CASES, ids=lambda c: "-".join(str(v) for v in c))
def test_auto_takes_the_faster_gather(case):
    photons, k, cap, w, h, spp, march = case
    say("case: gather mode of auto, %d photons, k=%d, r<=%g, %dx%dx%d, march %d" % case)
    c = pmamd.preset(1)
    c.n_emit, c.k_surface, c.k_volume, c.rcap_surface, c.rcap_volume = photons, k, k, cap, cap
    c.width, c.height, c.spp = w, h, spp
    g = pmamd.PhotonMapper(c)
    g.emit()
    g.build()
    g.set_option(pmamd.PM_OPT_RENDER_MEDIA, march)
    img, ms = {}, {}
    for mode in (1, 7, 5):
        g.set_option(pmamd.PM_OPT_GATHER_MODE, mode)
        for _ in range(4):
            img[mode] = g.render()
            ms[mode] = min(ms.get(mode, 1e9), g.stats().ms_render)
    say("ms: heap %.3f, packet %.3f, auto %.3f" % (ms[1], ms[7], ms[5]))
    # the two differ by twice and more; the margin is for the clock
    assert ms[5] < 1.4 * min(ms[1], ms[7]) + 0.02
    assert np.array_equal(img[5], img[1]) or np.array_equal(img[5], img[7])
    g.close()


def test_default_of_a_sparse_batch_is_a_heap():
    """A batch whose balls hold nothing is not given to the packet gather, the
    batched workload's scenes are."""
    say("case: default tuning of two batches")
    for cap, mode in ((0.004, 0), (0.05, 7)):
        cfgs = []
        for i in range(3):
            c = pmamd.batch_scene(5, i)
            c.n_emit, c.width, c.height = 3000, 300, 280 + i
            c.rcap_surface = c.rcap_volume = cap
            c.medium, c.sigma_s, c.sigma_a = pmamd.PM_MEDIUM_HOMOGENEOUS, 0.1, 0.01
            cfgs.append(c)
        b = pmamd.Batch(cfgs)
        assert b.stats().tuning.gather_mode == mode
        b.submit()
        imgs = [b.image(i) for i in range(3)]
        b.set_tuning(32, 64, 64, 2, 7 - mode, 0)
        b.submit()
        for i in range(3):
            np.testing.assert_allclose(b.image(i), imgs[i], rtol=RTOL, atol=0)


def test_cache_values_of_sparse_maps():
    """Auto gathers a cache frame's exact values with the heap where hardly any
    record has a photon within the cap (the packet gather: 2.5 to 5 times its
    time), and gives the same frame."""
    say("case: cache frame, 640x360, r <= 0.003, every record gathered")
    c = pmamd.preset(1)
    c.n_emit, c.width, c.height = 3000, 640, 360
    c.rcap_surface = c.rcap_volume = 0.003
    g = pmamd.PhotonMapper(c)
    g.emit()
    g.build()
    img, ms = {}, {}
    for mode in (1, 7, 5):
        g.cache_reset(1)
        g.cache_configure(threshold=0.0, train_samples=1 << 14, batch=1 << 14)
        g.set_option(pmamd.PM_OPT_GATHER_MODE, mode)
        for _ in range(4):
            img[mode] = g.render_cache()
            ms[mode] = min(ms.get(mode, 1e9), g.cache_stats().ms_fallback)
    say("ms of the exact values: heap %.3f, packet %.3f, auto %.3f" % (ms[1], ms[7], ms[5]))
    assert ms[5] < 1.4 * min(ms[1], ms[7]) + 0.02
    np.testing.assert_allclose(img[5], img[7], rtol=RTOL, atol=0)
    g.close()


def free_device_bytes():
    pmamd.load().pm_device_free(None)  # the runtime is up
    with open("/proc/self/maps") as f:  # the HIP runtime that libpm.so is linked to
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_work_list_memory_does_not_grow_with_the_frame():
    """Only launches of fewer tiles than 64 a CU use the work list (0.3 MB), so
    an 8192x8192 frame reserves no more for it: its build takes the trees of a
    thousand photons and that list."""
    say("case: device memory of a build, 8192x8192 frame")
    c = pmamd.preset(1)
    c.n_emit, c.width, c.height = 1000, 8192, 8192
    g = pmamd.PhotonMapper(c)
    g.emit()
    before = free_device_bytes()
    g.build()
    assert before - free_device_bytes() < 64 << 20
    # and a window of it renders from the list as ever
    g.set_option(pmamd.PM_OPT_GATHER_MODE, 7)
    a = g.render(4000, 4000, 64, 48)
    before = free_device_bytes()
    g.render(0, 0, 2048, 2048)
    assert before - free_device_bytes() < (2048 * 2048 * 12) + (16 << 20)  # the caller's image
    assert np.array_equal(a, g.render(4000, 4000, 64, 48))
    g.close()


def test_dense_windows_end_on_split_tiles():
    """Around the light of the fog scene a window of one sample a pixel is done
    in less time than one of four, and three in a lane's loop in less than twice
    theirs: without the heavy tiles first and in quarters, 1.1 and 3.3 times."""
    say("case: 480x270 window of the fog at 1, 3 and 4 samples")
    c = pmamd.preset(2)
    g = pmamd.PhotonMapper(c)
    g.emit()
    g.build()
    ms = {}
    for spp in (1, 3, 4):
        g.set_render(c.width, c.height, spp, c.k_surface, c.k_volume, c.rcap_surface, c.rcap_volume)
        for _ in range(3):
            g.render(720, 405, 480, 270)
            ms[spp] = min(ms.get(spp, 1e9), g.stats().ms_render)
    say("ms: %s" % ms)
    assert ms[1] < 0.75 * ms[4] and ms[3] < 2 * ms[4]
    g.close()


def test_cache_frames_of_growing_size():
    """A cache frame is the same after a smaller and a larger frame as in a new
    context: the records' buffers grow and keep nothing."""
    say("case: cache frames of 1, 4 and 2 samples in one context and alone")
    c = pmamd.preset(1)
    c.n_emit, c.width, c.height = 20000, 96, 64
    g = pmamd.PhotonMapper(c)
    g.emit()
    g.build()
    for spp in (1, 4, 2):
        imgs = []
        for own in (g, pmamd.PhotonMapper(c)):
            if own is not g:
                own.emit()
                own.build()
            own.set_render(96, 64, spp, c.k_surface, c.k_volume, c.rcap_surface, c.rcap_volume)
            own.cache_reset(1)
            own.cache_configure(threshold=0.05, train_samples=1 << 14, batch=1 << 12)
            imgs.append(own.render_cache())
        np.testing.assert_allclose(imgs[0], imgs[1], rtol=RTOL, atol=0)


def test_batch_that_fits_only_without_the_payload_copy():
    """The packet gather's copy of the payloads (32 bytes a record) is what a
    batch can do without: where it does not fit beside the rest, the batch starts
    with a heap, renders, refuses the packet gather without harm, and the
    autotuner chooses among the heaps."""
    cfgs = []
    for i in range(16):
        c = pmamd.batch_scene(5, i)
        c.n_emit, c.width, c.height = 2000000, 64, 64
        c.medium, c.sigma_s, c.sigma_a = pmamd.PM_MEDIUM_HOMOGENEOUS, 0.1, 0.01
        cfgs.append(c)
    before = free_device_bytes()
    b = pmamd.Batch(cfgs)
    used = before - free_device_bytes()
    st = b.stats()
    copy = 32 * (st.surface_records + st.volume_records)
    say("case: batch of %.1f GB, payload copy %.1f GB" % (used / 2**30, copy / 2**30))
    assert st.tuning.gather_mode == 7 and copy > 2 << 30
    b.submit()
    img = b.image(3)
    b.close()
    filler = pmamd.DeviceBuffer(free_device_bytes() - used + copy // 2)
    try:
        b = pmamd.Batch(cfgs)
        assert b.stats().tuning.gather_mode == 0
        # refused at the same and at another leaf size, whose forest fits
        for leaf in (32, 16):
            with pytest.raises(pmamd.PmError):
                b.set_tuning(leaf, 64, 64, 2, 7, 0)
            b.submit()
            np.testing.assert_allclose(b.image(3), img, rtol=RTOL, atol=0)
        best, _ = b.autotune(sample_stride=3)
        assert best[4] == 0 and b.stats().tuning.gather_mode == 0
        # a forest that does not fit: leaves of 2 give 47 million nodes of 48 bytes
        b.set_tuning(32, 64, 64, 2, 0, 0)
        rest = pmamd.DeviceBuffer(free_device_bytes() - (256 << 20))
        with pytest.raises(pmamd.PmError):
            b.set_tuning(2, 64, 64, 2, 0, 0)
        rest.free()
        assert b.stats().tuning.leaf_size == 32
        b.submit()
        np.testing.assert_allclose(b.image(3), img, rtol=RTOL, atol=0)
        b.close()
    finally:
        filler.free()
