"""The packet gather (mode 7) on emitted photon maps against the 8-byte heap
gather (mode 1), over what its launches vary in: samples in lanes or in the
wave's loop, the cone estimate, FP64 transmittance, BF16 payloads, the density
field and the homogeneous medium; and PM_OPT_TOP_LEVELS, which is accepted in
its range and has no effect.
"""
import sys

import numpy as np
import pytest

import pmamd

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


# Both sum a query's neighbours in FP64 and round once, and a pixel adds terms
# of one sign: its value is off by less than 5e-7 of itself between the two.
RTOL = 5e-7
# The cone filter's weights are 1 - x with x = d / (1.1 r) in [0, 0.91].  Mode 1
# rounds each x three times and 1.1 once (2.0e-7 of it) and the difference once;
# the packet gather rounds its two sums, 1.1, the product and the quotient
# (2.4e-7 of the power).  Together 4.5e-7 of the summed power, which is at most
# 11 times the summed weight x power.
RTOL_CONE = 11 * 4.5e-7 + RTOL


@pytest.mark.parametrize("medium", ["noise", "homogeneous"])
@pytest.mark.parametrize("variant", ["lanes", "loop", "cone", "fp64", "bf16"])
def test_packet_equals_heap_gather_on_emitted_maps(variant, medium):
    say("case: packet and heap gather, preset 2 reduced, %s, %s medium" % (variant, medium))
    c = pmamd.preset(2)
    c.cap_surface, c.cap_volume = 60000, 40000
    c.width, c.height, c.spp = 96, 64, 4
    if medium == "homogeneous":
        c.medium, c.sigma_s, c.sigma_a = pmamd.PM_MEDIUM_HOMOGENEOUS, 0.1, 0.01
    if variant == "cone":
        c.estimator = pmamd.PM_EST_CONE
    if variant in ("fp64", "bf16"):
        c.fp64_transmittance = 1
    if variant == "bf16":
        c.storage = pmamd.PM_STORE_BF16
    g = pmamd.PhotonMapper(c)
    g.emit()
    g.build()
    g.set_option(pmamd.PM_OPT_GATHER_MODE, 1)
    ref = g.render()
    rs = g.stats()
    g.set_option(pmamd.PM_OPT_GATHER_MODE, 7)
    g.set_option(pmamd.PM_OPT_SAMPLE_LANES, 0 if variant == "loop" else 1)
    img = g.render()
    s = g.stats()
    assert (s.surface_queries, s.volume_queries) == (rs.surface_queries, rs.volume_queries)
    assert s.volume_queries > 0
    np.testing.assert_allclose(img, ref, rtol=RTOL_CONE if variant == "cone" else RTOL, atol=0)
    g.close()


def test_top_levels_have_no_effect():
    say("case: PM_OPT_TOP_LEVELS")
    c = pmamd.preset(1)
    c.n_emit, c.width, c.height = 20000, 48, 32
    g = pmamd.PhotonMapper(c)
    g.emit()
    g.build()
    ref = g.render()
    g.set_option(pmamd.PM_OPT_TOP_LEVELS, 7)
    assert np.array_equal(bits(g.render()), bits(ref))
    with pytest.raises(pmamd.PmError):
        g.set_option(pmamd.PM_OPT_TOP_LEVELS, 8)
    g.close()


def test_option_ranges():
    """The options added beside the gather modes take only their documented values."""
    c = pmamd.preset(1)
    c.n_emit = 1000
    g = pmamd.PhotonMapper(c)
    for opt, bad in ((pmamd.PM_OPT_TOP_LEVELS, -1), (pmamd.PM_OPT_VOXEL_GRID, 3), (pmamd.PM_OPT_CACHE_NEAR_GROUPS, 17),
                     (pmamd.PM_OPT_CACHE_EMA, 1000), (pmamd.PM_OPT_CACHE_EMA, -1), (pmamd.PM_OPT_CACHE_SEEDS, 2),
                     (99, 0)):
        with pytest.raises(pmamd.PmError):
            g.set_option(opt, bad)
    for opt, ok in ((pmamd.PM_OPT_TOP_LEVELS, 7), (pmamd.PM_OPT_VOXEL_GRID, 2), (pmamd.PM_OPT_CACHE_NEAR_GROUPS, 0),
                    (pmamd.PM_OPT_CACHE_EMA, 0), (pmamd.PM_OPT_CACHE_EMA, 999), (pmamd.PM_OPT_CACHE_SEEDS, 0),
                    (pmamd.PM_OPT_CACHE_SEEDS, 1)):
        g.set_option(opt, ok)
    g.close()
