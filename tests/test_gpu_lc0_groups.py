"""Layered-crystal kernel (lcmode=0) at the edges of its work split: the
neutrons per workgroup follow from the batch size, the ranges are integrated in
rounds of a workgroup's list, and sampling finds its range in the round or, for
more plane sets than a round's masks hold, in a second pass.  None of that may
change a neutron's value."""
import math

import numpy as np
import pytest

from test_lcbragg_checker import FIX, WL2EKIN, checker_crystal, graphite_inputs, lchelper

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def core():
    from ncrystal_amd import _capi, core
    if _capi.lib().ncamd_device_count() < 1:
        pytest.fail("no GPU visible to libncrystal_amd")
    return core


def _layered(core, dcutoff, mosaic):
    def msd(e, d, T, m):
        return core.vdos_analyse((e, d), T, m)["msd"]
    cell, sp, v0n = graphite_inputs(msd)
    _, _, dsp, fsq, moff, mh = core.hkl_spacegroup_members(FIX["spacegroup"], cell, sp, dcutoff)
    return core.create_lcbragg(v0n, dsp, fsq, moff, mh, core.reci_lattice(cell), np.eye(3), FIX["lcaxis"],
                               math.radians(mosaic))


def _neutrons(n, lo, hi, seed):
    rng = np.random.default_rng(seed)
    d = rng.normal(size=(n, 3))
    return WL2EKIN / rng.uniform(lo, hi, n) ** 2, d / np.linalg.norm(d, axis=1)[:, None]


# 0.5-0.7 Aa: all plane sets in reach, several rounds per workgroup and, at 5
# degrees, ranges with backscattering points; 2.2-7 Aa: mostly none or a few
@pytest.mark.parametrize("lo,hi,mosaic", [(0.5, 0.7, 1.0), (0.5, 0.7, 5.0), (2.2, 7.0, 4.0)])
def test_batch_size_changes_nothing(core, lo, hi, mosaic):
    lc = _layered(core, 0.5, mosaic)
    n = 33000  # 64 neutrons per workgroup; the calls below use 4, 8, 16 and 32
    e, d = _neutrons(n, lo, hi, 3)
    xs = lc.crossSection(e, d)
    lc.setRNGState(17, 0)
    oe, od = lc.sampleScatter(e, d)
    assert np.array_equal(oe, e) and np.allclose(np.linalg.norm(od, axis=1), 1.0, atol=1e-12)
    for m in (1, 3, 63, 65, 2049, 5000, 9001, 20000):
        assert np.array_equal(lc.crossSection(e[:m], d[:m]), xs[:m])
        lc.setRNGState(17, 0)
        assert np.array_equal(lc.sampleScatter(e[:m], d[:m])[1], od[:m])


# workgroups of 128 and 256 neutrons: all beyond the last wavelength, around it,
# with the first plane set alone, with a few, and every kind mixed
@pytest.mark.parametrize("n", [262147, 2097157])
@pytest.mark.parametrize("lo,hi", [(6.9, 9.0), (6.6, 6.8), (4.3, 6.0), (3.0, 4.0), (1.0, 9.0)])
def test_sparse_batches(core, n, lo, hi):
    lc = _layered(core, 0.5, 4.0)
    e, d = _neutrons(n, lo, hi, 11)
    d[:64] = [0.0, 0.0, 1.0]  # along the axis
    e[100:110] = [0.0, -1.0, np.inf, np.nan, 1e-9, 1e3, 0.0, np.nan, -0.0, 1e-300]
    xs = lc.crossSection(e, d)
    lc.setRNGState(17, 0)
    oe, od = lc.sampleScatter(e, d)
    assert np.array_equal(oe, e, equal_nan=True)
    none = ~(e > WL2EKIN / 6.8 ** 2)  # the largest 2d is 6.71 Aa
    assert np.all(xs[none] == 0.0) and np.array_equal(od[none], d[none])
    for m in (130, 4999, 40000):  # 4, 8 and 64 neutrons per workgroup
        assert np.array_equal(lc.crossSection(e[:m], d[:m]), xs[:m], equal_nan=True)
        lc.setRNGState(17, 0)
        assert np.array_equal(lc.sampleScatter(e[:m], d[:m])[1], od[:m], equal_nan=True)
    k = n - 4000  # the batch's end
    assert np.array_equal(lc.crossSection(e[k:], d[k:]), xs[k:], equal_nan=True)


def test_more_plane_sets_than_a_round(core, oracle):
    """dcutoff 0.2 Aa gives the crystal over 256 plane sets; neutrons that
    reach only those down to 0.5 Aa see the same crystal as without the rest
    (same sums: identical), others are compared with the checker"""
    small, large = _layered(core, 0.5, 4.0), _layered(core, 0.2, 4.0)
    e, d = _neutrons(3000, 1.01, 3.0, 5)
    assert np.array_equal(small.crossSection(e, d), large.crossSection(e, d))
    for lc in (small, large):
        lc.setRNGState(4, 0)
    assert np.array_equal(small.sampleScatter(e, d)[1], large.sampleScatter(e, d)[1])
    o, fam = checker_crystal(oracle, 0.2)
    e, d = _neutrons(40, 0.41, 0.6, 6)
    got, want = large.crossSection(e, d), lchelper(oracle, o, fam).xs_dir(e, d)
    # the bound of the checker comparison of this model: device cosines in
    # ranges that lose up to 1e5 of their argument's precision
    assert np.max(np.abs(got - want) / want) < 1e-10
    gd = large.sampleScatter(e, d)[1]
    assert np.allclose(np.linalg.norm(gd, axis=1), 1.0, atol=1e-12)


def test_more_neutrons_than_a_grid(core):
    """2^30 neutrons and some: beyond what one launch takes at 256 work-items
    per 64 neutrons.  All but a few have zero energy (no scattering); the few,
    around the places where launches meet and at the end, get the values of a
    small call, and equal neutrons in different launches draw different numbers."""
    from ncrystal_amd import _capi as C
    lc = _layered(core, 0.5, 4.0)
    n, part, k = 2 ** 30 + 65, 2 ** 28, 40
    e, d = _neutrons(k, 0.6, 2.0, 7)
    xs = lc.crossSection(e, d)
    de, dd, o1, o2 = C.DeviceArray(n), C.DeviceArray(3 * n), C.DeviceArray(n), C.DeviceArray(3 * n)
    put = lambda a, i, x: C.call("ncamd_memcpy_htod", a.ptr + 8 * i, x.ctypes.data, 8 * x.size)

    def get(a, i, m):
        x = np.empty(m)
        C.call("ncamd_memcpy_dtoh", x.ctypes.data, a.ptr + 8 * i, 8 * m)
        return x

    zero = np.zeros(2 ** 25)
    for i in range(0, n, zero.size):
        put(de, i, zero[:min(zero.size, n - i)])
    at = [0, part - k // 2, 2 * part + k, 2 ** 30 - k // 2, n - k]
    for i in at:
        put(de, i, e)
        put(dd, 3 * i, d)
    lc.dev_crossSection(de.ptr, dd.ptr, n, o1.ptr)
    C.call("ncamd_stream_sync", None)
    for i in at:
        assert np.array_equal(get(o1, i, k), xs)
    for i in (k, part - k, part + k, 3 * part, 2 ** 30 - k):  # (up to the window after it)
        assert not get(o1, i, k // 2).any()
    lc.setRNGState(5, 0)
    lc.dev_sampleScatter(de.ptr, dd.ptr, n, o1.ptr, o2.ptr)
    C.call("ncamd_stream_sync", None)
    got = [get(o2, 3 * i, 3 * k).reshape(-1, 3) for i in at]
    lc.setRNGState(5, 0)
    assert np.array_equal(got[0], lc.sampleScatter(e, d)[1])
    for a in range(len(at)):
        assert np.array_equal(get(o1, at[a], k), e)
        assert np.allclose(np.linalg.norm(got[a], axis=1), 1.0, atol=1e-12)
        for b in range(a):
            assert np.any(got[a][xs > 0] != got[b][xs > 0])
