"""SCBragg's Romberg queue (one wave per neutron, several of a narrow beam, or
one lane), its candidate lists and the family guide, at the sizes where they can go wrong, against the checker: cross
sections and samples on the same Philox streams."""
import math

import numpy as np
import pytest

from ncrystal_amd import synth
from conftest import assert_streams_match

pytestmark = pytest.mark.gpu
WL2EKIN = 0.081804209605330899


@pytest.fixture(scope="module")
def core():
    from ncrystal_amd import _capi, core
    if _capi.lib().ncamd_device_count() < 1:
        pytest.fail("no GPU visible to libncrystal_amd")
    return core


def _crystal(core, oracle, cr, mosaic_deg):
    sp = [(s.csl, oracle.debye_msd(s.debye_temp, cr.temperature, s.mass), s.positions) for s in cr.species]
    _, _, dsp, fsq, moff, mh = oracle.hkl_orthogonal_members(cr.a, cr.b, cr.c, sp, cr.dcutoff)
    v0n, R, mos = cr.volume * cr.n_atoms, synth.random_rotation(7), math.radians(mosaic_deg)
    L = core.reci_lattice_orthogonal(cr.a, cr.b, cr.c)
    return (core.create_scbragg(v0n, dsp, fsq, moff, mh, L, R, mos),
            oracle.scbragg(cr.a, cr.b, cr.c, v0n, dsp, fsq, moff, mh, R, mos), dsp)


def _compare(g, o, e, d, label):
    x, y = g.crossSection(e, d), o.xs_dir(e, d, nthreads=8)
    # the same arithmetic with the device's acos, sqrt and cosine in the circle
    # integral; its density has a logarithmic slope of 1/sigma^2 <= 2e4 here
    assert np.max(np.abs(x - y) / np.maximum(y, 1e-300)) < 1e-10
    assert np.array_equal(x == 0, y == 0)
    g.setRNGState(9, 0)
    ge, gd = g.sampleScatter(e, d)
    _, od, nerr = o.sample_dir(e, d, seed=9, nthreads=8)
    assert nerr == 0 and np.array_equal(ge, e)
    assert_streams_match(np.max(np.abs(gd - od), axis=1) > 1e-9, label)
    return x


@pytest.mark.parametrize("n", [1, 5, 700])
def test_backscattering_along_normals(core, oracle, n):
    """neutrons within the mosaic spread of backscattering: nearly all queued"""
    g, o, dsp = _crystal(core, oracle, synth.fcc_powder(dcutoff=0.4), 1.0)
    t = g.tables()
    rng = np.random.default_rng(n)
    f = rng.integers(0, len(t["inv2d"]), n)
    nrm = t["normals"][t["off"][f]]
    d = nrm + rng.normal(scale=3e-3, size=(n, 3))
    e = WL2EKIN / ((1.0 - 10.0 ** rng.uniform(-8, -4, n)) / t["inv2d"][f]) ** 2
    x = _compare(g, o, e, d, f"backscattering {n}")
    assert np.mean(x > 0) > 0.9


# a narrow beam near backscattering from one family: waves that take three
# neutrons and more, and lanes from 65536 queued ones on; wide: single ones at the
# same sizes.  5 degrees: more integrals in a batch of candidates than the wave
# does together.
@pytest.mark.parametrize("n,mosaic,spread", [(9001, 0.5, 0.3), (9001, 5.0, 0.3), (80001, 0.5, 0.3), (80001, 5.0, 0.3),
                                             (13001, 0.5, None)])
def test_many_queued(core, oracle, n, mosaic, spread):
    g, o, dsp = _crystal(core, oracle, synth.fcc_powder(dcutoff=0.7), mosaic)
    t = g.tables()
    rng = np.random.default_rng(n)
    f = rng.integers(0, len(t["inv2d"]), n) if spread is None else np.full(n, len(t["inv2d"]) // 3)
    d = t["normals"][t["off"][f]] + rng.normal(scale=(spread or 0.3) * math.radians(mosaic), size=(n, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    e = WL2EKIN / ((1.0 - 10.0 ** rng.uniform(-8, -4, n)) / t["inv2d"][f]) ** 2
    x = _compare(g, o, e, d, f"queued {n} {mosaic}")
    assert np.mean(x > 0) > 0.95
    g.setRNGState(9, 0)
    od = g.sampleScatter(e, d)[1]
    for m in (1, 700):  # a wave each: the same sums and integrals in the same order
        assert np.array_equal(g.crossSection(e[:m], d[:m]), x[:m])
        g.setRNGState(9, 0)
        assert np.array_equal(g.sampleScatter(e[:m], d[:m])[1], od[:m])


def test_long_lists(core, oracle):
    """0.25 Aa and 5 degrees: thousands of candidates per neutron, more than a
    wave's list"""
    g, o, _ = _crystal(core, oracle, synth.ortho_random(seed=2, dcutoff=0.45), 5.0)
    n = 24
    d = synth.isotropic_dirs(n, 4)
    t = g.tables()
    d[: n // 2] = t["normals"][t["off"][np.arange(n // 2) + len(t["inv2d"]) // 2]]
    e = np.full(n, WL2EKIN / 0.25 ** 2)
    e[: n // 2] = WL2EKIN / ((1 - 1e-6) / t["inv2d"][np.arange(n // 2) + len(t["inv2d"]) // 2]) ** 2
    _compare(g, o, e, d, "long lists")


def test_family_thresholds(core, oracle):
    """wavelengths at every family's 2d and one rounding either side, beyond
    the last family and above the threshold"""
    g, o, dsp = _crystal(core, oracle, synth.ortho_random(seed=3, dcutoff=0.8), 0.5)
    wl = 2.0 * dsp
    e = WL2EKIN / wl ** 2
    e = np.concatenate([e, np.nextafter(e, 0), np.nextafter(e, 9), e * (1 + 1e-12), [1e-7, 1e3, 1e9]])
    x, y = (c(e, synth.isotropic_dirs(e.size, 8)) for c in (g.crossSection, o.xs_dir))
    assert np.max(np.abs(x - y) / np.maximum(y, 1e-300)) < 1e-10 and np.array_equal(x == 0, y == 0)
