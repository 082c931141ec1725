"""PowderBragg's search guides: plane lookups and picks equal, to the last bit,
to plain binary searches over the same tables, for few and many planes, equal
and widely uneven spacings and contributions, and energies at the thresholds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def core():
    from ncrystal_amd import _capi, core
    if _capi.lib().ncamd_device_count() < 1:
        pytest.fail("no GPU visible to libncrystal_amd")
    return core


def _planes(n, kind, rng):
    if kind == "dense":       # a crystal's density of planes
        d = (1000.0 - rng.uniform(size=n) * 999.9) ** (-1.0 / 3.0)
        f = rng.uniform(0.01, 5.0, size=n)
    elif kind == "wide":      # 12 decades of energy, all planes in few buckets
        d = 10.0 ** rng.uniform(-3, 3, size=n)
        f = 10.0 ** rng.uniform(-12, 0, size=n)
    else:                     # clusters, zero contributions, one dominant plane
        d = np.where(rng.uniform(size=n) < 0.5, 2.0, 0.7) * (1.0 + 1e-9 * rng.permutation(n))
        f = np.where(rng.uniform(size=n) < 0.5, 0.0, 1.0)
        f[n // 2] = 1e6
    return np.sort(d)[::-1].copy(), f


@pytest.mark.parametrize("kind", ["dense", "wide", "clusters"])
@pytest.mark.parametrize("n", [1, 2, 65, 5000, 40000])
def test_lookup_and_pick(core, oracle, n, kind):
    rng = np.random.default_rng(n)
    p = core.create_powderbragg(3000.0, *_planes(n, kind, rng), fp32_tables=False)
    e2d, fdm, _ = core.powderbragg_tables(p)
    at = e2d[rng.integers(0, len(e2d), 600)]
    e = np.concatenate([at, np.nextafter(at, 0), np.nextafter(at, np.inf), e2d[:1], e2d[-1:], 2 * e2d[-1:],
                        e2d[0] * (e2d[-1] / e2d[0]) ** rng.uniform(size=1500), [0.0, 1e-30, 1e300, np.inf]])
    idx = np.searchsorted(e2d, e, side="right") - 1
    on = (idx >= 0) & np.isfinite(e)
    xs = np.where(on, fdm[idx] * (1.0 / np.where(on, e, 1.0)), 0.0)
    assert np.array_equal(p.crossSectionIsotropic(e), xs)
    p.setRNGState(5, 0)
    ge, mu = p.sampleScatterIsotropic(e)
    u = np.array([oracle.rng_fill(5, 0, i, 1)[0] for i in range(len(e))])
    pick = np.searchsorted(fdm, u * fdm[idx])
    ref = np.where(on, 1.0 - 2.0 * (e2d[np.minimum(pick, len(e2d) - 1)] / np.where(on, e, 1.0)), 1.0)
    assert np.array_equal(ge, e) and np.array_equal(mu, ref)


def test_batches_beyond_the_last_level_cache(core):
    """17e6 neutrons, 272 MB and 408 MB of arrays, pass by the caches: the values of
    smaller calls"""
    rng = np.random.default_rng(1)
    p = core.create_powderbragg(3000.0, *_planes(5000, "dense", rng), fp32_tables=False)
    n, m = 17_000_001, 9_000_000
    e = 10.0 ** rng.uniform(-4, 0, n)
    xs = p.crossSectionIsotropic(e)
    assert np.array_equal(xs[:m], p.crossSectionIsotropic(e[:m]))
    assert np.array_equal(xs[m:], p.crossSectionIsotropic(e[m:]))
    p.setRNGState(5, 0)
    ge, mu = p.sampleScatterIsotropic(e)
    p.setRNGState(5, 0)
    assert np.array_equal(mu[:m], p.sampleScatterIsotropic(e[:m])[1])
    assert np.array_equal(ge, e) and np.all(np.abs(mu) <= 1.0)
