"""The streamed S(alpha,beta) sampler (a try per lane and step, refilled lanes)
and the two-ended queues of the staged compositions, against the checker on the
same Philox streams: batches around a wave and around the launch's capacity,
tables whose small arrays fit LDS and ones whose do not, energies below the grid,
inside it and above Emax, isotropic and oriented calls, repeats."""
import numpy as np
import pytest

from ncrystal_amd import synth
from conftest import assert_streams_match

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def core():
    from ncrystal_amd import _capi, core
    if _capi.lib().ncamd_device_count() < 1:
        pytest.fail("no GPU visible to libncrystal_amd")
    return core


@pytest.fixture(scope="module", params=["lds", "global"])
def sab(request, core, oracle):
    # na + 2 nb + 3 ne against 4096: 40 + 120 + 900, 60 + 3600 + 900
    t = synth.small_sab_table(mass_amu=26.98) if request.param == "lds" else synth.freegas_like_sab(60, 1800, 12.0)
    args = (t["alpha"], t["beta"], t["sab"], t["temperature"], t["mass"], t["sigma_bound"])
    return core.create_sabscatter(*args), oracle.sab(*args)


def _energies(n, emax, seed):
    """a tenth below the grid, a fifth above Emax, some on grid edges"""
    rng = np.random.default_rng(seed)
    e = np.exp(rng.uniform(np.log(1e-5), np.log(emax), n))
    e[rng.random(n) < 0.1] *= 1e-4
    hi = rng.random(n) < 0.2
    e[hi] = emax * rng.uniform(1.0, 6.0, hi.sum())
    return e


# a difference beyond 1e-9 would be a flipped decision (none seen); the sampled
# values themselves agree to 1e-10 where they cancel most
def _check(a, b, label):
    assert_streams_match(np.max([np.abs(x - y) > 1e-9 * np.maximum(1.0, np.abs(y)) for x, y in zip(a, b)], axis=0), label)


@pytest.mark.parametrize("n", [1, 63, 65, 257, 5000, 300001])
def test_single_process(core, sab, n):
    g, o = sab
    eg = g.egrid()[0]
    e = _energies(n, eg[-1], n)
    e[: min(n, 4)] = [eg[0], np.nextafter(eg[-1], 0), eg[-1], eg[len(eg) // 2] / 1.05][: min(n, 4)]
    g.setRNGState(5, 0)
    ge, gm = g.sampleScatterIsotropic(e)
    oe, om, nerr = o.sample_iso(e, seed=5, nthreads=8)
    assert nerr == 0
    _check((ge, gm), (oe, om), f"single {n}")


@pytest.mark.parametrize("n", [1, 65, 1025, 40000, 131072, 131073, 262144, 262145])
def test_composition(core, oracle, sab, n):
    """two S(alpha,beta) components beside incoherent elastic: both ends of two
    lists, within workgroups up to 262144 neutrons and in queues above"""
    g, o = sab
    t = synth.small_sab_table(seed=5, mass_amu=12.0)
    args = (t["alpha"], t["beta"], t["sab"], t["temperature"], t["mass"], t["sigma_bound"])
    gc = core.create_composition([core.create_elincscatter([0.01], [1.0], [1.0]), g, core.create_sabscatter(*args)],
                                 [1.0, 0.7, 0.3])
    oc = oracle.composition([oracle.elinc([0.01], [1.0], [1.0]), o, oracle.sab(*args)], [1.0, 0.7, 0.3])
    e = _energies(n, g.egrid()[0][-1], n + 1)
    d = synth.isotropic_dirs(n, 3)
    gc.setRNGState(8, 0)
    _check(gc.sampleScatterIsotropic(e), oc.sample_iso(e, seed=8, nthreads=8)[:2], f"composition {n}")
    gc.setRNGState(8, 0)
    ge, gd = gc.sampleScatter(e, d)
    oe, od, nerr = oc.sample_dir(e, d, seed=8, nthreads=8)
    assert nerr == 0
    _check((ge, *gd.T), (oe, *np.asarray(od).reshape(-1, 3).T), f"oriented {n}")


@pytest.mark.parametrize("n", [300001, 1200001])  # pieces of 64 and of 256 places per wave
def test_ordered_energies(core, sab, n):
    """a list in the order of its energies, most of it above Emax: whole waves keep
    neutrons for the high-energy queue"""
    g, o = sab
    emax = g.egrid()[0][-1]
    e = np.concatenate([np.sort(_energies(n - n // 2, emax, n)), emax * np.linspace(1.0, 5.0, n // 2)])
    for x in (e, e[::-1].copy()):
        g.setRNGState(5, 0)
        ge, gm = g.sampleScatterIsotropic(x)
        oe, om, nerr = o.sample_iso(x, seed=5, nthreads=8)
        assert nerr == 0
        _check((ge, gm), (oe, om), f"ordered {n}")


def test_repeat_and_batch(core, oracle, sab):
    g, o = sab
    gc = core.create_composition([core.create_elincscatter([0.01], [1.0], [1.0]), g], [1.0, 1.0])
    e = _energies(700, g.egrid()[0][-1], 2)
    gc.setRNGState(3, 0)
    r = gc.sampleScatterIsotropic(e, repeat=5)
    gc.setRNGState(3, 0)
    s = gc.sampleScatterIsotropic(np.tile(e, 5))  # the same streams without the repeat layout
    assert np.array_equal(r[0], s[0]) and np.array_equal(r[1], s[1])
    import ctypes
    from ncrystal_amd import _capi as C
    n = 5000
    e = _energies(2 * n, g.egrid()[0][-1], 4)
    b = core.Batch([gc, gc], [n, n])
    de, d1, d2 = C.DeviceArray.from_numpy(e), C.DeviceArray(2 * n), C.DeviceArray(2 * n)
    gc.setRNGState(6, 0)
    b.dev_sampleScatterIsotropic(de.ptr, d1.ptr, d2.ptr)
    got = d1.numpy(), d2.numpy()
    assert b.dev_check_errors() == 0
    for part, ctr in ((slice(0, n), 0), (slice(n, 2 * n), 1)):
        gc.setRNGState(6, ctr)
        w = gc.sampleScatterIsotropic(e[part])
        assert np.array_equal(got[0][part], w[0]) and np.array_equal(got[1][part], w[1])
