"""Host-array calls around the size that goes through pinned staging: the same
values as larger calls on the same streams, repeats, poisoned outputs, and several
threads on handles of their own."""
import ctypes
import threading

import numpy as np
import pytest

from ncrystal_amd import materials, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mat():
    from ncrystal_amd import _capi
    if _capi.lib().ncamd_device_count() < 1:
        pytest.fail("no GPU visible to libncrystal_amd")
    return materials.Material(synth.fcc_powder(), sab=synth.small_sab_table(mass_amu=26.98)).scatter


@pytest.mark.parametrize("n,repeat", [(1, 1), (4096, 1), (4097, 1), (1, 4096), (1, 4097), (512, 8), (513, 8)])
def test_sizes(mat, n, repeat):
    e = synth.energies_logu(n, 1e-5, 10.0, seed=n)
    big = np.tile(e, -(-5000 // n))  # always past the staging size
    assert np.array_equal(mat.crossSectionIsotropic(e, repeat=repeat),
                          np.tile(mat.crossSectionIsotropic(big)[:n], repeat))
    mat.setRNGState(3, 0)
    a = mat.sampleScatterIsotropic(e, repeat=repeat)
    mat.setRNGState(3, 0)
    b = mat.sampleScatterIsotropic(np.concatenate([np.tile(e, repeat), big]))
    assert np.array_equal(a[0], b[0][:n * repeat]) and np.array_equal(a[1], b[1][:n * repeat])


def test_error_then_clean_call(mat):
    from ncrystal_amd import _capi as C
    from ncrystal_amd import core
    g = core.create_freegas(293.0, 4.0, 0.7)
    with pytest.raises(C.NCCalcError):  # an infinite energy cannot be sampled
        g.sampleScatterIsotropic(np.array([0.02, np.inf]))
    oe, om = g.sampleScatterIsotropic(np.array([0.02, 0.03]))
    assert np.all(oe >= 0) and np.all(np.abs(om) <= 1)


def test_threads(mat):
    from ncrystal_amd import _capi as C
    from ncrystal_amd import core
    e = synth.energies_logu(900, 1e-4, 1.0, seed=4)
    mat.setRNGState(11, 0)
    want = mat.sampleScatterIsotropic(e)
    got = [None] * 24

    def work(i):
        c = core.Scatter(C.call("ncamd_clone", mat.handle, 5))
        for _ in range(10):
            c.setRNGState(11, 0)
            got[i] = c.sampleScatterIsotropic(e)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(len(got))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert all(np.array_equal(g[0], want[0]) and np.array_equal(g[1], want[1]) for g in got)


@pytest.mark.parametrize("n", [64, 5000])  # either side of the staging size
def test_null_and_device_arrays(mat, n):
    """no energies are an error that poisons the outputs, and device memory in
    place of host arrays is copied like them, at every size"""
    from ncrystal_amd import _capi as C
    e = synth.energies_logu(n, 1e-4, 1.0, seed=5)
    x, oe, om = np.zeros(n), np.zeros(n), np.zeros(n)
    with pytest.raises(C.NCAMDError, match="HIPError"):
        C.call("ncamd_crosssection_nonoriented_many", mat.handle, None, n, 1, C.dptr(x))
    with pytest.raises(C.NCAMDError, match="HIPError"):
        C.call("ncamd_samplescatterisotropic_many", mat.handle, None, n, 1, C.dptr(oe), C.dptr(om))
    assert np.all(x == -1.0) and np.all(oe == -1.0) and np.all(om == -999.0)
    want = mat.crossSectionIsotropic(e)
    mat.setRNGState(3, 0)
    ws = mat.sampleScatterIsotropic(e)
    de, dx, do, dm = C.DeviceArray.from_numpy(e), C.DeviceArray(n), C.DeviceArray(n), C.DeviceArray(n)
    p = lambda d: ctypes.cast(d.ptr, C._dp)
    C.call("ncamd_crosssection_nonoriented_many", mat.handle, p(de), n, 1, C.dptr(x))
    C.call("ncamd_crosssection_nonoriented_many", mat.handle, C.dptr(e), n, 1, p(dx))
    mat.setRNGState(3, 0)
    C.call("ncamd_samplescatterisotropic_many", mat.handle, p(de), n, 1, p(do), p(dm))
    assert np.array_equal(x, want) and np.array_equal(dx.numpy(), want)
    assert np.array_equal(do.numpy(), ws[0]) and np.array_equal(dm.numpy(), ws[1])
