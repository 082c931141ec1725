"""Measured cases of the per-neutron path, through the framework's public
Python interface (ncrystal_amd.core).

Each case is one call sequence that a transport code or an analysis script
makes on a prepared material: neutrons in, cross sections and scattered
neutrons out.  The Philox state of a process is set before each pass, as a
program that wants reproducible histories does, so a pass is a function of its
state alone.  Materials are fixed by the case; neutrons come from the seed.
"""
import functools
import math

import numpy as np
import torch

from ncrystal_amd import core, materials, synth

WL2EKIN = 0.081804209605330899


def listed():
    return [
        # a script asks for a handful of neutrons through the host-array calls:
        # launches, copies and host work count, not throughput
        dict(name="host_call_64", kind="host", n=64),
        # the usual transport batch: a powder (incoherent elastic, Bragg,
        # S(alpha,beta) of its Debye spectrum), cross sections and oriented
        # scattering on device arrays
        dict(name="powder_1e6", kind="powder", n=1_000_000),
        # a compound with one S(alpha,beta) per element, a ragged batch as an
        # event generator leaves it, isotropic scattering
        dict(name="compound_100k", kind="compound", n=100_003),
        # one element's S(alpha,beta) alone, the plain sampler, a large batch
        dict(name="sab_plain_3e7", kind="sab", n=30_000_001, nalpha=200, nbeta=800, envelope=False),
        # the same table with the envelope sampler: the benchmark's batch
        dict(name="sab_envelope_1e8", kind="sab", n=100_000_000, nalpha=200, nbeta=800, envelope=True),
        # a low-symmetry powder with very many planes
        dict(name="powderbragg_5e7", kind="powderbragg", n=50_000_000, planes=262_067),
        # a mosaic single crystal in a collimated beam
        dict(name="scbragg_beam_2e6", kind="scbragg", n=2_000_000, dcutoff=0.2, mosaic=30.0, cone=2.0),
        # a single-crystal material (mosaic crystal, the short-d powder rest,
        # incoherent elastic, S(alpha,beta)) deep in a transport: directions
        # in every sense, a ragged batch
        dict(name="sc_material_200k", kind="scmaterial", n=200_003, mosaic=40.0),
        # pyrolytic graphite (monochromators, filters): the layered-crystal model
        dict(name="layered_131k", kind="layered", n=131_072, mosaic=4.0),
        # a whole transport run: a beam through a sphere of powder
        dict(name="minimc_8e6", kind="minimc", n=8_000_000, wl=4.0),
        # many materials of uneven sizes in one launch
        dict(name="batch_32", kind="batch", nmat=32, scale=1.0),
        # material set-up: a vibrational spectrum expanded to S(alpha,beta) at
        # two temperatures
        dict(name="vdos_lux4", kind="vdos", lux=4, mass=26.98),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "powder", "compound", "sab", "sab", "powderbragg", "scbragg", "scmaterial", "layered",
                       "minimc", "batch", "vdos"])
    if kind == "host":
        return dict(kind=kind, n=_logint(rng, 1, 4096))
    if kind == "powder":
        return dict(kind=kind, n=_logint(rng, 1e3, 2e6) | 1)
    if kind == "compound":
        return dict(kind=kind, n=_logint(rng, 1e3, 1e6))
    if kind == "sab":
        env = rng.random() < 0.5
        return dict(kind=kind, n=_logint(rng, 1e4, 1e8 if env else 3e7), nalpha=_logint(rng, 60, 200),
                    nbeta=_logint(rng, 100, 800), envelope=env)
    if kind == "powderbragg":
        return dict(kind=kind, n=_logint(rng, 1e4, 5e7) | 1, planes=_logint(rng, 100, 3e5))
    if kind == "scbragg":
        return dict(kind=kind, n=_logint(rng, 1e4, 2e6), dcutoff=rng.choice([0.25, 0.3, 0.4, 0.5]),
                    mosaic=rng.uniform(10.0, 60.0), cone=rng.uniform(0.5, 15.0))
    if kind == "scmaterial":
        return dict(kind=kind, n=_logint(rng, 1e3, 2e5), mosaic=rng.uniform(20.0, 60.0))
    if kind == "layered":
        return dict(kind=kind, n=_logint(rng, 1e3, 131072), mosaic=rng.uniform(1.0, 5.0))
    if kind == "minimc":
        return dict(kind=kind, n=_logint(rng, 2e6, 8e6), wl=rng.uniform(1.0, 4.5))
    if kind == "batch":
        return dict(kind=kind, nmat=rng.randint(3, 32), scale=math.exp(rng.uniform(math.log(0.05), 0.0)))
    return dict(kind=kind, lux=rng.choice([2, 3, 4]), mass=rng.uniform(10.0, 60.0))


# ---------------------------------------------------------------- materials

def _powder():
    """fcc powder: ElInc + PowderBragg + S(alpha,beta) of the Debye spectrum"""
    cr = synth.fcc_powder()
    s = cr.species[0]
    dyn = {"vdos": s.debye_temp, "mass": s.mass, "sigma_bound": 4 * math.pi * s.csl ** 2 + s.sigma_inc, "vdoslux": 3}
    return cr, materials.Material(cr, dynamics=[(1.0, dyn)])


def _compound():
    """rock-salt cell of a light and a heavy element, one spectrum each"""
    fcc = [(0, 0, 0), (0, .5, .5), (.5, 0, .5), (.5, .5, 0)]
    light = synth.Species("A", 0.5375, 0.08, 0.06, 24.305, 743.0, np.array(sorted(fcc), dtype=float))
    heavy = synth.Species("B", 0.5805, 0.0008, 0.0002, 15.999, 743.0,
                          np.array(sorted([((x + .5) % 1, (y + .5) % 1, (z + .5) % 1) for x, y, z in fcc])))
    cr = synth.Crystal(4.2113, 4.2113, 4.2113, [light, heavy], 293.0, 0.4, name="rocksalt")
    dyn = [(0.5, {"vdos": s.debye_temp, "mass": s.mass, "sigma_bound": 4 * math.pi * s.csl ** 2 + s.sigma_inc,
                  "vdoslux": 3}) for s in (light, heavy)]
    return materials.Material(cr, dynamics=dyn)


@functools.lru_cache(maxsize=4)
def _sab_table(nalpha, nbeta):
    return synth.sab_table_c3(seed=1, nalpha=nalpha, nbeta=nbeta)


@functools.lru_cache(maxsize=2)
def _small_sab():
    return synth.small_sab_table(mass_amu=26.98)


def _create_sab(t):
    return core.create_sabscatter(t["alpha"], t["beta"], t["sab"], t["temperature"], t["mass"], t["sigma_bound"])


def _planes(n):
    """n plane spacings with density ~ d^-4 and their |F|^2 x multiplicity"""
    r = np.random.default_rng(n)
    dmin, dmax = 0.1, 8.0
    d = np.sort((dmin ** -3 - r.uniform(size=n) * (dmin ** -3 - dmax ** -3)) ** (-1.0 / 3.0))[::-1].copy()
    f = r.uniform(0.01, 5.0, size=n) * 2 * r.integers(1, 25, size=n) * np.exp(-0.008 * (2 * np.pi / d) ** 2)
    return 24000.0, d, f


@functools.lru_cache(maxsize=2)
def _ortho_families(dcutoff):
    cr = synth.ortho_random(seed=1, dcutoff=dcutoff)
    sp = [(s.csl, core.debye_msd(s.debye_temp, cr.temperature, s.mass), s.positions) for s in cr.species]
    return cr, core.hkl_orthogonal_members(cr.a, cr.b, cr.c, sp, dcutoff)


def _subset(fams, keep):
    _, _, dsp, fsq, moff, mh = fams
    idx = np.nonzero(keep)[0]
    parts = [mh[moff[i]:moff[i + 1]] for i in idx]
    off = np.concatenate([[0], np.cumsum([len(p) for p in parts])]).astype(np.int64)
    return dsp[idx], fsq[idx], off, np.concatenate(parts).astype(np.int32)


def _sc_material(mosaic):
    """fcc single crystal: SCBragg for d >= 0.4 Aa, PowderBragg below"""
    cr = synth.fcc_powder(dcutoff=0.25)
    s = cr.species[0]
    msd = core.debye_msd(s.debye_temp, cr.temperature, s.mass)
    fams = core.hkl_orthogonal_members(cr.a, cr.b, cr.c, [(s.csl, msd, s.positions)], cr.dcutoff)
    v0n = cr.volume * cr.n_atoms
    low = fams[2] < 0.4
    scb = core.create_scbragg(v0n, *_subset(fams, ~low), core.reci_lattice_orthogonal(cr.a, cr.b, cr.c),
                              synth.random_rotation(11), math.radians(mosaic / 60.0))
    parts = [core.create_elincscatter([msd], [s.sigma_inc], [1.0]), scb,
             core.create_powderbragg(v0n, fams[2][low], fams[3][low] * fams[1][low]), _create_sab(_small_sab())]
    return core.create_composition(parts, [1.0] * 4)


def _graphite(mosaic):
    """pyrolytic graphite, layer axis (0,0,1)"""
    a, c = 2.464, 6.711
    cell = (a, a, c, 90, 90, 120)
    pos = np.array([[0, 0, 0.25], [0, 0, 0.75], [1 / 3, 2 / 3, 0.25], [2 / 3, 1 / 3, 0.75]])
    csl = math.sqrt(5.5504799463874 / (4 * math.pi))
    _, _, dsp, fsq, moff, mh = core.hkl_spacegroup_members(194, cell, [(csl, 0.006, pos)], 0.5)
    return core.create_lcbragg(35.285743880564 * 4, dsp, fsq, moff, mh, core.reci_lattice(cell), np.eye(3),
                               [0.0, 0.0, 1.0], math.radians(mosaic))


# ----------------------------------------------------------------- neutrons

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def _energies(g, n, lo, hi):
    """log-uniform energies [eV]"""
    return torch.exp(math.log(lo) + _rand(g, n) * (math.log(hi) - math.log(lo)))


def _wl_energies(g, n, lo, hi):
    """energies of uniform wavelengths [Aa]"""
    return WL2EKIN / (lo + (hi - lo) * _rand(g, n)) ** 2


def _isotropic(g, n):
    uz = 2.0 * _rand(g, n) - 1.0
    ph = 2.0 * math.pi * _rand(g, n)
    s = torch.sqrt(1.0 - uz * uz)
    return torch.stack([s * torch.cos(ph), s * torch.sin(ph), uz], dim=1).contiguous()


def _cone(g, n, degrees):
    """directions uniform in a cone about a fixed beam axis"""
    ax = torch.tensor(synth.random_unit_vector(5), device="cuda")
    e1 = torch.linalg.cross(ax, torch.tensor([0.0, 0.0, 1.0], device="cuda", dtype=torch.float64))
    e1 = e1 / torch.linalg.norm(e1)
    e2 = torch.linalg.cross(ax, e1)
    cmin = math.cos(math.radians(degrees))
    ct = cmin + (1.0 - cmin) * _rand(g, n)
    st = torch.sqrt(1.0 - ct * ct)
    ph = 2.0 * math.pi * _rand(g, n)
    return (ct[:, None] * ax + (st * torch.cos(ph))[:, None] * e1 + (st * torch.sin(ph))[:, None] * e2).contiguous()


def _out(*shape):
    return torch.empty(*shape, device="cuda", dtype=torch.float64)


def _stream():
    return torch.cuda.current_stream().cuda_stream


# -------------------------------------------------------------------- cases

def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    s = dict(kind=kind, seed=int(seed) & 0x7FFFFFFF)
    if kind == "host":
        s["proc"] = _powder()[1].scatter
        s["e"] = _energies(g, case["n"], 1e-5, 10.0).cpu().numpy()
        return s
    if kind == "vdos":
        e, rho = (x[1:] for x in synth.vdos_3gauss(seed=3))  # from the first point above E = 0
        t = 250.0 + 100.0 * float(_rand(g, 1)[0])
        s.update(vdos=(e, rho), temps=(t, t + 37.5), lux=case["lux"], mass=case["mass"])
        return s
    if kind == "minimc":
        cr, m = _powder()
        nd = cr.n_atoms / cr.volume
        ekin = WL2EKIN / case["wl"] ** 2
        r = 0.5 / (nd * 100.0 * m.scatter.crossSectionIsotropic(np.array([ekin]))[0])
        s.update(proc=m.scatter, absn=core.create_absoov(cr.species[0].sigma_abs), nd=nd, r=r, ekin=ekin, n=case["n"])
        return s
    if kind == "batch":
        mats = synth.batch_materials(nmat=case["nmat"], seed=11)
        procs, counts = [], []
        for m in mats:
            procs.append(core.create_composition(
                [core.create_elincscatter(m["elinc"]["msd"], m["elinc"]["bixs"], m["elinc"]["scale"]),
                 core.create_powderbragg(*m["pb"]), _create_sab(m["sab"])], [1.0, 1.0, 1.0]))
            counts.append(max(1, int(m["count"] * case["scale"])))
        b = core.Batch(procs, counts)
        n = b.total
        s.update(procs=procs, batch=b, e=_energies(g, n, 1e-4, 1.0), xs=_out(n), oe=_out(n), omu=_out(n))
        return s
    n = s["n"] = case["n"]
    if kind == "powder":
        s.update(proc=_powder()[1].scatter, e=_energies(g, n, 1e-5, 10.0), d=_isotropic(g, n))
    elif kind == "compound":
        s.update(proc=_compound().scatter, e=_energies(g, n, 1e-4, 5.0))
    elif kind == "sab":
        p = _create_sab(_sab_table(case["nalpha"], case["nbeta"]))
        if case["envelope"]:
            p.use_envelope_sampler(nintervals=256, emin=0.999e-3, emax=1.001, nbox_w=128, nbox_k=32)
        s.update(proc=p, e=_energies(g, n, 1e-3, 1.0))
    elif kind == "powderbragg":
        s.update(proc=core.create_powderbragg(*_planes(case["planes"])), e=_energies(g, n, 1e-4, 1.0))
    elif kind == "scbragg":
        cr, (_, _, dsp, fsq, moff, mh) = _ortho_families(case["dcutoff"])
        s.update(proc=core.create_scbragg(cr.volume * cr.n_atoms, dsp, fsq, moff, mh,
                                          core.reci_lattice_orthogonal(cr.a, cr.b, cr.c), synth.random_rotation(4),
                                          math.radians(case["mosaic"] / 60.0)),
                 e=_wl_energies(g, n, 1.0, 6.0), d=_cone(g, n, case["cone"]))
    elif kind == "scmaterial":
        s.update(proc=_sc_material(case["mosaic"]), e=_wl_energies(g, n, 0.8, 6.0), d=_isotropic(g, n))
    elif kind == "layered":
        s.update(proc=_graphite(case["mosaic"]), e=_wl_energies(g, n, 0.5, 7.0), d=_isotropic(g, n))
    s.update(xs=_out(n), oe=_out(n))
    s["o2"] = _out(n, 3) if "d" in s else _out(n)
    return s


def run(s):
    kind = s["kind"]
    if kind == "vdos":
        out = []
        for t in s["temps"]:
            k = core.vdos_kernel(s["vdos"], t, s["mass"], vdoslux=s["lux"])
            out.append((k["alpha"], k["beta"], k["sab"]))
        return out
    if kind == "minimc":
        h = core.minimc_sphere(s["proc"], s["absn"], s["nd"], s["r"], s["ekin"], s["n"],
                               pos=(0.0, 0.0, -s["r"] * (1 - 1e-13)), nbins=30, seed=s["seed"])
        return {k: (v["content"], v["errorsq"]) for k, v in h.items() if k != "info"}
    if kind == "batch":
        for i, p in enumerate(s["procs"]):
            p.setRNGState(s["seed"] + i, 0)
        st = _stream()
        s["batch"].dev_crossSection(s["e"].data_ptr(), s["xs"].data_ptr(), stream=st)
        s["batch"].dev_sampleScatterIsotropic(s["e"].data_ptr(), s["oe"].data_ptr(), s["omu"].data_ptr(), stream=st)
        return s["xs"], s["oe"], s["omu"]
    p = s["proc"]
    p.setRNGState(s["seed"], 0)
    if kind == "host":
        xs = p.xsect(ekin=s["e"])
        return (xs,) + tuple(p.sampleScatterIsotropic(s["e"]))
    st, n = _stream(), s["n"]
    e, xs, oe, o2 = (s[k].data_ptr() for k in ("e", "xs", "oe", "o2"))
    if kind == "sab":  # sampling alone: the benchmark's step
        p.dev_sampleScatterIsotropic(e, n, oe, o2, stream=st)
        return s["oe"], s["o2"]
    if kind in ("scbragg", "layered"):
        p.dev_crossSection(e, s["d"].data_ptr(), n, xs, stream=st)
        p.dev_sampleScatter(e, s["d"].data_ptr(), n, oe, o2, stream=st)
    elif kind == "scmaterial":
        # the oriented calls of a composition go through the handle's C entry
        core.C.call("ncamd_dev_crosssection_many_dirs", p.handle, e, s["d"].data_ptr(), n, xs, st)
        p.dev_sampleScatter(e, s["d"].data_ptr(), n, oe, o2, stream=st)
    elif kind == "powder":
        p.dev_crossSectionIsotropic(e, n, xs, stream=st)
        p.dev_sampleScatter(e, s["d"].data_ptr(), n, oe, o2, stream=st)
    else:
        p.dev_crossSectionIsotropic(e, n, xs, stream=st)
        p.dev_sampleScatterIsotropic(e, n, oe, o2, stream=st)
    return s["xs"], s["oe"], s["o2"]


def work(case):
    """bytes: neutrons in, cross sections and scattered neutrons out (tables
    stay in cache); flops: the arithmetic of one evaluation per neutron"""
    kind = case["kind"]
    if kind == "vdos":
        # order sum of the table: rows x columns x orders (2 flops each)
        na, nb, orders = {2: (200, 400, 153), 3: (400, 800, 240), 4: (800, 1600, 368)}[case["lux"]]
        return dict(bytes=2 * 8.0 * (na * nb + na + nb), flops=2 * 2.0 * na * nb * orders)
    if kind == "batch":
        n = sum(max(1, int(m["count"] * case["scale"])) for m in synth.batch_materials(nmat=case["nmat"], seed=11))
        return dict(bytes=(16.0 + 24.0) * n, flops=400.0 * n)
    n = float(case["n"])
    if kind == "minimc":
        # a source neutron and its later steps (about two in all): state in
        # and out once per step
        return dict(bytes=2 * 160.0 * n, flops=2 * 600.0 * n)
    if kind == "sab":
        return dict(bytes=24.0 * n, flops=300.0 * n)
    if kind in ("host", "compound"):
        return dict(bytes=40.0 * n, flops=400.0 * n)
    if kind == "powderbragg":
        return dict(bytes=40.0 * n, flops=60.0 * n)
    if kind == "powder":
        return dict(bytes=(16.0 + 64.0) * n, flops=450.0 * n)
    # oriented crystals: the reflections in reach of the neutron, some tens,
    # at about 80 flops (layered: 17 points of a rotation integral for each of
    # some tens of plane sets)
    per = {"scbragg": 2000.0, "scmaterial": 1000.0, "layered": 20000.0}[kind]
    return dict(bytes=(40.0 + 64.0) * n, flops=per * n)


def tolerance(case):
    """FP64 throughout.  Against the CPU checker on the same Philox streams
    (another libm, the same draws) cross sections differ by 1e-17 in the
    2-norm, sampled energies and angles by 8e-14, and by 7e-11 where they
    cancel most (1e6 neutrons; the largest grows with the batch); sums in
    another order (layered model, expansion) stay below that.  The transport
    run compacts its neutrons in the order in which workgroups finish, so
    equal seeds agree statistically: its histograms differ by 0.7 to 2 % from
    one call to the next (2-norm, 30 bins)."""
    if case["kind"] == "minimc":
        return dict(rel=0.03, max=0.3)
    return dict(rel=1e-11, max=1e-8)


def exact(case, seed):
    """PowderBragg in plain torch: the cross section is the cumulated plane
    strength up to the largest reachable plane over E, and the scattering is
    elastic.  The other processes' cross sections are defined by an
    integration procedure (S(alpha,beta), mosaic spline, rotation averages)
    and sampled values by a random stream: no value of their own."""
    if case["kind"] != "powderbragg":
        return None
    v0n, d, f = _planes(case["planes"])
    e = _energies(_gen(seed), case["n"], 1e-4, 1.0)
    thr = torch.tensor(WL2EKIN / (4.0 * d * d), device="cuda")
    cum = torch.cumsum(torch.tensor(d * f * WL2EKIN / (2.0 * v0n), device="cuda"), 0)
    idx = torch.searchsorted(thr, e, right=True)
    xs = torch.where(idx > 0, cum[(idx - 1).clamp(min=0)] / e, torch.zeros_like(e))
    return xs, e, None
