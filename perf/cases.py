"""Performance cases: the GFN2-xTB work that a QCxMS run has this library do.

A mass-spectrum run calls the library in six ways, and each kind of case is
one of them:

  call   one structure through get_xtb_egrad, as iniqm.f90 does for every
         single point of one trajectory: the latency of one evaluation;
  many   unrelated structures of many sizes in one egrad_many call;
  ips    fragment_ips_batch for finished trajectories: very small single
         points of every fragment, neutral and ionised;
  batch  a Batch kept from call to call (same molecules, new geometries),
         with the options that programs set on it;
  md     an MdEnsemble advanced by a few steps and read, through the
         persistent kernel or the per-step kernels;
  cid    a CidEnsemble (ion and collision gas) advanced and read.

Everything is FP64, the only precision the library has.  Molecules are the
saturated C/H/N/O chains of qcxms_amd.workloads; their composition follows
from the case and their geometry, velocities and energies from the seed.
The library takes and returns host arrays, so the inputs are host arrays and
the device state is the plan (Batch, MdEnsemble, CidEnsemble) that a program
keeps.
"""
import random

import numpy as np

import qcxms_amd
from qcxms_amd import workloads as W

OCTANE, STRETCHED, LARGE = "octane", "c12h24o2n2", "c20h36o2n2"
FS = W.FSTOAU


def listed():
    return [
        # latency: the smallest molecules of a run are fragments such as water
        dict(name="call_water", kind="call", mol="chain", nsys=1, lo=1, hi=1, hetero=1.0, charge=0, etemp=300.0),
        # latency of one step of the README's molecule (26 atoms, 50 basis functions)
        dict(name="call_octane", kind="call", mol=OCTANE, nsys=1, lo=8, hi=8, hetero=0.0, charge=1, etemp=5000.0),
        # latency near the library's size limit (60 atoms, 132 basis functions)
        dict(name="call_c20", kind="call", mol=LARGE, nsys=1, lo=22, hi=22, hetero=0.0, charge=1, etemp=5000.0),
        # ionisation potentials of the fragments of 96 finished trajectories
        dict(name="ips_96", kind="ips", mol="chain", nsys=96, lo=4, hi=9, hetero=0.15, charge=1, etemp=300.0),
        # the uneven batch: 1024 molecules of 3 to 62 atoms in one call
        dict(name="many_1024", kind="many", mol="chain", nsys=1024, lo=1, hi=20, hetero=0.2, charge=-1, etemp=5000.0),
        # 64 stretched C12H24O2N2+ (88 basis functions): fewer systems than compute units
        dict(name="batch_stretched64", kind="batch", mol=STRETCHED, nsys=64, lo=16, hi=16, hetero=0.0, charge=1,
             etemp=5000.0, stored=False, tight=False),
        # one system per compute unit at the thresholds of the parity tests,
        # gradient from stored derivative blocks
        dict(name="batch_octane256", kind="batch", mol=OCTANE, nsys=256, lo=8, hi=8, hetero=0.0, charge=1,
             etemp=5000.0, stored=True, tight=True),
        # the headline production MD: 256 x C8H18+ in the persistent kernel
        dict(name="md_octane256", kind="md", mol=OCTANE, nsys=256, lo=8, hi=8, hetero=0.0, charge=1, etemp=-1.0,
             steps=8, fused=True),
        # one trajectory on its own through the per-step kernels (library default)
        dict(name="md_octane1", kind="md", mol=OCTANE, nsys=1, lo=8, hi=8, hetero=0.0, charge=1, etemp=-1.0,
             steps=8, fused=False),
        # a later fragmentation generation: 512 fragments of uneven size
        dict(name="md_fragments512", kind="md", mol="chain", nsys=512, lo=2, hi=11, hetero=0.15, charge=1, etemp=-1.0,
             steps=6, fused=True),
        # large molecules: 256 x C20H36O2N2+ through the per-step kernels
        dict(name="md_c20_256", kind="md", mol=LARGE, nsys=256, lo=22, hi=22, hetero=0.0, charge=1, etemp=-1.0,
             steps=3, fused=False),
        # CID: 256 x (C8H18+ + N2), 58 basis functions
        dict(name="cid_256", kind="cid", mol=OCTANE, nsys=256, lo=8, hi=8, hetero=0.0, charge=1, etemp=5000.0,
             steps=6),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """Any kind, 1 to 20 heavy atoms a molecule, 1 to 768 molecules (fewer where they are large)."""
    kind = rng.choice(["call", "ips", "many", "batch", "batch", "md", "md", "md", "cid"])
    base = dict(kind=kind, mol="chain", hetero=round(rng.uniform(0.0, 0.4), 3), charge=1, etemp=5000.0)
    if kind == "call":
        h = _log_int(rng, 1, 20)
        return dict(base, nsys=1, lo=h, hi=h, charge=rng.choice([0, 1]), etemp=rng.choice([300.0, 5000.0]))
    if kind == "ips":
        lo = rng.randint(2, 8)
        return dict(base, nsys=_log_int(rng, 2, 200), lo=lo, hi=rng.randint(lo, 14), etemp=300.0)
    if kind == "many":
        lo = rng.randint(1, 12)
        return dict(base, nsys=_log_int(rng, 2, 768), lo=lo, hi=rng.randint(lo, 20), charge=-1,
                    etemp=rng.choice([300.0, 5000.0]))
    hi = _log_int(rng, 1, 20)
    nsys = _log_int(rng, 1, 512 if hi <= 10 else 128)
    if kind == "batch":
        return dict(base, nsys=nsys, lo=hi, hi=hi, stored=rng.random() < 0.3, tight=rng.random() < 0.3)
    if kind == "cid":
        hi = min(max(hi, 5), 14)
        return dict(base, nsys=min(max(nsys, 24), 256), lo=hi, hi=hi, steps=rng.randint(2, 6))
    lo = rng.randint(max(1, hi // 2), hi)
    return dict(base, nsys=nsys, lo=lo, hi=hi, etemp=-1.0, steps=rng.randint(2, 6), fused=rng.random() < 0.5)


# ------------------------------------------------------------------ molecules
def _backbones(case):
    """Heavy-atom chains of the case (no seed: every seed has the same molecules)."""
    r = random.Random("%s %d %d %d %.3f" % (case["kind"], case["nsys"], case["lo"], case["hi"], case["hetero"]))
    out = []
    for _ in range(case["nsys"]):
        n = r.randint(case["lo"], case["hi"])
        z = [r.choice([7, 8]) if r.random() < case["hetero"] else 6 for _ in range(n)]
        if n == 1 and case["hetero"] == 1.0:
            z = [8]
        out.append(z)
    return out


def _structures(case, seed):
    """[(num, xyz in Bohr)] of the case."""
    rng = np.random.default_rng(seed)
    seeds = rng.integers(0, 2**31 - 10**6, size=case["nsys"])
    if case["mol"] == OCTANE:
        return [W.octane(seed=int(s)) for s in seeds]
    if case["mol"] == STRETCHED:
        return [W.chain_c12h24o2n2(seed=int(s)) for s in seeds]
    if case["mol"] == LARGE:
        return [W.chain_c20h36o2n2(seed=int(s)) for s in seeds]
    noise = 0.02 if case["kind"] in ("md", "cid") else 0.03
    return [W.build_chain(z, noise=noise, seed=int(s)) for z, s in zip(_backbones(case), seeds)]


def _charges(case):
    if case["charge"] >= 0:
        return [case["charge"]] * case["nsys"]
    r = random.Random(case["nsys"] * 31 + case["hi"])
    return [r.randint(0, 1) for _ in range(case["nsys"])]


def _trajectories(case, seed, structures):
    """Starting states of trajectories after ionisation: Maxwell-Boltzmann
    velocities at 500 K, internal excess energy of 0.6 eV per atom on
    average, 100 fs of heating (single trajectories and small fragments
    colder, so that they live through the steps that are timed)."""
    rng = np.random.default_rng(seed + 1)
    mean = 0.6 if case["mol"] == OCTANE and case["nsys"] > 1 else 0.25
    out = []
    for num, xyz in structures:
        mass = np.array([W.atomic_mass(int(z)) for z in num])
        s = int(rng.integers(0, 2**31))
        out.append(dict(num=num, xyz=xyz, velo=W.maxwell_boltzmann(mass, 500.0, s), mass=mass,
                        eimp=W.iee_poisson(len(num), mean, 2.5 * mean, s + 1), tadd=100.0 * FS))
    return out


def _split(num, xyz):
    """Two fragments of a chain, cut at its middle heavy atom and pulled apart
    along the chain; the labels fragment_structure would give them."""
    heavy = np.flatnonzero(num != 1)
    cut = int(heavy[len(heavy) // 2])
    far = xyz.copy()
    far[cut:, 0] += 15.0
    label = np.ones(len(num), dtype=np.int32)
    label[cut:] = 2
    return far, label


# -------------------------------------------------------------------- passes
def prepare(case, seed):
    kind = case["kind"]
    st = _structures(case, seed)
    s = dict(case=case, kind=kind)
    if kind == "call":
        s.update(num=st[0][0], xyz=st[0][1])
        qcxms_amd.library()
    elif kind == "many":
        s.update(systems=[(n, c) for (n, _), c in zip(st, _charges(case))], xyz=[x for _, x in st])
    elif kind == "ips":
        parts = [_split(n, x) for n, x in st]
        s.update(nums=[n for n, _ in st], xyz=[p[0] for p in parts], lists=[p[1] for p in parts],
                 mchrg=[case["charge"]] * case["nsys"])
    elif kind == "batch":
        b = qcxms_amd.Batch([(n, c) for (n, _), c in zip(st, _charges(case))])
        if case["tight"]:
            b.set_scc(econv=1e-11, pconv=1e-9)
        if case["stored"]:
            b.set_stored_derivatives(True)
        s.update(batch=b, xyz=np.concatenate([x for _, x in st]))
    elif kind == "md":
        # no limit on the number of steps; ten fragments end a trajectory (the
        # library's cap is six), so that the timed steps are steps of all of them
        s.update(md=qcxms_amd.MdEnsemble(_trajectories(case, seed, st), max_steps=100000, nfragexit=10,
                                         etempin=case["etemp"], fused=case["fused"]))
    else:
        # slow ions: the steps that are timed lie before the collision
        rng = np.random.default_rng(seed + 2)
        s.update(md=qcxms_amd.CidEnsemble(
            [qcxms_amd.cid_setup(t["num"], t["xyz"], t["velo"], t["mass"], 0.5 * FS, gas="N2", elab_ev=10.0,
                                 rand=tuple(rng.random(4))) for t in _trajectories(case, seed, st)],
            charge=case["charge"], etemp=case["etemp"]))
    return s


def run(s):
    case, kind = s["case"], s["kind"]
    if kind == "call":
        q, e, g, stat = qcxms_amd.get_xtb_egrad(s["num"], s["xyz"], case["charge"], 1, qcxms_amd.GFN2_XTB,
                                                case["etemp"])
        return dict(charges=q, energy=e, gradient=g, status=stat)
    if kind == "many":
        e, g, q, stat = qcxms_amd.egrad_many(s["systems"], s["xyz"], etemp=case["etemp"])
        return dict(charges=np.concatenate(q), energy=e, gradient=np.concatenate(g), status=stat)
    if kind == "ips":
        ip, ok, stat = qcxms_amd.fragment_ips_batch(s["nums"], s["xyz"], s["lists"], s["mchrg"])
        return dict(ips=ip, ok=ok, status=stat)
    if kind == "batch":
        e, g, q, stat = s["batch"].egrad(s["xyz"], case["etemp"])
        return dict(charges=q, energy=e, gradient=g, status=stat)
    running = s["md"].run(case["steps"])
    o = s["md"].read()
    keys = ("nstep", "nfrag", "epot", "ekin")
    out = {k: np.array([getattr(r, k) for r in o["results"]]) for k in keys}
    out.update(running=running, xyz=o["xyz"], velocities=o["velo"], gradient=o["grad"], charges=o["qat"],
               fragments=o["list"])
    return out


def exact(case, seed):
    """None: the outputs are fixed points of a self-consistent calculation
    whose parameters and reference data exist in this repository alone, so
    plain torch or numpy gives no value for them without its code."""
    return None


# ---------------------------------------------------------------------- work
NPRIM = {1: (3,), 6: (4, 4), 7: (4, 4), 8: (4, 4)}


def _flops(num, iterations):
    """Operations of one energy and gradient: SCC iterations of 15 n^3 + 30
    n^2 (eigenvectors, two basis changes, density, Fock matrix and moments),
    the factorisation of S, integrals and their derivatives by primitive
    pairs (half of all ordered pairs), pair terms."""
    n = sum(4 if z != 1 else 1 for z in num)
    prim = sum(p for z in num for p in NPRIM[int(z)])
    wide = sum(p * (2 * k + 1) for z in num for k, p in enumerate(NPRIM[int(z)]))
    nat = len(num)
    return (iterations * (15.0 * n**3 + 30.0 * n**2) + 10.0 / 3.0 * n**3 + 0.5 * prim**2 * 2474.0
            + 0.5 * wide**2 * 240.0 + 1421.0 * nat**2 + 14.0 * nat**3)


def work(case):
    """12 SCC iterations a step of MD and 16 a single point from scratch;
    bytes are the arrays that go in and come out."""
    plain = dict(case, mol=case["mol"])
    nums = [n for n, _ in _structures(plain, 0)]
    kind, atoms = case["kind"], sum(len(n) for n in nums)
    if kind in ("md", "cid"):
        if kind == "cid":
            nums = [np.concatenate([n, [7, 7]]) for n in nums]
            atoms += 2 * case["nsys"]
        return dict(flops=case["steps"] * sum(_flops(n, 12) for n in nums), bytes=atoms * (24 + 24 + 24 + 24 + 24 + 12))
    if kind == "ips":
        parts = [n[lab == k] for n, x in _structures(plain, 0) for lab in [_split(n, x)[1]] for k in (1, 2)]
        return dict(flops=2.0 * sum(_flops(n, 16) for n in parts), bytes=atoms * 36 + 252.0 * case["nsys"])
    return dict(flops=sum(_flops(n, 16) for n in nums), bytes=atoms * (24 + 24 + 8) + 20 * case["nsys"])
