"""Performance cases: the work a user of this engine gives it, through its public entry points.

Kinds of case
  tild       a block of particle-mesh steps between two log lines of a run, with the logged energies and the forces
             at the positions it ends with (TildEngine.step_energies, compute_forces)
  replicas   the same for several small independent boxes advanced as one group (TildGroup)
  fts        complex-Langevin iterations between two log lines: observables, densities and fields (FtsSystem)
  sweep      many complex-Langevin replicas of uneven shapes advanced together (FtsBatch)
  fft        the batched 3D transform, forward and back (mft_fft_exec)
  particles  one force evaluation of a caller that keeps its own loop and calls the TILD kernels one by one
             (mft_tild_grid_weights, _fill_density, _pair_force, _map_forces)
  chains     the same for a field-theory caller: species fields -> propagators -> Q -> densities
             (mft_fts_propagate, _partition_function, _density)
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "matilda.ft_amd"))
import mft  # noqa: E402
from mft import systems  # noqa: E402

GPU = "cuda"
FFT_LENGTHS = (8, 10, 12, 16, 20, 24, 32, 40, 48, 64, 80, 96, 128, 160, 192, 256)
TILD_LENGTHS = (16, 20, 24, 32, 40, 48, 64, 80, 96, 128)
FTS_LENGTHS = (16, 20, 24, 32, 40, 48, 64, 80, 96)


# ------------------------------------------------------------------ cases ----
def listed():
    return [
        # the plain AB diblock melt, 2000 chains of 20 beads: the smallest run in earnest, bound by launches
        dict(name="tild_melt_40k", kind="tild", nx=32, ny=32, nz=32, spacing=0.625, density=5.0, chain=20, charged=False,
             pme=3, integrator="GJF", steps=25),
        # a charged polycation / polyanion / solvent mixture of ordinary size (the coacervate's density, an eighth
        # of its volume)
        dict(name="tild_coacervate_225k", kind="tild", nx=64, ny=64, nz=64, spacing=0.46875, density=25.0 / 3.0, chain=20,
             charged=True, pme=3, integrator="GJF", steps=40),
        # the large coacervate of the benchmark
        dict(name="tild_coacervate_1800k", kind="tild", nx=128, ny=128, nz=128, spacing=0.46875, density=25.0 / 3.0,
             chain=20, charged=True, pme=3, integrator="GJF", steps=40),
        # a box that is no cube, chains of odd length, quadratic splines and the Euler-Maruyama integrator
        dict(name="tild_slab_em", kind="tild", nx=96, ny=64, nz=40, spacing=0.5, density=6.0, chain=33, charged=False,
             pme=2, integrator="EM", steps=40),
        # independent replicas of a small melt for statistics, one graph for all
        dict(name="tild_replicas_8", kind="replicas", replicas=8, nx=24, ny=24, nz=24, spacing=0.625, density=5.0,
             chain=20, charged=False, pme=3, integrator="GJF", steps=32),
        # the smallest field-theory solve of the served mix
        dict(name="fts_diblock_32", kind="fts", nx=32, ny=32, nz=32, spacing=0.125, beads=50, first=25, arch="diblock",
             scheme="EM", iterations=40),
        # the plain diblock of the benchmark
        dict(name="fts_diblock_64", kind="fts", nx=64, ny=64, nz=64, spacing=0.125, beads=100, first=50, arch="diblock",
             scheme="EM", iterations=20),
        # the largest grid of the served mix, an uneven diblock with the predictor-corrector scheme (two density
        # passes an iteration)
        dict(name="fts_diblock_96_empc", kind="fts", nx=96, ny=96, nz=96, spacing=0.125, beads=50, first=17,
             arch="diblock", scheme="EMPC", iterations=8),
        # a parameter sweep: uneven grids, chain lengths, compositions and chi N in one batch
        dict(name="fts_sweep_16", kind="sweep", replicas=16, sweep=7, iterations=10),
        # transforms of a batch of fields on a grid that is no cube and no power of two
        dict(name="fft_96x80x64_b4", kind="fft", nx=96, ny=80, nz=64, batch=4),
        # a TILD caller's own loop, one force evaluation of a two-species melt
        dict(name="particles_160k", kind="particles", nx=64, ny=64, nz=64, spacing=0.5, density=5.0, pme=3),
        # a field-theory caller's own loop, an ABC triblock
        dict(name="chains_48", kind="chains", nx=48, ny=48, nz=48, spacing=0.125, beads=60, first=20, arch="abc"),
    ]


def _spread(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _grid(rng, lengths, most):
    """Three grid lengths, a cube as often as not, of at most `most` points and spread over the logarithm of that."""
    while True:
        goal = _spread(rng, 16 ** 3, most) ** (1.0 / 3.0)
        near = sorted(lengths, key=lambda n: abs(math.log(n / goal)))[:4]
        n = [rng.choice(near)] * 3 if rng.random() < 0.5 else [rng.choice(near) for _ in range(3)]
        if n[0] * n[1] * n[2] <= most:
            return dict(nx=n[0], ny=n[1], nz=n[2])


def draw(rng):
    kind = rng.choice(("tild", "tild", "replicas", "fts", "fts", "sweep", "fft", "particles", "chains"))
    if kind == "tild":
        return dict(kind=kind, **_grid(rng, TILD_LENGTHS, 128 ** 3), spacing=round(rng.uniform(0.42, 0.65), 4),
                    density=round(rng.uniform(3.0, 25.0 / 3.0), 4), chain=rng.randint(5, 40), charged=rng.random() < 0.5,
                    pme=rng.choice((2, 3, 3)), integrator=rng.choice(("GJF", "GJF", "EM")), steps=rng.randint(10, 20))
    if kind == "replicas":
        n = rng.choice((16, 20, 24, 32))
        return dict(kind=kind, replicas=rng.randint(3, 12), nx=n, ny=n, nz=n, spacing=round(rng.uniform(0.5, 0.65), 4),
                    density=round(rng.uniform(3.0, 6.0), 4), chain=rng.randint(10, 30), charged=False, pme=3,
                    integrator="GJF", steps=rng.randint(9, 33))
    if kind == "fts":
        beads = rng.randint(20, 100)
        return dict(kind=kind, **_grid(rng, FTS_LENGTHS, 96 ** 3 * 100 // (2 * beads)),
                    spacing=round(rng.uniform(0.1, 0.16), 4), beads=beads, first=rng.randint(5, beads - 5),
                    arch=rng.choice(("diblock", "diblock", "aba", "abc")), scheme=rng.choice(("EM", "EM", "EMPC")),
                    iterations=rng.randint(4, 10))
    if kind == "sweep":
        return dict(kind=kind, replicas=rng.randint(4, 12), sweep=rng.randint(1, 10 ** 6), iterations=rng.randint(4, 8))
    if kind == "fft":
        g = _grid(rng, FFT_LENGTHS, 128 ** 3)
        if rng.random() < 0.2:
            g["nz"] = 1  # a plane, as two-dimensional data has it
        return dict(kind=kind, **g, batch=rng.randint(1, 6))
    if kind == "particles":
        return dict(kind=kind, **_grid(rng, TILD_LENGTHS, 96 ** 3), spacing=round(rng.uniform(0.42, 0.65), 4),
                    density=round(rng.uniform(2.0, 6.0), 4), pme=rng.choice((1, 2, 3, 3)))
    beads = rng.randint(20, 80)
    return dict(kind=kind, **_grid(rng, FTS_LENGTHS, 64 ** 3), spacing=round(rng.uniform(0.1, 0.16), 4), beads=beads,
                first=rng.randint(5, beads // 2 - 4), arch=rng.choice(("diblock", "aba", "abc")))


def work(case):
    """Bytes and operations one pass cannot do without."""
    k = case["kind"]
    if k in ("tild", "replicas"):
        # per step: the particle state streamed once (positions, previous positions, noise, topology, forces), per
        # density channel the density written and the transforms' and force fields' one read and write each
        M = case["nx"] * case["ny"] * case["nz"]
        N = _nparticles(case)
        chan = 3 if case["charged"] else 2
        G = (case["pme"] + 1) ** 3
        b = case["steps"] * (112.0 * N + 80.0 * chan * M) + 12.0 * N
        f = case["steps"] * (N * G * 10.0 + 2.5 * chan * 5.0 * M * math.log2(M) + 100.0 * N)
        r = case.get("replicas", 1)
        return {"bytes": b * r, "flops": f * r}
    if k in ("fts", "sweep"):
        b = f = 0.0
        for spec, _ in _specs(case, None):
            M = int(np.prod(spec["Nx"]))
            n = sum(x for x, _ in spec["molecules"][0]["blocks"])
            passes = 2 if spec["potentials"][0].get("scheme") == "EMPC" else 1
            chains = 1 if _symmetric(spec["molecules"][0]["blocks"]) else 2
            b += case["iterations"] * passes * M * 8.0 * (2 * chains * n + 12)
            f += case["iterations"] * passes * M * (chains * (n - 1) * (10.0 * math.log2(M) + 8.0) + 16.0 * n)
        return {"bytes": b, "flops": f}
    M = case["nx"] * case["ny"] * case["nz"]
    if k == "fft":
        return {"bytes": 32.0 * M * case["batch"], "flops": 10.0 * M * math.log2(max(2, M)) * case["batch"]}
    if k == "particles":
        N = 2 * _per_species(case)
        G = (case["pme"] + 1) ** 3
        # the tables written and read by the density and by the force map, the fields of four pair forces
        return {"bytes": N * (12.0 + 24.0 * G + 12.0) + M * (2 * 4.0 + 4 * (4 + 24 + 24)),
                "flops": N * G * 12.0 + 4 * 4 * 5.0 * M * math.log2(M)}
    n = sum(x for x, _ in _blocks(case))
    return {"bytes": M * 8.0 * (4 * n + 8), "flops": M * (2 * (n - 1) * 10.0 * math.log2(M) + 16.0 * n)}


def tolerance(case):
    """About four times the distance from 64 bits that was measured."""
    k = case["kind"]
    if k in ("tild", "replicas"):
        # 1e-4 in the forces: positions are 32-bit floats of up to the box length, and their rounding enters the
        # integrators as a velocity, so it grows with the 3/2 power of the number of steps
        return {"rel": 4e-4, "max": 2e-2}
    if k in ("fts", "sweep"):
        return {"rel": 2e-6, "max": 1e-4}
    if k == "fft":
        return {"rel": 1e-6, "max": 4e-5}
    return {"rel": 3e-6, "max": 1e-4}  # chains: up to 6.5e-7 along long chains of a small grid


# ----------------------------------------------------------------- inputs ----
def _nparticles(case):
    V = case["nx"] * case["ny"] * case["nz"] * case["spacing"] ** 3
    chains = max(2, int(case["density"] * V / case["chain"]))
    if not case["charged"]:
        return chains * case["chain"]
    pairs = max(1, int(0.89 * chains / 2))
    return 2 * pairs * case["chain"] + int((chains - 2 * pairs) * case["chain"])


def _tild(case, seed):
    """Positions, topology and potentials of a melt of AB diblocks, or of polycations, polyanions and solvent."""
    rng = np.random.default_rng(seed)
    Nx = (case["nx"], case["ny"], case["nz"])
    L = tuple(float(np.float32(n * case["spacing"])) for n in Nx)
    N, c = _nparticles(case), case["chain"]
    V = L[0] * L[1] * L[2]
    if case["charged"]:
        pairs = max(1, int(0.89 * max(2, int(case["density"] * V / c)) / 2))
        nchain = 2 * pairs
        type_ = np.full(N, 2, np.int32)
        type_[: pairs * c] = 0
        type_[pairs * c: nchain * c] = 1
        charge = np.zeros(N, np.float32)
        charge[: pairs * c] = 1.0
        charge[pairs * c: nchain * c] = -1.0
    else:
        nchain = N // c
        type_ = np.tile((np.arange(c) >= c // 2).astype(np.int32), nchain)
        charge = None
    x = np.empty((N, 3))
    walk = rng.standard_normal((nchain, c, 3), np.float32) * np.float32(math.sqrt(1.0 / 3.0))
    walk[:, 0, :] = rng.random((nchain, 3)) * np.asarray(L)
    x[: nchain * c] = np.cumsum(walk, axis=1, dtype=np.float64).reshape(-1, 3)
    if N > nchain * c:
        x[nchain * c:] = rng.random((N - nchain * c, 3)) * np.asarray(L)
    x = np.mod(x, np.asarray(L)).astype(np.float32)
    x[x >= np.asarray(L, np.float32)] = 0.0
    i = np.arange(N)
    pos = i % c
    chained = i < nchain * c
    prev, nxt = chained & (pos > 0), chained & (pos < c - 1)
    bonded = np.zeros((N, 2), np.int32)
    bonded[:, 0] = np.where(prev, i - 1, np.where(nxt, i + 1, 0))
    bonded[:, 1] = np.where(prev & nxt, i + 1, 0)
    rho0, kappa, chi = N / V, 50.0, 1.0
    sig = float(np.float32(math.sqrt(0.5)))
    ns = 3 if case["charged"] else 2
    pots = [dict(kind="gaussian", maskI=1 << s, maskJ=1 << s, A=float(np.float32(kappa / (2 * rho0))), sigma=sig)
            for s in range(ns)]
    for a in range(ns):
        for b in range(a + 1, ns):
            extra = chi if b == ns - 1 else 0.0
            pots.append(dict(kind="gaussian", maskI=1 << a, maskJ=1 << b, A=float(np.float32((kappa + extra) / rho0)),
                             sigma=sig))
    if case["charged"]:
        pots.append(dict(kind="charges", A=2.0, sigma=0.5))
    return dict(Nx=Nx, L=L, pmeorder=case["pme"], species=list("PNS"[:ns]), x=x.reshape(-1), potentials=pots,
                topo=dict(type=type_, charge=charge, nBonds=(prev.astype(np.int32) + nxt.astype(np.int32)),
                          bondedTo=bonded.reshape(-1), bondType=np.zeros(2 * N, np.int32)),
                bond_k=[1.5], bond_r0=[0.0], bond_style=[0], delt=0.005, mass=[1.0] * ns, mobility=[1.0] * ns,
                has_charges=case["charged"], seed=int(seed) % (1 << 40) + 17)


def _blocks(case):
    n, a = case["beads"], case["first"]
    if case["arch"] == "diblock":
        return [(a, 0), (n - a, 1)]
    if case["arch"] == "aba":  # a symmetric triblock: its two propagators are one
        h = max(1, a // 2)
        return [(h, 0), (n, 1), (h, 0)]
    b = max(1, (n - a) // 2)
    return [(a, 0), (b, 1), (max(1, n - a - b), 0)]


def _symmetric(blocks):
    return blocks == blocks[::-1]


def _specs(case, seed):
    """[(description, seed of its fields)] of the field-theory systems of a case."""
    if case["kind"] == "sweep":
        rng = np.random.default_rng(case["sweep"])
        rows = []
        for _ in range(case["replicas"]):
            g = int(rng.choice([24, 32, 48, 64]))
            L, chi, fA = rng.uniform(4.0, 10.0), rng.uniform(10.0, 20.0), rng.uniform(0.3, 0.5)
            n = int(rng.choice([50, 100]))
            a = int(round(fA * n))
            rows.append(((g, g, g), (float(np.float32(L)),) * 3, [(a, 0), (n - a, 1)], float(chi), "EM"))
    else:
        Nx = (case["nx"], case["ny"], case["nz"])
        L = tuple(float(np.float32(n * case["spacing"])) for n in Nx)
        rows = [(Nx, L, _blocks(case), 16.0, case["scheme"])]
    out = []
    for r, (Nx, L, blocks, chi, scheme) in enumerate(rows):
        dt = systems.cl_step(min(a / n for a, n in zip(L, Nx)))
        Nr = float(sum(n for n, _ in blocks))
        s = 0 if seed is None else int(seed) * 1009 + r
        out.append((dict(Nx=Nx, L=L, Nr=Nr, C=50.0, nspecies=2, cl=True, seed=s,
                         potentials=[dict(kind="Helfand", kappaN=100.0, dt_pl=dt, scheme=scheme),
                                     dict(kind="Flory", I=0, J=1, chiN=chi, dt_pl=dt, dt_mi=dt, scheme=scheme)],
                         molecules=[dict(blocks=blocks, phi=1.0)]), s))
    return out


def _fields(spec, seed):
    """w+ of the excluded volume, w+ and w- of the exchange: real parts N(0, 0.1^2), imaginary parts zero."""
    rng = np.random.default_rng(seed)
    M = int(np.prod(spec["Nx"]))
    return [(rng.standard_normal(M, np.float32) * np.float32(0.1)).astype(np.complex64) for _ in range(3)]


def _per_species(case):
    V = case["nx"] * case["ny"] * case["nz"] * case["spacing"] ** 3
    return max(8, int(case["density"] * V / 2))


def _c3(v, t):
    return (t * 3)(*v)


def prepare(case, seed):
    k = case["kind"]
    if k in ("tild", "replicas"):
        engines = []
        for r in range(case.get("replicas", 1)):
            cfg = _tild(case, seed * 131 + r)
            engines.append(systems.tild_engine(cfg, case["integrator"]))
        return dict(case=case, engines=engines, group=mft.TildGroup(engines) if k == "replicas" else None)
    if k == "fts":
        spec, s = _specs(case, seed)[0]
        f = _fields(spec, s)
        return dict(case=case, sys=systems.fts_system(spec, {(0, "pl"): f[0], (1, "pl"): f[1], (1, "mi"): f[2]}))
    if k == "sweep":
        specs = _specs(case, seed)
        b = mft.FtsBatch([s for s, _ in specs])
        for r, (spec, s) in enumerate(specs):
            f = _fields(spec, s)
            b.set_fields(r, 0, f[0])
            b.set_fields(r, 1, f[1], f[2])
        b.init()
        return dict(case=case, batch=b)
    Nx = (case["nx"], case["ny"], case["nz"])
    M = Nx[0] * Nx[1] * Nx[2]
    L = tuple(float(np.float32(n * case.get("spacing", 0.125))) for n in Nx)
    st = dict(case=case, M=M, Nx=_c3(Nx, ctypes.c_int), L=_c3(L, ctypes.c_float))
    if k == "fft":
        plan = ctypes.c_void_p()
        mft.check(mft.lib().mft_fft_plan_create(ctypes.byref(plan), *Nx, case["batch"]))
        a = _fft_input(case, seed)
        return dict(st, plan=plan, a=a, f=torch.empty_like(a), b=torch.empty_like(a))
    if k == "particles":
        n = _per_species(case)
        G = (case["pme"] + 1) ** 3
        x = _mesh_input(case, L, seed)
        e = lambda *s: torch.empty(*s, dtype=torch.float32, device=GPU)  # noqa: E731
        fk = []
        for A in _mesh_amplitudes(case, L):
            u, f = e(M, 2), e(M, 3, 2)
            mft.check(mft.lib().mft_tild_kspace_table(_p(u), _p(f), 0, ctypes.c_float(A), ctypes.c_float(math.sqrt(0.5)),
                                                      ctypes.c_float(0.0), st["Nx"], st["L"], None))
            fk.append(f)
        sites = torch.arange(2 * n, dtype=torch.int32, device=GPU)
        return dict(st, n=n, G=G, x=x, W=e(2 * n, G), I=torch.empty(2 * n, G, dtype=torch.int32, device=GPU), rho=e(2, M),
                    F=e(2, M, 3), f=e(2 * n, 3), fk=fk, sites=sites, work=e(4 * M),
                    dx=_c3([a / b for a, b in zip(L, Nx)], ctypes.c_float),
                    gvol=float(np.float32(L[0] * L[1] * L[2] / M)))
    n = sum(x for x, _ in _blocks(case))
    W, V = _chain_input(case, seed), L[0] * L[1] * L[2]
    e = lambda *s: torch.empty(*s, dtype=torch.complex64, device=GPU)  # noqa: E731
    g = e(M)
    mft.check(mft.lib().mft_fts_bond_factor(_p(g), st["Nx"], st["L"], ctypes.c_double(float(n)), None))
    mol = mft.FtsMoleculeC()
    mol.nblocks, mol.phi = len(_blocks(case)), 1.0
    for j, (b, s) in enumerate(_blocks(case)):
        mol.N[j], mol.species[j] = b, s
    return dict(st, W=W, g=g, mol=mol, q=e(n, M), qd=e(n, M), rho=e(2, M), V=V, gvol=V / M, nmol=50.0 * V,
                work=torch.empty(4 * ((M + 255) // 256), dtype=torch.float64, device=GPU))


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _gen(seed):
    g = torch.Generator(device=GPU)
    g.manual_seed(int(seed))
    return g


def _fft_input(case, seed):
    shape = (case["batch"], case["nz"], case["ny"], case["nx"])
    return torch.randn(shape, dtype=torch.complex64, device=GPU, generator=_gen(seed))


def _mesh_input(case, L, seed):
    """Uniform particles of two species; the first half of the ids is species 0."""
    r = torch.rand(2 * _per_species(case), 3, dtype=torch.float32, device=GPU, generator=_gen(seed))
    return (r * torch.tensor(L, dtype=torch.float32, device=GPU)).contiguous()


def _mesh_amplitudes(case, L):
    rho0 = 2 * _per_species(case) / (L[0] * L[1] * L[2])
    return [float(np.float32(50.0 / (2 * rho0))), float(np.float32(51.0 / rho0))]


def _chain_input(case, seed):
    """Species fields as a solve has them: per bead, real part within some tenths over the chain's length."""
    M = case["nx"] * case["ny"] * case["nz"]
    n = sum(x for x, _ in _blocks(case))
    return (torch.randn(2, M, dtype=torch.complex64, device=GPU, generator=_gen(seed)) * (3.0 / n)).contiguous()


# -------------------------------------------------------------------- run ----
def run(st):
    case = st["case"]
    k, lib = case["kind"], mft.lib()
    if k == "tild":
        e = st["engines"][0]
        pe, be = e.step_energies(case["steps"])
        return {"pair": pe, "bond": be, "force": e.compute_forces()}
    if k == "replicas":
        st["group"].step(case["steps"])
        return {"energy": [e.energies() for e in st["engines"]], "force": [e.compute_forces() for e in st["engines"]]}
    if k == "fts":
        s = st["sys"]
        s.step(case["iterations"])
        Q, _, parts = s.observables()
        return {"Q": Q, "H": parts, "rho": s.densities(), "w": [s.get_fields(0), *s.get_fields(1, minus=True)]}
    if k == "sweep":
        b = st["batch"]
        b.step(case["iterations"])
        obs = [b.observables(r) for r in range(case["replicas"])]
        return {"Q": np.array([o[0] for o in obs]), "H": np.array([o[2] for o in obs]),
                "rho": [b.densities(r) for r in range(case["replicas"])],
                "w": [b.get_fields(r, 1, minus=True)[1] for r in range(case["replicas"])]}
    if k == "fft":
        mft.check(lib.mft_fft_exec(st["plan"], _p(st["a"]), _p(st["f"]), 1, None))
        mft.check(lib.mft_fft_exec(st["plan"], _p(st["f"]), _p(st["b"]), -1, None))
        return st["f"], st["b"]
    if k == "particles":
        n, G, M = st["n"], st["G"], st["M"]
        mft.check(lib.mft_tild_grid_weights(_p(st["W"]), _p(st["I"]), _p(st["x"]), 2 * n, st["Nx"], st["dx"], case["pme"],
                                            None))
        st["rho"].zero_()
        st["F"].zero_()
        st["f"].zero_()
        sites = [ctypes.c_void_p(st["sites"].data_ptr() + 4 * n * s) for s in range(2)]
        for s in range(2):
            mft.check(lib.mft_tild_fill_density(_p(st["rho"][s]), None, None, sites[s], n, 2 * n, _p(st["I"]), _p(st["W"]),
                                                G, M, None))
        for s in range(2):
            for t in range(2):  # a species on itself counts twice
                mft.check(lib.mft_tild_pair_force(_p(st["F"][s]), _p(st["rho"][t]), _p(st["fk"][int(s != t)]), st["Nx"],
                                                  ctypes.c_float(2.0 if s == t else 1.0), _p(st["work"]), None))
        for s in range(2):
            mft.check(lib.mft_tild_map_forces(_p(st["f"]), _p(st["F"][s]), None, sites[s], n, 2 * n, _p(st["I"]),
                                              _p(st["W"]), G, ctypes.c_float(st["gvol"]), M, None))
        return {"index": st["I"], "weight": st["W"], "rho": st["rho"], "F": st["F"], "f": st["f"]}
    Q = (ctypes.c_double * 2)()
    last = st["q"][-1]
    M = ctypes.c_long(st["M"])
    mft.check(lib.mft_fts_propagate(_p(st["q"]), _p(st["qd"]), _p(st["W"]), _p(st["g"]), ctypes.byref(st["mol"]), st["Nx"],
                                    None))
    mft.check(lib.mft_fts_partition_function(Q, _p(last), ctypes.c_double(st["gvol"]), ctypes.c_double(st["V"]), M,
                                             _p(st["work"]), None))
    f = st["nmol"] / (complex(Q[0], Q[1]) * st["V"])
    st["rho"].zero_()
    mft.check(lib.mft_fts_density(_p(st["rho"]), _p(st["q"]), _p(st["qd"]), _p(st["W"]), ctypes.byref(st["mol"]),
                                  ctypes.c_double(f.real), ctypes.c_double(f.imag), M, None))
    return {"Q": np.array([Q[0], Q[1]]), "q": st["q"], "qdag": st["qd"], "rho": st["rho"]}


# ------------------------------------------------------------------ exact ----
def exact(case, seed):
    """The same outputs in 64 bits, plain torch."""
    k = case["kind"]
    if k == "tild":
        return _exact_tild(case, _tild(case, seed * 131))
    if k == "replicas":
        got = [_exact_tild(case, _tild(case, seed * 131 + r), final=True) for r in range(case["replicas"])]
        return {"energy": [(g["pair"], g["bond"]) for g in got], "force": [g["force"] for g in got]}
    if k in ("fts", "sweep"):
        got = [_exact_fts(spec, _fields(spec, s), case["iterations"]) for spec, s in _specs(case, seed)]
        if k == "fts":
            return got[0]
        return {"Q": np.array([g["Q"] for g in got]), "H": np.array([g["H"] for g in got]), "rho": [g["rho"] for g in got],
                "w": [g["w"][2] for g in got]}
    L = tuple(float(np.float32(case[a] * case.get("spacing", 0.125))) for a in ("nx", "ny", "nz"))
    if k == "fft":
        a = _fft_input(case, seed).to(torch.complex128)
        f = torch.fft.fftn(a, dim=(1, 2, 3), norm="forward")
        return f, a
    if k == "particles":
        return _exact_particles(case, L, seed)
    W = _chain_input(case, seed).to(torch.complex128)
    blocks = _blocks(case)
    shape = (case["nz"], case["ny"], case["nx"])
    n = float(sum(x for x, _ in blocks))
    q, qd = _propagate(W, blocks, shape, _bond_factor(shape, L, n))
    Q = q[-1].mean()
    rho = _densities(q, qd, W, blocks, 50.0 / Q)
    return {"Q": torch.view_as_real(Q).cpu().numpy(), "q": q, "qdag": qd, "rho": rho}


def _kvec(shape, L):
    """k components (z, y, x order of the grid), the Nyquist index negative."""
    out = []
    for n, l in zip(shape, L[::-1]):
        i = torch.arange(n, device=GPU, dtype=torch.float64)
        out.append(2.0 * math.pi * torch.where(2 * i < n, i, i - n) / l)
    kz, ky, kx = out
    return kz[:, None, None], ky[None, :, None], kx[None, None, :]


def _bond_factor(shape, L, Nr):
    kz, ky, kx = _kvec(shape, L)
    return torch.exp(-(kx * kx + ky * ky + kz * kz) / (Nr - 1.0))


def _propagate(W, blocks, shape, g):
    E = torch.exp(-W)
    seq = [s for n, s in blocks for _ in range(n)]
    out = []
    for order in (seq, seq[::-1]):
        q = torch.empty(len(seq), W.shape[1], dtype=torch.complex128, device=GPU)
        q[0] = E[order[0]]
        for s in range(1, len(seq)):
            q[s] = E[order[s]] * torch.fft.ifftn(g * torch.fft.fftn(q[s - 1].reshape(shape))).reshape(-1)
        out.append(q)
    return out


def _densities(q, qd, W, blocks, factor):
    rho = torch.zeros(2, W.shape[1], dtype=torch.complex128, device=GPU)
    s, n = 0, q.shape[0]
    for b, sp in blocks:
        acc = torch.zeros(W.shape[1], dtype=torch.complex128, device=GPU)
        for j in range(s, s + b):
            acc += q[j] * qd[n - 1 - j]
        rho[sp] += factor * torch.exp(W[sp]) * acc
        s += b
    return rho


def _philox_normal(n, c1, c2, c3, seed):
    """Four normals for each of n counters: Philox4x32-10, Box-Muller on 24-bit uniforms."""
    m32 = 0xFFFFFFFF

    def mul(a, x):  # (high, low) words of the product of two 32-bit words
        ah, al, xh, xl = a >> 16, a & 0xFFFF, x >> 16, x & 0xFFFF
        low, m1, m2 = al * xl, ah * xl, al * xh
        mid = (low >> 16) + (m1 & 0xFFFF) + (m2 & 0xFFFF)
        return ah * xh + (m1 >> 16) + (m2 >> 16) + (mid >> 16), ((mid & 0xFFFF) << 16) | (low & 0xFFFF)

    c = [torch.arange(n, device=GPU, dtype=torch.int64)] + [torch.full((n,), int(v) & m32, device=GPU, dtype=torch.int64)
                                                            for v in (c1, c2, c3)]
    k0, k1 = int(seed) & m32, (int(seed) >> 32) & m32
    for _ in range(10):
        h0, l0 = mul(0xD2511F53, c[0])
        h1, l1 = mul(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & m32, (k1 + 0xBB67AE85) & m32
    z = []
    for h in range(2):
        u1 = ((c[2 * h] >> 8) + 1).double() * 2.0 ** -24
        u2 = (c[2 * h + 1] >> 8).double() * 2.0 ** -24
        r = torch.sqrt(-2.0 * torch.log(u1))
        z += [r * torch.cos(2 * math.pi * u2), r * torch.sin(2 * math.pi * u2)]
    return z


def _exact_fts(spec, fields, iterations):
    shape, L, Nr, C = spec["Nx"][::-1], spec["L"], spec["Nr"], spec["C"]
    M = int(np.prod(shape))
    V = L[0] * L[1] * L[2]
    gvol = V / M
    P, F = spec["potentials"]
    blocks = spec["molecules"][0]["blocks"]
    g = _bond_factor(shape, L, Nr)
    wh, wp, wm = [torch.from_numpy(f).to(GPU).to(torch.complex128) for f in fields]
    nmol = C * V * Nr / sum(n for n, _ in blocks)

    def species():
        return torch.stack([(1j * (wh + wp) - wm) / Nr, (1j * (wh + wp) + wm) / Nr])

    def density():
        q, qd = _propagate(species(), blocks, shape, g)
        Q = q[-1].mean()
        return _densities(q, qd, species(), blocks, nmol / (V * Q)), Q

    def force(rho):
        tot = rho[0] + rho[1]
        return (C / P["kappaN"] * wh + 1j * (tot / Nr - C), 2 * C / F["chiN"] * wp + 1j * tot / Nr,
                2 * C / F["chiN"] * wm + (rho[1] - rho[0]) / Nr)

    rho, Q = density()
    dts = (P["dt_pl"], F["dt_pl"], F["dt_mi"])
    for it in range(iterations):
        z = _philox_normal(M, it, 0x4654534E, 0, spec["seed"])
        noise = [math.sqrt(2 * dt / gvol) * z[j] for j, dt in enumerate(dts)]
        old, f = (wh, wp, wm), force(rho)
        wh, wp, wm = [w - dt * a + n for w, dt, a, n in zip(old, dts, f, noise)]
        rho, Q = density()
        if P.get("scheme") == "EMPC":
            f2 = force(rho)
            wh, wp, wm = [w - 0.5 * dt * (a + b) + n for w, dt, a, b, n in zip(old, dts, f, f2, noise)]
            rho, Q = density()
    H = [(wh * wh).sum() * gvol * C / 2 / P["kappaN"] - 1j * C * wh.sum() * gvol,
         ((wp * wp).sum() + (wm * wm).sum()) * gvol * C / F["chiN"], -nmol * torch.log(Q)]
    return {"Q": torch.stack([Q]).cpu().numpy(), "H": torch.stack(H).cpu().numpy(), "rho": rho.cpu().numpy(),
            "w": [w.cpu().numpy() for w in (wh, wp, wm)]}


def _splines(x, dx, p):
    """Base grid index and the p + 1 cardinal B-spline weights of every coordinate."""
    if p % 2 == 0:
        g = torch.floor(x / dx + 0.5)
        s = x / dx - g
    else:
        g = torch.floor(x / dx)
        s = x / dx - g - 0.5
    if p == 1:
        w = [0.5 - s, 0.5 + s]
    elif p == 2:
        w = [0.5 * (0.5 - s) ** 2, 0.75 - s * s, 0.5 * (0.5 + s) ** 2]
    else:
        w = [(1 - 2 * s) ** 3 / 48, (23 - 30 * s - 12 * s ** 2 + 24 * s ** 3) / 48,
             (23 + 30 * s - 12 * s ** 2 - 24 * s ** 3) / 48, (1 + 2 * s) ** 3 / 48]
    return g.long(), w


def _stencil(x, Nx, L, p):
    """Grid indices and weights [points of the stencil] of every particle, x outermost, z innermost."""
    ax = [_splines(x[:, j], L[j] / Nx[j], p) for j in range(3)]
    n = [[torch.remainder(ax[j][0] + o - p // 2, Nx[j]) for o in range(p + 1)] for j in range(3)]
    for a in range(p + 1):
        for b in range(p + 1):
            wab, nab = ax[0][1][a] * ax[1][1][b], n[0][a] + Nx[0] * n[1][b]
            for c in range(p + 1):
                yield nab + Nx[0] * Nx[1] * n[2][c], wab * ax[2][1][c]


def _exact_tild(case, cfg, final=False):
    """final: the energies at the positions the steps end with, not at those the last step starts from."""
    Nx, L, p, ns = cfg["Nx"], cfg["L"], cfg["pmeorder"], len(cfg["species"])
    M, V = Nx[0] * Nx[1] * Nx[2], L[0] * L[1] * L[2]
    gvol, shape = V / M, Nx[::-1]
    t = cfg["topo"]
    type_ = torch.from_numpy(t["type"]).to(GPU).long()
    q = torch.from_numpy(t["charge"]).to(GPU).double() if cfg["has_charges"] else None
    Lt = torch.tensor(L, dtype=torch.float64, device=GPU)
    x = torch.from_numpy(cfg["x"].reshape(-1, 3)).to(GPU).double()
    N = x.shape[0]
    has = torch.from_numpy((np.arange(2)[None, :] < t["nBonds"][:, None])).to(GPU)
    to = torch.from_numpy(t["bondedTo"].reshape(-1, 2)).to(GPU).long()
    kz, ky, kx = _kvec(shape, L)
    k2 = kx * kx + ky * ky + kz * kz
    u = []
    for P in cfg["potentials"]:
        if P["kind"] == "gaussian":
            u.append(P["A"] * torch.exp(-0.5 * k2 * P["sigma"] ** 2))
        else:
            u.append(torch.where(k2 > 0, 4 * math.pi * P["A"] / k2 * torch.exp(-k2 * P["sigma"] ** 2), torch.zeros_like(k2)))

    def bonds():
        f, e = torch.zeros_like(x), 0.0
        for b in range(2):
            d = x - x[to[:, b]]
            d -= Lt * torch.round(d / Lt)
            d *= has[:, b, None]
            f -= 2 * cfg["bond_k"][0] * d
            e = e + cfg["bond_k"][0] * (d * d).sum()
        return f, float(0.5 * e)

    def forces():
        rho = torch.zeros(ns * M, dtype=torch.float64, device=GPU)
        for g, w in _stencil(x, Nx, L, p):
            rho.index_add_(0, g + M * type_, w / gvol)
        rho = rho.reshape(ns, *shape)
        rk = torch.fft.fftn(rho, dim=(1, 2, 3), norm="forward")
        rq = None
        if q is not None:
            qs = [float(q[type_ == s][0]) if bool((type_ == s).any()) else 0.0 for s in range(ns)]
            rq = sum(qs[s] * rk[s] for s in range(ns))
        e, zk = [], [torch.zeros_like(rk[0]) for _ in range(ns)]
        for P, uk in zip(cfg["potentials"], u):
            if P["kind"] == "gaussian":
                i, j = int(math.log2(P["maskI"])), int(math.log2(P["maskJ"]))
                e.append(float(V * (rk[i].conj() * uk * rk[j]).real.sum()))
                zk[i] += uk * rk[j]
                zk[j] += uk * rk[i]
            else:
                e.append(float(0.5 * V * (rq.conj() * uk * rq).real.sum()))
                for s in range(ns):
                    zk[s] += qs[s] * uk * rq
        f = torch.zeros_like(x)
        F = torch.empty(3, ns * M, dtype=torch.float64, device=GPU)
        for s in range(ns):
            for j, kj in enumerate((kx, ky, kz)):
                F[j, s * M:(s + 1) * M] = torch.fft.ifftn(-1j * kj * zk[s], norm="forward").real.reshape(-1)
        for g, w in _stencil(x, Nx, L, p):
            at = g + M * type_
            for j in range(3):
                f[:, j] += F[j, at] * w
        return f, e

    dt = float(np.float32(cfg["delt"]))
    b = 1.0 / (1.0 + dt / 2.0)
    a = (1.0 - dt / 2.0) / (1.0 + dt / 2.0)
    nm = math.sqrt(2.0 * dt)
    xo, no = x.clone(), torch.zeros_like(x)
    for step in range(case["steps"]):
        fp, e = forces()
        f = fp + bonds()[0]
        z = torch.stack(_philox_normal(N, step, 0x54494C44, 0, cfg["seed"])[:3], dim=1) * nm
        if case["integrator"] == "GJF":
            xo = xo - Lt * torch.round((xo - x) / Lt)
            new = 2 * b * x - a * xo + b * dt * dt * f + b * dt / 2 * (z + no)
            xo, no = x, z
        else:
            new = x + dt * f + z
        x = torch.remainder(new, Lt)
    fp, last = forces()
    fb, eb = bonds()
    return {"pair": np.array(last if final else e), "bond": eb, "force": (fp + fb).reshape(-1).cpu().numpy()}


def _exact_particles(case, L, seed):
    Nx = (case["nx"], case["ny"], case["nz"])
    M, p, n = Nx[0] * Nx[1] * Nx[2], case["pme"], _per_species(case)
    gvol, shape = L[0] * L[1] * L[2] / M, Nx[::-1]
    x = _mesh_input(case, L, seed).double()
    half = [slice(0, n), slice(n, 2 * n)]
    st = list(_stencil(x, Nx, L, p))
    rho = torch.zeros(2, M, dtype=torch.float64, device=GPU)
    for g, w in st:
        for s in range(2):
            rho[s].index_add_(0, g[half[s]], w[half[s]] / gvol)
    kz, ky, kx = _kvec(shape, L)
    shape_k = torch.exp(-0.25 * (kx * kx + ky * ky + kz * kz))
    A = _mesh_amplitudes(case, L)
    rk = torch.fft.fftn(rho.reshape(2, *shape), dim=(1, 2, 3), norm="forward")
    F = torch.empty(2, M, 3, dtype=torch.float64, device=GPU)
    for s in range(2):
        zk = shape_k * (2.0 * A[0] * rk[s] + A[1] * rk[1 - s])
        for j, kj in enumerate((kx, ky, kz)):
            F[s, :, j] = torch.fft.ifftn(-1j * kj * zk, norm="forward").real.reshape(-1)
    f = torch.zeros(2 * n, 3, dtype=torch.float64, device=GPU)
    for g, w in st:
        for s in range(2):
            f[half[s]] += F[s][g[half[s]]] * w[half[s], None]
    # no value for the tables: a particle on a cell's edge takes the cell that its 32-bit position falls into
    return {"index": None, "weight": None, "rho": rho, "F": F, "f": f}
