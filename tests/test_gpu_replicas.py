"""Replica groups whose engines share every launch: the same bits as each engine
stepped alone, for boxes of one description with different seeds and topologies,
mixed with boxes that cannot join, through state changes between the calls."""
import numpy as np
import pytest

from mft import systems

pytestmark = pytest.mark.gpu


def state(e):
    return e.get_state() + (e.compute_forces(),)


@pytest.mark.parametrize("grid, box, pme, integrator, charged", [
    (16, 6.0, 3, "GJF", False), (24, 9.0, 2, "EM", False), (32, 10.0, 3, "GJF", True), (40, 12.0, 1, "GJF", False),
    (64, 14.0, 3, "EM", True)])
def test_batched_replicas_equal_engines_alone(gpu, grid, box, pme, integrator, charged):
    def cfg(seed, n=90):
        if charged:
            return systems.tild_coacervate(nchains=n // 2, Nchain=7, nsolvent=301, box=box, grid=grid, pmeorder=pme,
                                           seed=seed)
        return systems.tild_diblock(nchains=n, NA=5, NB=6, box=box, grid=grid, pmeorder=pme, seed=seed)

    # three that batch, one with fewer particles, two more of a second description
    cfgs = [cfg(1), cfg(2), cfg(3, 60), cfg(4), dict(cfg(5), delt=0.004), dict(cfg(6), delt=0.004)]
    alone, grouped = ([systems.tild_engine(c, integrator) for c in cfgs] for _ in range(2))
    grp = gpu.TildGroup(grouped)
    for k, n in enumerate((1, 2, 5)):
        for e in alone:
            e.step(n)
        grp.step(n)
        if k == 1:  # one leaves the others' step, then follows again with a new state
            alone[1].step(1)
            grouped[1].step(1)
        if k == 2:
            continue  # read through the engines' own streams without a synchronisation
        grp.synchronize()
        for a, b in zip(alone, grouped):
            for u, v in zip(state(a), state(b)):
                assert np.array_equal(u, v), (k, n)
    for a, b in zip(alone, grouped):
        for u, v in zip(state(a), state(b)):
            assert np.array_equal(u, v)
    # new positions and another topology for one of them
    topo = dict(cfgs[3]["topo"])
    for e in (alone[3], grouped[3]):
        e.set_topology(topo["type"], topo["charge"] if charged else None, np.zeros_like(topo["nBonds"]),
                       topo["bondedTo"], topo["bondType"])
        e.set_state(cfgs[1]["x"])
    for e in alone:
        e.step(4)
    grp.step(4)
    for a, b in zip(alone, grouped):
        for u, v in zip(state(a), state(b)):
            assert np.array_equal(u, v)
    grp.close()
    for e in alone + grouped:
        e.close()


@pytest.mark.parametrize("counts", [(2,), (3,), (4,), (2, 1), (2, 3)])
def test_two_or_three_large_boxes_and_more(gpu, counts):
    """Up to three boxes over 48 points that would be alone on their streams step there, more of them or small ones
    share launches: either way the bits of each engine alone."""
    cfgs = []
    for k, n in enumerate(counts):  # the first description 64 points, the second 24
        cfgs += [systems.tild_diblock(nchains=120 - 20 * k, NA=5, NB=6, box=(14.0, 8.0)[k], grid=(64, 24)[k],
                                      seed=10 * k + r) for r in range(n)]
    alone, grouped = ([systems.tild_engine(c, "GJF") for c in cfgs] for _ in range(2))
    grp = gpu.TildGroup(grouped)
    for n in (1, 3, 2):
        for e in alone:
            e.step(n)
        grp.step(n)
    for a, b in zip(alone, grouped):
        for u, v in zip(state(a), state(b)):
            assert np.array_equal(u, v), counts
    grp.close()
    for e in alone + grouped:
        e.close()


def engine(cfg, integrator, bonds):
    t = cfg["topo"]
    import mft
    e = mft.TildEngine(cfg["Nx"], cfg["L"], cfg["pmeorder"], len(cfg["species"]), t["type"].size, cfg["potentials"],
                       bonds["k"], bonds["r0"], bonds["style"], integrator=integrator, delt=cfg["delt"],
                       mass=cfg["mass"], mobility=cfg["mobility"], seed=cfg["seed"])
    e.set_topology(t["type"], None, t["nBonds"], t["bondedTo"], t["bondType"])
    e.set_state(cfg["x"])
    return e


@pytest.mark.parametrize("grid, box, style, erf", [(24, 9.0, 0, True), (20, 8.0, 1, True), (40, 13.0, 1, False),
                                                   (48, 15.0, 0, True)])
def test_batched_tables_bond_kinds_and_scan_sizes(gpu, grid, box, style, erf):
    """Shared launches with potentials that are tables, two bond types, FENE bonds (style 1), and key counts on either
    side of what one workgroup scans (16 384: 40^3 in bricks of 8 has 16 000, 48^3 27 648)."""
    cfgs = []
    for seed in range(4):
        c = systems.tild_diblock(nchains=150, NA=5, NB=6, box=box, grid=grid, seed=40 + seed)
        c["topo"]["bondType"] = (np.arange(c["topo"]["bondType"].size) // 22 % 2).astype(np.int32)
        if erf:
            c["potentials"] = c["potentials"] + [dict(kind="erf2", maskI=1, maskJ=2, A=0.3, sigma=0.4, Rp=0.6)]
        cfgs.append(c)
    bonds = dict(k=[1.5, 2.5], r0=[0.0, 0.3] if style == 0 else [9.0, 10.0], style=[0, style])
    alone, grouped = ([engine(c, "GJF", bonds) for c in cfgs] for _ in range(2))
    grp = gpu.TildGroup(grouped)
    for n in (1, 4):
        for e in alone:
            e.step(n)
        grp.step(n)
        for a, b in zip(alone, grouped):
            for u, v in zip(state(a), state(b)):
                assert np.isfinite(u).all() and np.array_equal(u, v), n
    grp.close()
    for e in alone + grouped:
        e.close()
