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
