"""Groups of a batch run side by side on the batch's streams: more grids and
update schemes than streams, replayed from the captured graph with host reads and
the program's own steps between, give the bits of each replica alone."""
import numpy as np
import pytest

from mft import systems

pytestmark = pytest.mark.gpu


def spec(r, grid, scheme="EM", zero_mean=False):
    s, f = systems.fts_diblock(grid_shape=grid, L=tuple(0.12 * n for n in grid), Nr=14.0, NA=5 + r % 3, NB=9 - r % 3,
                               dt=1e-3, seed=70 + r)
    for p in s["potentials"]:
        p["scheme"] = scheme
    s["potentials"][0]["zero_mean"] = zero_mean
    return s, f


@pytest.mark.parametrize("ngroups", [1, 2, 4, 6])
def test_groups_side_by_side_equal_replicas_alone(gpu, ngroups):
    kinds = [((16, 16, 16), "EM", False), ((24, 16, 20), "EMPC", False), ((12, 10, 8), "EM", False),
             ((16, 16, 16), "1S", False), ((32, 20, 16), "EM", True), ((20, 20, 12), "EM", False)][:ngroups]
    reps = [spec(r, *kinds[r % ngroups]) for r in range(ngroups + 2)]
    b = gpu.FtsBatch([s for s, _ in reps])
    alone = [systems.fts_system(s, f) for s, f in reps]
    for k, (s, f) in enumerate(reps):
        systems.load_fields(b.set_fields, s, f, rep=k)
    b.init()
    for n in (1, 4, 3):
        b.step(n)
        for k, a in enumerate(alone):
            a.step(n)
            assert np.array_equal(a.densities(), b.densities(k)), (n, k)
            assert np.array_equal(a.observables()[0], b.observables(k)[0]), (n, k)
    for a in alone:
        a.close()
    b.close()
