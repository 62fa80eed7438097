"""The one-launch-per-bead propagator kernel over its plane shapes: every line
length it takes along x and along the other two axes, cubes and slabs, against
the FP64 oracle.

Tolerance: a bead of this kernel rounds some eight times per axis (orbit sums,
products, the joining sums) and once for e^{-W}; over the 5 beads of the chain
that is a random walk of about 100 roundings of 2^-25 relative to the largest
value, at most about five standard deviations over the points: 1.5e-6.
"""
import numpy as np
import pytest

import orc
from mft import systems
from test_gpu_fts import build, rel, say
from test_oracle_fts import random_fields, tiny_spec

pytestmark = pytest.mark.gpu

LENGTHS = (16, 20, 24, 32, 40, 48, 64, 80, 96, 128)
GRIDS = [(n, 16, 20) for n in LENGTHS] + [(24, n, 16) for n in LENGTHS] + [(20, 16, n) for n in LENGTHS] + [
    (48, 48, 24), (40, 80, 16), (96, 20, 64), (128, 128, 16), (16, 128, 96)]


@pytest.mark.parametrize("grid", sorted(set(GRIDS)))
@pytest.mark.parametrize("blocks", [((2, 0), (3, 1)), ((1, 0), (3, 1), (1, 0))])
def test_bead_kernel_matches_oracle(gpu, grid, blocks):
    spec = tiny_spec(Nx=grid, L=tuple(0.14 * n for n in grid), blocks=blocks)
    say("case: bead kernel", grid, blocks)
    s, o = build(gpu, spec, random_fields(spec, 0.3, seed=7))
    q, qd = s.propagators(0)
    ref = orc.fts_molecule_densities(o, keep=True)[0]
    e = rel(q, ref["q"]), rel(qd, ref["qdag"]), rel(s.densities(), o.rho)
    s.close()
    say("  q %.2e qdag %.2e rho %.2e" % e)
    assert max(e) < 1.5e-6


@pytest.mark.parametrize("grid", [(16, 20, 24), (48, 48, 48), (96, 16, 80), (32, 128, 40)])
def test_a_constant_slice_stays_the_constant(gpu, grid):
    """Zero fields: every bead is 1 to the bit, and Q = M gvol / V up to the roundings of that factor in double."""
    spec = tiny_spec(Nx=grid, L=tuple(0.1 * n for n in grid), blocks=((20, 0), (15, 1)))
    s = gpu.FtsSystem(spec)
    s.init()
    q, qd = s.propagators(0)
    Q = s.observables()[0]
    s.close()
    assert np.array_equal(q, np.ones_like(q)) and np.array_equal(qd, np.ones_like(qd))
    assert abs(Q[0] - 1.0) < 8 * 2.0 ** -53


def test_chains_past_the_inline_descriptors_give_the_same_bits(gpu):
    """A batch with more chains than travel as kernel arguments = each alone."""
    reps = []
    for r in range(6):
        spec, f = systems.fts_diblock(grid_shape=(24, 16, 20), L=(2.4, 1.6, 2.0), Nr=12.0, NA=3 + r, NB=9 - r, dt=1e-3,
                                      seed=50 + r)
        reps.append((spec, f))
    b = gpu.FtsBatch([s for s, _ in reps])
    for k, (spec, f) in enumerate(reps):
        systems.load_fields(b.set_fields, spec, f, rep=k)
    b.init()
    b.step(2)
    for k, (spec, f) in enumerate(reps):
        s = systems.fts_system(spec, f)
        s.step(2)
        assert np.array_equal(s.densities(), b.densities(k)), k
        s.close()
    b.close()
