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


@pytest.mark.parametrize("grid, beads", [((64, 20, 16), 400), ((16, 96, 20), 400), ((20, 16, 128), 400),
                                         ((48, 16, 24), 400), ((16, 80, 16), 400)])
def test_long_chains_in_a_structured_field(gpu, grid, beads):
    """A lamellar field of +-4 over the chain along the longest axis with noise on it, a saddle point's imaginary w+ and
    400 beads: operands rounded to nearest put each long wave off by 1e-8 to 4e-8 a bead, which adds up to 1e-6.
    e^{-W} is taken as the engine rounds it (bead 0 of either chain): a rounding of the input, the same for every bead.

    Tolerance: a bead's some 25 roundings of 2^-25 a point are 9e-8 rms, and the beads after it average them over a
    volume that grows as their number to the 3/2, so that the sum over the beads stays at two to three times one
    bead's, 2.3e-7; twice that.
    """
    axis = int(np.argmax(grid))
    M, L = int(np.prod(grid)), tuple(float(np.float32(0.125 * n)) for n in grid)
    j = np.meshgrid(*[np.arange(n) / n for n in grid[::-1]], indexing="ij")[::-1]
    noise = np.random.default_rng(beads).normal(size=grid[::-1]) # lines that round alike would not average
    wm = (4.0 * np.cos(2 * np.pi * j[axis]) + noise).astype(np.complex64).reshape(-1)
    wh = (2.0j * np.sin(2 * np.pi * j[axis])).astype(np.complex64).reshape(-1)
    a = beads // 2
    spec = dict(Nx=grid, L=L, Nr=float(beads), C=50.0, nspecies=2, cl=True, seed=1,
                potentials=[dict(kind="Helfand", kappaN=100.0, dt_pl=1e-3),
                            dict(kind="Flory", I=0, J=1, chiN=16.0, dt_pl=1e-3, dt_mi=1e-3)],
                molecules=[dict(blocks=[(a, 0), (beads - a, 1)], phi=1.0)])
    say("case: structured field", grid, beads)
    s = systems.fts_system(spec, {(0, "pl"): wh, (1, "pl"): np.zeros(M, np.complex64), (1, "mi"): wm})
    q, qd = (v.reshape(beads, M) for v in s.propagators(0))
    Q = s.observables()[0][0]
    s.close()
    k = [np.where(2 * np.arange(n) < n, np.arange(n), np.arange(n) - n) * 2 * np.pi / l for n, l in zip(grid, L)]
    k2 = k[2][:, None, None] ** 2 + k[1][None, :, None] ** 2 + k[0][None, None, :] ** 2
    g, E = np.exp(-k2 / (beads - 1.0)), (q[0].astype(complex), qd[0].astype(complex))
    W = [(1j * wh.astype(complex) + c * wm) / beads for c in (-1, 1)]
    assert max(rel(e, np.exp(-w)) for e, w in zip(E, W)) < 1.2e-7  # two roundings: W and e^{-W}
    r = E[0]
    for b in range(1, beads):
        r = E[int(b >= a)] * np.fft.ifftn(g * np.fft.fftn(r.reshape(grid[::-1]))).reshape(-1)
    e = rel(q[-1], r), abs(Q / r.mean() - 1)
    say("  last bead %.2e Q %.2e" % e)
    assert max(e) < 5e-7
