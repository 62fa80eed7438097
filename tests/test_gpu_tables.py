"""Table kernels and the pair force of the per-kernel entry points where their
work split has edges: particle counts around a workgroup's share, every spline
order, table rows that are no multiple of the lanes that share them, site lists
with entries out of range, and grids down to two points with a k-space table of
no symmetry.

Tolerances: a mapped force adds G <= 125 products in float, at most G + 8
roundings of 2^-24 relative to the sum of their magnitudes; the pair force is
three float transforms of at most log2(M) <= 16 levels each way, 4 roundings of
2^-24 a level and an rms growth of its square root, within 2e-6 normwise.
"""
import ctypes

import numpy as np
import pytest

import orc
from test_gpu_fts import rel, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("ns", [1, 31, 32, 33, 257])
def test_tables_around_a_workgroups_share(gpu, p, ns):
    rng = np.random.default_rng(100 * p + ns)
    Nx, L = (12, 10, 16), np.array([4.0, 3.0, 5.0], np.float32)
    dx = (L / np.array(Nx, np.float32)).astype(np.float32)
    x = (rng.random((ns, 3)) * L).astype(np.float32).reshape(-1)
    G, M, gvol = (p + 1) ** 3, int(np.prod(Nx)), float(np.prod(dx.astype(np.float64)))
    inds, W = gpu.grid_weights(x, Nx, dx, p)
    inds_o, W_o = orc.grid_weights(x, Nx, dx, p)
    assert np.array_equal(inds, inds_o)
    assert rel(W, W_o) < 1e-6  # three weights, a product and a division
    # a group of every second particle, with sites that are no particles
    sites = np.concatenate([np.arange(0, ns, 2), [-1, ns, ns + 7]]).astype(np.int32)
    q = rng.normal(size=ns).astype(np.float32)
    Wd = W.astype(np.float64).reshape(ns, G)
    rho, rhoq = gpu.fill_density(M, sites, inds, W, G, q=q)
    own = np.arange(0, ns, 2)
    want, wantq = np.zeros(M), np.zeros(M)
    np.add.at(want, inds.reshape(ns, G)[own], Wd[own])
    np.add.at(wantq, inds.reshape(ns, G)[own], Wd[own] * q[own, None])
    # fixed point of 2^-32 a product, one rounding of the sum
    lim = len(own) * G * 2.0 ** -33
    assert np.max(np.abs(rho - want)) <= lim + 2.0 ** -24 * np.max(np.abs(want))
    assert np.max(np.abs(rhoq - wantq)) <= lim + 2.0 ** -23 * np.max(np.abs(Wd)) * 4 * len(own)
    F = rng.normal(size=(M, 3)).astype(np.float32)
    f = gpu.map_forces(ns, F.reshape(-1), sites, inds, W, G, gvol, q=q).reshape(ns, 3)
    terms = F.astype(np.float64)[inds.reshape(ns, G)] * (Wd * gvol)[:, :, None]
    want = terms.sum(1) * q[:, None]
    bound = (G + 8) * 2.0 ** -24 * np.abs(terms).sum(1) * np.abs(q)[:, None]
    assert np.all(np.abs(f - want)[own] <= bound[own])
    assert not f[np.setdiff1d(np.arange(ns), own)].any()


@pytest.mark.parametrize("grid", [(2, 3, 5), (16, 2, 4), (12, 20, 24), (40, 6, 48), (64, 10, 3), (8, 64, 80)])
def test_pair_force_of_a_table_without_symmetry(gpu, grid):
    rng = np.random.default_rng(sum(grid))
    M = int(np.prod(grid))
    rho = rng.normal(size=M).astype(np.float32)
    fk = (rng.normal(size=(M, 3)) + 1j * rng.normal(size=(M, 3))).astype(np.complex64)
    F0 = rng.normal(size=(M, 3)).astype(np.float32)
    got = gpu.pair_force(F0.reshape(-1), rho, fk, grid, factor=1.7).reshape(M, 3)
    sh = grid[::-1]
    S = np.fft.fftn(rho.reshape(sh).astype(np.float64)) / M
    for j in range(3):
        V = np.fft.ifftn(fk[:, j].reshape(sh) * S) * M
        e = rel(got[:, j], F0[:, j] + 1.7 * V.real.reshape(-1))
        say("pair force", grid, j, "%.2e" % e)
        assert e < 2e-6


def test_calls_of_more_threads_than_a_launch_takes(gpu):
    """A launch takes fewer than 2^32 threads.  2^28 + 2000 sites at 16 lanes a site (force map) or 64 entries a
    site (density), nearly all of them empty, and the weights of 2^29 + 37 particles at eight threads each."""
    n, ns, G, Nx = 2 ** 28 + 2000, 700, 64, (12, 10, 16)
    M = int(np.prod(Nx))
    rng = np.random.default_rng(5)
    L = np.array([4.0, 3.0, 5.0], np.float32)
    dx = (L / np.array(Nx, np.float32)).astype(np.float32)
    x = (rng.random((ns, 3)) * L).astype(np.float32)
    inds, W = gpu.grid_weights(x.reshape(-1), Nx, dx, 3)
    F = rng.normal(size=(M, 3)).astype(np.float32)
    own = np.concatenate([np.arange(300), n - 1 - np.arange(300), 2 ** 26 - 50 + np.arange(100)])
    sites = np.full(n, -1, np.int32)
    sites[own] = np.arange(ns, dtype=np.int32)
    few = np.arange(ns, dtype=np.int32)
    say("case: table calls past 2^32 threads")
    assert np.array_equal(gpu.fill_density(M, sites, inds, W, G)[0], gpu.fill_density(M, few, inds, W, G)[0])
    assert np.array_equal(gpu.map_forces(ns, F.reshape(-1), sites, inds, W, G, 0.1),
                          gpu.map_forces(ns, F.reshape(-1), few, inds, W, G, 0.1))
    del sites
    # order 0: one entry a particle; all at the origin but some at either side of a sweep of the grid
    n = 2 ** 29 + 37
    at = np.array([0, 31, 2 ** 28 - 1, 2 ** 28, 2 ** 28 + 33, n - 2, n - 1])
    xd, Wd, Id = gpu.DeviceBuffer(12 * n), gpu.DeviceBuffer(4 * n), gpu.DeviceBuffer(4 * n)
    xd.zero()
    for k, i in enumerate(at):
        gpu.check(gpu.lib().mft_memcpy_h2d(ctypes.c_void_p(xd.ptr.value + 12 * int(i)),
                                           x[k].ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(12)))
    gpu.check(gpu.lib().mft_tild_grid_weights(Wd.ptr, Id.ptr, xd.ptr, n, (ctypes.c_int * 3)(*Nx),
                                              (ctypes.c_float * 3)(*dx), 0, None))
    want, wantW = gpu.grid_weights(x[: at.size].reshape(-1), Nx, dx, 0)
    got = Id.to_array(np.int32, (n,))
    assert np.array_equal(got[at], want)
    got[at] = 0
    assert not got.any()
    got = Wd.to_array(np.float32, (n,))
    assert np.array_equal(got[at], wantW) and np.all(got == wantW[0])
    for b in (xd, Wd, Id):
        b.free()


@pytest.mark.parametrize("grid", [(16, 20, 24), (64, 48, 12), (12, 12, 96)])
def test_pair_force_of_a_density_far_from_zero_mean(gpu, grid):
    """The transforms round relative to the density's fluctuations, not to its mean: the bound of the table without
    symmetry holds for a mean of 200 fluctuations, whose rounding alone would be 200 times 1e-7."""
    rng = np.random.default_rng(sum(grid))
    M, sh = int(np.prod(grid)), grid[::-1]
    rho = (200.0 + rng.normal(size=M)).astype(np.float32)
    k = np.meshgrid(*[2 * np.pi * np.fft.fftfreq(n) for n in sh], indexing="ij")
    u = np.exp(-sum(a * a for a in k))
    fk = np.stack([-1j * a * u for a in k[::-1]], -1).reshape(M, 3).astype(np.complex64)
    got = gpu.pair_force(np.zeros(3 * M, np.float32), rho, fk, grid, factor=1.0).reshape(M, 3)
    S = np.fft.fftn((rho.astype(np.float64) - 200.0).reshape(sh))
    want = np.stack([np.fft.ifftn(fk[:, j].reshape(sh) * S).real.reshape(-1) for j in range(3)], -1)
    e = rel(got, want)
    say("pair force, mean of 200", grid, "%.2e" % e)
    assert e < 2e-6
