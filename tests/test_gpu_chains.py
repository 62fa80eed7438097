"""mft_fts_propagate over the grids its two forms take (x-y planes in one
workgroup, or line passes), every subset of its outputs, and blocks whose species
starts no chain, against the transforms of numpy in FP64.

Tolerance: each bead is a forward and an inverse float transform (at most 16
levels each, four roundings of 2^-24 a level adding up as a random walk: rms
5e-7), the product with g and with exp(-W); over the 6 beads normwise 3e-6.
"""
import ctypes

import numpy as np
import pytest

from test_gpu_fts import rel, say

pytestmark = pytest.mark.gpu

PLANES = [(n, n, z) for n, z in zip((16, 20, 24, 32, 40, 48, 64, 80, 96, 128), (3, 2, 5, 12, 4, 6, 10, 2, 4, 3))]
LINES = [(2, 3, 5), (12, 12, 8), (16, 20, 24), (64, 48, 5), (160, 160, 2), (6, 96, 10)]


def chains(gpu, W, g, blocks, Nx, want):
    """(q, qdag) with the outputs not in `want` null; want = 'same' gives one array for both."""
    M, n = int(np.prod(Nx)), sum(b for b, _ in blocks)
    mol = gpu.FtsMoleculeC()
    mol.nblocks = len(blocks)
    for j, (b, s) in enumerate(blocks):
        mol.N[j], mol.species[j] = b, s
    Wb, gb = gpu.DeviceBuffer.from_array(W.astype(np.complex64)), gpu.DeviceBuffer.from_array(g.astype(np.complex64))
    q, qd = gpu.DeviceBuffer(8 * M * n), gpu.DeviceBuffer(8 * M * n)
    gpu.check(gpu.lib().mft_fts_propagate(
        qd.ptr if want == "same" else (q.ptr if "q" in want else None), qd.ptr if want == "same" or "d" in want else None,
        Wb.ptr, gb.ptr, ctypes.byref(mol), (ctypes.c_int * 3)(*Nx), None))
    return q.to_array(np.complex64, (n, M)), qd.to_array(np.complex64, (n, M))


@pytest.mark.parametrize("grid", PLANES + LINES)
@pytest.mark.parametrize("blocks, want", [(((2, 0), (3, 1), (1, 0)), "qd"), (((2, 0), (2, 2), (2, 1)), "qd"),
                                          (((3, 1), (3, 0)), "q"), (((3, 1), (3, 0)), "d"), (((3, 1), (3, 0)), "same"),
                                          (((1, 1),), "qd")])
def test_propagate_matches_numpy(gpu, grid, blocks, want):
    rng = np.random.default_rng(sum(grid) + len(blocks))
    M, sh = int(np.prod(grid)), grid[::-1]
    W = (rng.normal(size=(3, M)) + 1j * rng.normal(size=(3, M))) * 0.2
    g = np.exp(-rng.random(M)) + 0.1j * rng.normal(size=M)  # no product of axis factors, no symmetry
    W, g = W.astype(np.complex64).astype(complex), g.astype(np.complex64).astype(complex)
    seq = [s for n, s in blocks for _ in range(n)]
    got = chains(gpu, W, g, blocks, grid, want)
    for c, order in enumerate((seq, seq[::-1])):
        if want != "same" and "qd"[c] not in want or want == "same" and c == 0:
            continue
        ref = [np.exp(-W[order[0]])]
        for s in order[1:]:
            ref.append(np.exp(-W[s]) * np.fft.ifftn(g.reshape(sh) * np.fft.fftn(ref[-1].reshape(sh))).reshape(-1))
        e = rel(got[c], np.array(ref))
        say("propagate", grid, blocks, want, c, "%.2e" % e)
        assert e < 3e-6


@pytest.mark.parametrize("grid", [(20, 20, 2), (12, 12, 8), (16, 20, 24), (6, 96, 10)])
def test_chains_an_odd_number_of_floats_apart(gpu, grid):
    """The arrays are floats to the caller: a complementary chain that starts at any float of an allocation gives the
    bits it gives at an aligned address, on grids of either form."""
    rng = np.random.default_rng(sum(grid))
    M, n = int(np.prod(grid)), 5
    W = ((rng.normal(size=(2, M)) + 1j * rng.normal(size=(2, M))) * 0.2).astype(np.complex64)
    g = np.exp(-rng.random(M)).astype(np.complex64)
    want = chains(gpu, W, g, ((2, 0), (3, 1)), grid, "qd")
    mol = gpu.FtsMoleculeC()
    mol.nblocks = 2
    mol.N[0], mol.species[0], mol.N[1], mol.species[1] = 2, 0, 3, 1
    Wb, gb = gpu.DeviceBuffer.from_array(W), gpu.DeviceBuffer.from_array(g)
    q, qd = gpu.DeviceBuffer(8 * M * n), gpu.DeviceBuffer(8 * M * n + 4)
    gpu.check(gpu.lib().mft_fts_propagate(q.ptr, ctypes.c_void_p(qd.ptr.value + 4), Wb.ptr, gb.ptr, ctypes.byref(mol),
                                          (ctypes.c_int * 3)(*grid), None))
    assert np.array_equal(q.to_array(np.complex64, (n, M)), want[0])
    assert np.array_equal(qd.to_array(np.float32, 2 * M * n + 1)[1:].view(np.complex64).reshape(n, M), want[1])
