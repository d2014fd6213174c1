"""NDFT2_2D_GPU at the edges of its tiles: grids of odd and even lengths (an odd one's centre row is a pair of
its own), one past a 16-pair and a 64-pair tile, off-centre and with steps other than one, in both flattenings;
scattered outputs over the 512-output blocks; point counts around the 16-point chunk.  Against a float64 direct
sum; the phases reach ~100 turns, so a term's error is below 2 pi * 100 * 2^-52 = 1.4e-13: tolerance 1e-12."""
import numpy as np
import pytest
import torch

import miscellaneous_amd as m

pytestmark = pytest.mark.gpu


def call(X, Y, u, v, d, Nu, Nv):
    dev = torch.device("cuda:0")
    t = [torch.from_numpy(np.ascontiguousarray(a)).to(dev) for a in (X, Y, u, v, d)]
    out = torch.empty(u.size, dtype=torch.complex128, device=dev)
    m.NDFT2_2D_GPU(0, *t, out, Nu, Nv, X.size, u.size)
    return out.cpu().numpy()


def direct(X, Y, u, v, d, Nu, Nv):
    ph = np.outer(u, X) / Nu + np.outer(v, Y) / Nv
    return np.exp(-2j * np.pi * (ph - np.rint(ph))) @ d


@pytest.mark.parametrize("M", [1, 15, 17, 300])
@pytest.mark.parametrize("nu,nv,vmajor", [(1, 1, False), (2, 129, False), (127, 3, True), (33, 34, False), (130, 16, True)])
def test_grid_pairs(nu, nv, vmajor, M):
    rng = np.random.default_rng(nu * 1000 + nv + M)
    Nu, Nv = 88, 64
    X, Y = (rng.random(M) - 0.5) * Nu, (rng.random(M) - 0.5) * Nv
    d = rng.standard_normal(M) + 1j * rng.standard_normal(M)
    a, b = 3.0 - nu // 2 + 0.5 * np.arange(nu), -5.0 - 2.0 * np.arange(nv)
    u, v = (np.tile(a, nv), np.repeat(b, nu)) if vmajor else (np.repeat(a, nv), np.tile(b, nu))
    out, ref = call(X, Y, u, v, d, Nu, Nv), direct(X, Y, u, v, d, Nu, Nv)
    assert m.ndft_grid_info()[0]
    assert np.linalg.norm(out - ref) <= 1e-12 * np.linalg.norm(ref)


@pytest.mark.parametrize("N,M", [(2, 1), (511, 40), (513, 300), (2000, 17)])
def test_scattered_outputs(N, M):
    rng = np.random.default_rng(N + M)
    Nu, Nv = 60, 90
    X, Y = (rng.random(M) - 0.5) * Nu, (rng.random(M) - 0.5) * Nv
    d = rng.standard_normal(M) + 1j * rng.standard_normal(M)
    u, v = (rng.random(N) - 0.5) * Nu, (rng.random(N) - 0.5) * Nv
    u[0], v[-1] = u[0] + 0.25, v[-1] - 0.25
    out, ref = call(X, Y, u, v, d, Nu, Nv), direct(X, Y, u, v, d, Nu, Nv)
    assert np.linalg.norm(out - ref) <= 1e-12 * np.linalg.norm(ref)
