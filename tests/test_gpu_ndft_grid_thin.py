"""NDFT2_2D_GPU on thin grids: one 16-pair row or column of a tile in use (its products on four waves), one more (two
rows), edge tiles of both kinds, and so many tiles that the point ranges are merged.  Against a float64 direct sum; the
phases stay below 100 turns, so a term's error is below 2 pi * 100 * 2^-52 = 1.4e-13: tolerance 1e-12."""
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


@pytest.mark.parametrize("nu,nv,vmajor,M", [(1, 500, False, 700), (500, 1, True, 700), (32, 33, False, 33), (31, 100, True, 700),
                                            (34, 100, False, 700), (200, 31, False, 700), (160, 150, True, 40),
                                            (1, 4096, False, 700), (4096, 2, False, 1), (3000, 31, True, 260),
                                            (150, 220, False, 5000)])
def test_grid_thin(nu, nv, vmajor, M):
    rng = np.random.default_rng(nu * 1000 + nv + M)
    X, Y = rng.random(M) - 0.5, rng.random(M) - 0.5
    d = rng.standard_normal(M) + 1j * rng.standard_normal(M)
    a, b = 0.0625 * (np.arange(nu) - nu // 3), -0.03125 * (np.arange(nv) - nv // 2)
    u, v = (np.tile(a, nv), np.repeat(b, nu)) if vmajor else (np.repeat(a, nv), np.tile(b, nu))
    out = call(X, Y, u, v, d, 1, 1)
    ok, gu, gv, vm = m.ndft_grid_info()
    assert ok and gu * gv == nu * nv
    A, B = np.exp(-2j * np.pi * np.outer(a, X)), np.exp(-2j * np.pi * np.outer(b, Y))
    ref = (A * d) @ B.T
    ref = ref.T.reshape(-1) if vmajor else ref.reshape(-1)
    assert np.linalg.norm(out - ref) <= 1e-12 * np.linalg.norm(ref)
