"""Chirp-z passes of long lines (FFTs of 4,096, 8,192 and 16,384 points; at 16,384 a thread holds two parts of a
line): the smallest and largest N of each length, along contiguous rows and along strided columns.  Type-2 and adjoint
against float64 direct sums (complex64 1e-5, complex128 1e-9, as the other transform tests)."""
import numpy as np
import pytest
import torch

import miscellaneous_amd as m
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,N", [(torch.complex64, n) for n in (1364, 1366, 2730, 2732, 4094)] +
                         [(torch.complex128, n) for n in (1364, 1366, 2046)])
@pytest.mark.parametrize("cols", [True, False])
def test_long_lines(dtype, N, cols):
    real, tol = (np.float32, 1e-5) if dtype == torch.complex64 else (np.float64, 1e-9)
    N1, N2 = (N, 24) if cols else (24, N)
    M = 257
    rng = np.random.default_rng(N + cols)
    x, y = ((rng.random(M) - 0.5) * N1).astype(real), ((rng.random(M) - 0.5) * N2).astype(real)
    cn = lambda *s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)
    f, d = cn(N1, N2), cn(M)
    t = lambda a: torch.from_numpy(a).cuda()
    plan = m.Plan(N1, N2, dtype)
    out = plan.setpts_type2(t(x), t(y), t(f).to(dtype)).cpu().numpy()
    e2 = oracle.rel_l2(out, oracle.ndft_type2(f.astype(np.complex128), x, y))
    F = plan.adjoint(t(d).to(dtype)).cpu().numpy()
    e1 = oracle.rel_l2(F, np.conj(oracle.ndft_type1(np.conj(d).astype(np.complex128), x, y, N1, N2)))
    print(f"chirp-z {dtype} {N1}x{N2}: type-2 {e2:.2e}, adjoint {e1:.2e}", flush=True)
    assert e2 < tol and e1 < tol
