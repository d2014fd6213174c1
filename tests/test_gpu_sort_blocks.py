"""setpts at the edge of its two-launch form in histogram blocks: 64 blocks of 2,048 points in two launches, 65 in
three, on grids with few bins (the blocks' rows alone would fit).  Type-2 on sampled points against float64 direct
sums and the adjoint identity, FP32 1e-5 and FP64 1e-9 (the bounds of the other transform tests)."""
import numpy as np
import pytest
import torch

import miscellaneous_amd as m
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.complex64, torch.complex128])
@pytest.mark.parametrize("N1,N2,M", [(64, 64, 131072), (64, 64, 131073), (16, 24, 131073), (64, 64, 600000)])
def test_sort_blocks(N1, N2, M, dtype):
    rng = np.random.default_rng(M + N1)
    real, tol = (np.float32, 1e-5) if dtype == torch.complex64 else (np.float64, 1e-9)
    u = rng.random((2, M)) - 0.5
    u[:, M // 2:] *= 0.1
    x, y = (u[0] * N1).astype(real), (u[1] * N2).astype(real)
    cn = lambda *s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)
    f, d = cn(N1, N2), cn(M)
    t = lambda a: torch.from_numpy(a).cuda()
    plan = m.Plan(N1, N2, dtype)
    full = plan.setpts_type2(t(x), t(y), t(f).to(dtype)).cpu().numpy().astype(np.complex128)
    s = np.unique(rng.integers(0, M, 200))
    assert oracle.rel_l2(full[s], oracle.ndft_type2(f.astype(np.complex128), x[s], y[s])) < tol
    F = plan.adjoint(t(d).to(dtype)).cpu().numpy().astype(np.complex128)
    a, b = np.vdot(d, full), np.vdot(F, f)
    assert abs(a - b) <= tol * np.linalg.norm(d) * np.linalg.norm(full)
