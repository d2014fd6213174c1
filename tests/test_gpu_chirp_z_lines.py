"""Chirp-z passes where the lines do not fill their blocks: several lines share a block in the strided passes and in a
batch (m = 512: 8 or 4 lines, 1,024: 4 or 2), at the smallest and largest N of each FFT length.  Type-2 and adjoint
against float64 direct sums (complex64 1e-5, complex128 1e-9, as the other transform tests); a batch's type-2 has its
plan's bits."""
import numpy as np
import pytest
import torch

import miscellaneous_amd as m
import oracle

pytestmark = pytest.mark.gpu
SIZES = [(130, 134), (170, 132), (172, 342), (342, 170), (344, 22), (30, 682), (684, 22)]


def inputs(N1, N2, M, real):
    rng = np.random.default_rng(N1 + 7 * N2)
    x, y = ((rng.random(M) - 0.5) * N1).astype(real), ((rng.random(M) - 0.5) * N2).astype(real)
    cn = lambda *s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)
    return x, y, cn(N1, N2), cn(M)


@pytest.mark.parametrize("dtype", [torch.complex64, torch.complex128])
@pytest.mark.parametrize("N1,N2", SIZES)
def test_plan_lines(N1, N2, dtype):
    real, tol = (np.float32, 1e-5) if dtype == torch.complex64 else (np.float64, 1e-9)
    x, y, f, d = inputs(N1, N2, 300, real)
    t = lambda a: torch.from_numpy(a).cuda()
    plan = m.Plan(N1, N2, dtype)
    out = plan.setpts_type2(t(x), t(y), t(f).to(dtype)).cpu().numpy()
    assert oracle.rel_l2(out, oracle.ndft_type2(f.astype(np.complex128), x, y)) < tol
    F = plan.adjoint(t(d).to(dtype)).cpu().numpy()
    ref = np.conj(oracle.ndft_type1(np.conj(d).astype(np.complex128), x, y, N1, N2))
    assert oracle.rel_l2(F, ref) < tol


def test_batch_lines():
    ins = [inputs(a, b, 300, np.float32) for a, b in SIZES]
    t = lambda a: torch.from_numpy(a).cuda()
    xs, ys, fs, ds = ([t(i[k]) for i in ins] for k in range(4))
    out2 = [torch.empty(300, dtype=torch.complex64, device="cuda") for _ in SIZES]
    out1 = [torch.empty(a, b, dtype=torch.complex64, device="cuda") for a, b in SIZES]
    b = m.Batch([(a, c, 300) for a, c in SIZES]).set_points(xs, ys)
    b.set_io(fs, out2)
    b.setpts_type2()
    b.set_io_type1(ds, out1)
    b.type1()
    for k, (N1, N2) in enumerate(SIZES):
        if max(N1, N2) <= 682:   # longer lines take a batch's direct passes: equal to rounding only
            assert torch.equal(out2[k], m.Plan(N1, N2).setpts_type2(xs[k], ys[k], fs[k])), (N1, N2)
        x, y, f, d = ins[k]
        assert oracle.rel_l2(out2[k].cpu().numpy(), oracle.ndft_type2(f.astype(np.complex128), x, y)) < 1e-5
        ref = oracle.ndft_type1(d.astype(np.complex128), x, y, N1, N2)
        assert oracle.rel_l2(out1[k].cpu().numpy(), ref) < 1e-5, (N1, N2)
