"""NdftPlan (fp32, bf16x3): modes whose pair sums exceed the FP32 range while the results are inside it.

Four conjugate modes of 1e38 sum to 4e38 > FLT_MAX (3.4e38); at the points used here every result is below
3e38.  Tolerances: the operand roundings, as in tests/test_gpu_ndft.py."""
import numpy as np
import pytest
import torch

import miscellaneous_amd as m
import oracle

pytestmark = pytest.mark.gpu
TOL = {"fp32": 2e-6, "bf16x3": 2e-5}


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("mag", [1e38, 1.6e38])
def test_pair_sums_beyond_the_range(prec, mag):
    rng = np.random.default_rng(17)
    N1, N2, M = 16, 18, 1500
    f = np.zeros((N1, N2), np.complex64)
    for a, b in ((10, 12), (10, 5), (5, 12), (5, 5)):       # k = (2, 3), (2, -4), (-3, 3), (-3, -4)
        f[a, b] = mag * np.exp(2j * np.pi * 0.02 * rng.random())
    x1 = ((rng.random(M) - 0.5) * N1).astype(np.float32)
    x2 = ((rng.random(M) - 0.5) * N2).astype(np.float32)
    ref = oracle.ndft_type2(f.astype(np.complex128) * 1e-38, x1, x2)
    fits = np.abs(ref) < 3.0
    assert fits.sum() > 500
    dev = torch.device("cuda:0")
    y = m.NdftPlan(N1, N2, prec, device=dev).type2(*(torch.from_numpy(a).to(dev) for a in (f, x1, x2))).cpu().numpy()
    got = y[fits].astype(np.complex128) * 1e-38
    assert np.isfinite(got).all(), int((~np.isfinite(got)).sum())
    err = oracle.rel_l2(got, ref[fits])
    print(f"ndft pairs {prec} modes of {mag:g}: rel-L2 {err:.3e} over {fits.sum()} results")
    assert err <= TOL[prec], err
