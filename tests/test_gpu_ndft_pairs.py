"""The conjugate-pair contraction of NdftPlan (fp32, bf16x3) at the edges of its tiles: one pair per
dimension, a last partial K-step (8 pairs) or column group (16 pairs), a second column chunk (64 pairs), and
points several periods out (the half steps change sign there).  Tolerances: the operand roundings, as in
tests/test_gpu_ndft.py."""
import numpy as np
import pytest
import torch

import miscellaneous_amd as m
import oracle

pytestmark = pytest.mark.gpu
TOL = {"fp32": 2e-6, "bf16x3": 2e-5}


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("N1,N2", [(2, 2), (2, 130), (130, 2), (34, 18), (258, 66)])
def test_pairs_vs_oracle(prec, N1, N2):
    rng = np.random.default_rng(31 * N1 + N2)
    M = 321
    f = ((rng.standard_normal((N1, N2)) + 1j * rng.standard_normal((N1, N2))) / np.sqrt(2)).astype(np.complex64)
    x1 = ((rng.random(M) - 0.5) * N1 + N1 * rng.integers(-3, 4, M)).astype(np.float32)
    x2 = ((rng.random(M) - 0.5) * N2 + N2 * rng.integers(-3, 4, M)).astype(np.float32)
    dev = torch.device("cuda:0")
    y = m.NdftPlan(N1, N2, prec, device=dev).type2(*(torch.from_numpy(a).to(dev) for a in (f, x1, x2))).cpu().numpy()
    err = oracle.rel_l2(y, oracle.ndft_type2(f.astype(np.complex128), x1, x2))
    print(f"ndft pairs {prec} {N1}x{N2}: rel-L2 {err:.3e}")
    assert err <= TOL[prec], err
