"""NdftPlan (fp32, bf16x3): modes near the denormals lose only what their own operand's spacing takes.

The smallest spacing q of an operand is 2^-149 (FP32) or, of BF16x3's low part, 2^-133.  A pair's operand entry,
the sum of four modes of magnitude a and random phase, has the rms sqrt(2) a; rounding it to q, and an FP32 sum
over it twice, gives an rms of sqrt(3) q / sqrt(12).  Tolerance: 1.5 times that over the entry's rms, beside what
the types give at ordinary magnitudes.  An operand scaled down by 4 has 4 times the first part."""
import math

import numpy as np
import pytest
import torch

import miscellaneous_amd as m
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec, mag, spacing, ordinary", [("fp32", 2.0**-130, 2.0**-149, 4e-7),
                                                          ("bf16x3", 2.0**-119, 2.0**-133, 2.0**-17)])
def test_small_modes(prec, mag, spacing, ordinary):
    rng = np.random.default_rng(18)
    N1, N2, M = 64, 64, 1500
    f = (mag * np.exp(2j * np.pi * rng.random((N1, N2)))).astype(np.complex64)
    x1 = ((rng.random(M) - 0.5) * N1).astype(np.float32)
    x2 = ((rng.random(M) - 0.5) * N2).astype(np.float32)
    ref = oracle.ndft_type2(f.astype(np.complex128) / mag, x1, x2)
    dev = torch.device("cuda:0")
    y = m.NdftPlan(N1, N2, prec, device=dev).type2(*(torch.from_numpy(a).to(dev) for a in (f, x1, x2))).cpu().numpy()
    err = oracle.rel_l2(y.astype(np.complex128) / mag, ref)
    tol = math.hypot(ordinary, 1.5 * math.sqrt(3 / 12) * spacing / (math.sqrt(2) * mag))
    print(f"ndft pairs {prec} modes of {mag:g}: rel-L2 {err:.3e} (tolerance {tol:.3e})")
    assert err <= tol, (err, tol)
