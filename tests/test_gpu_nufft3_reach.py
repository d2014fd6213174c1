"""Type-3 NUFFT where its kernels change form: taps masked (eps >= 1e-3: the tails past msp still count), all msp taps
without a mask (1e-4), fewer taps than msp (from 1e-5 on); one output, outputs along one line, two inputs, input
counts around a batch of 32 and a chunk of 64.  Against the oracle's restatement, which sums exactly msp taps: the
two differ by FP64 rounding and by tails under 2^-54 of a tap, amplified at most ~1e3 by the compensation, so the
bound of the other type-3 tests, rel-L2 1e-11, holds."""
import numpy as np
import pytest
import torch

import miscellaneous_amd as m
import oracle

pytestmark = pytest.mark.gpu


def check(x, y, s, t, f, eps):
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    F = m.NUFFT_2D(T(x), T(y), T(s), T(t), T(f), eps).cpu().numpy()
    R, _ = oracle.nufft3_2d(x, y, s, t, f, eps)
    assert oracle.rel_l2(F, R) < 1e-11


def points(seed, n_in, n_out, sx=5.0, sy=5.0):
    rng = np.random.default_rng(seed)
    f = rng.standard_normal(n_in) + 1j * rng.standard_normal(n_in)
    x, y = rng.uniform(-4, 4, n_in), rng.uniform(-3, 3, n_in)
    return x, y, rng.uniform(-sx, sx, n_out), rng.uniform(-sy, sy, n_out), f


@pytest.mark.parametrize("eps", [0.5, 1e-2, 1e-3, 1e-4, 1e-5, 1e-9, 1e-13])
def test_tap_forms(eps):
    check(*points(3, 500, 400), eps)


@pytest.mark.parametrize("n_in,n_out", [(2, 1), (31, 17), (32, 16), (33, 15), (64, 1), (129, 300)])
def test_counts(n_in, n_out):
    check(*points(n_in, n_in, n_out), 1e-6)


def test_outputs_along_a_line():
    check(*points(9, 300, 200, 9.0, 0.0), 1e-6)
