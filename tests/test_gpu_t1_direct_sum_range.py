"""Direct type-1 sums over the magnitudes of FP32: samples of 1e-37 (some of them denormal) to 1e35.

Tolerance: the sums work on samples scaled by a power of two, which is exact at every magnitude, so the
relative error is that of samples of order 1 (below 5e-7 rel-L2); the results here are normal numbers
(10 times the samples and more), so their own rounding adds 6e-8: 1e-6."""
import numpy as np
import pytest
import torch

import miscellaneous_amd as m
import oracle

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def inputs(N, M, scale, seed):
    rng = np.random.default_rng(seed)
    x, y = (((rng.random(M) - 0.5) * N).astype(np.float32) for _ in range(2))
    d = (scale * (rng.standard_normal(M) + 1j * rng.standard_normal(M)) / np.sqrt(2)).astype(np.complex64)
    return x, y, d, oracle.ndft_type1(d.astype(np.complex128) / scale, x, y, N, N)


@pytest.mark.parametrize("scale", [1e-37, 1e-35, 1e-33, 1e-30, 1e35])
@pytest.mark.parametrize("N,M", [(16, 500), (88, 1936)])
def test_dropin_sample_range(N, M, scale):
    x, y, d, ref = inputs(N, M, scale, N)
    out = torch.empty(N * N, dtype=torch.complex64, device=DEV)
    m.NFFT2_2D_GPU(out, T(d), T(x), T(y), N, N, M)
    e = oracle.rel_l2(out.cpu().numpy().reshape(N, N).astype(np.complex128) / scale, ref)
    print(f"direct sum {N}x{N} M={M} samples {scale:g}: rel-L2 {e:.2e}", flush=True)
    assert e < 1e-6


@pytest.mark.parametrize("scale", [1e-37, 1e-33, 1e35])
def test_batch_sample_range(scale):
    """One transform per block (no partial sums): the scale of one transform is no other's."""
    N, M, P = 88, 400, 300
    x, y, d, ref = inputs(N, M, scale, 3)
    d1 = (d / np.float32(scale)).astype(np.complex64)
    outs = [torch.empty(N * N, dtype=torch.complex64, device=DEV) for _ in range(P)]
    b = m.Batch([(N, N, M)] * P, device=DEV).set_points([T(x)] * P, [T(y)] * P)
    b.set_io_type1([T(d1 if t % 2 else d) for t in range(P)], outs).setpts_type1()
    for t in (0, 1, P - 2, P - 1):
        got = outs[t].cpu().numpy().reshape(N, N).astype(np.complex128) / (1.0 if t % 2 else scale)
        e = oracle.rel_l2(got, ref)
        print(f"batch direct sum transform {t} samples {scale:g}: rel-L2 {e:.2e}", flush=True)
        assert e < 1e-6
