"""The direct type-1 sums are no further from FP64 sums than the passes they replace, at the longest FP32 chains that
their rule allows (few ranges of many points), on lengths of the matrix-core, chirp-z and FFT passes.  The passes' own
error differs by a few per cent between runs (the order in which a bin's points arrive): factor 1.05."""
import numpy as np
import pytest
import torch

import miscellaneous_amd as m
import oracle

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def inputs(N1, N2, M, seed):
    rng = np.random.default_rng(seed)
    x, y = ((rng.random(M) - 0.5) * N1).astype(np.float32), ((rng.random(M) - 0.5) * N2).astype(np.float32)
    d = ((rng.standard_normal(M) + 1j * rng.standard_normal(M)) / np.sqrt(2)).astype(np.complex64)
    ref = oracle.ndft_type1(d.astype(np.complex128), x, y, N1, N2)
    return [torch.from_numpy(a).to(DEV) for a in (x, y, d)], ref


def error(out, ref):
    return oracle.rel_l2(out.cpu().numpy().reshape(ref.shape), ref)


@pytest.mark.parametrize("P,N1,N2,M", [(250, 88, 88, 4096), (250, 22, 22, 1200), (120, 126, 126, 2500), (120, 64, 128, 1500),
                                       (40, 130, 88, 1500), (40, 250, 200, 1500)])
def test_batch_error_against_the_passes(P, N1, N2, M):
    (x, y, d), ref = inputs(N1, N2, M, P + N1)
    outs = [torch.empty(N1 * N2, dtype=torch.complex64, device=DEV) for _ in range(P)]
    b = m.Batch([(N1, N2, M)] * P, device=DEV).set_points([x] * P, [y] * P).set_io_type1([d] * P, outs)
    assert b.type1_ranges() > 0
    b.setpts_type1()
    sums = error(outs[P // 2], ref)
    b.type1()
    passes = error(outs[P // 2], ref)
    print(f"{N1}x{N2} x{P} M={M}: direct sums {sums:.2e}, passes {passes:.2e}", flush=True)
    assert sums <= 1.05 * passes


@pytest.mark.parametrize("N1,N2,M", [(88, 88, 1936), (22, 22, 6144), (126, 126, 6000), (256, 250, 6000), (128, 64, 6144)])
def test_dropin_error_against_the_passes(N1, N2, M):
    (x, y, d), ref = inputs(N1, N2, M, N1 + M)
    out = torch.empty(N1 * N2, dtype=torch.complex64, device=DEV)
    m.NFFT2_2D_GPU(out, d, x, y, N1, N2, M)
    sums, passes = error(out, ref), error(m.Plan(N1, N2, torch.complex64).setpts(x, y).type1(d), ref)
    print(f"{N1}x{N2} M={M}: direct sum {sums:.2e}, passes {passes:.2e}", flush=True)
    assert sums <= 1.05 * passes
