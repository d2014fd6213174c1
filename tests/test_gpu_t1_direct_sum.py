"""Small complex64 type-1 transforms as direct sums on the matrix cores (NFFT2_2D_GPU, and the
setpts_type1 of a batch of equal sizes) against FP64 direct sums.

Tolerance: every operand is a pair of FP16 values (2^-22 relative), phases are exact to
(2j + 1) 2^-33 turns (below 1e-7 rad at N = 256) with phasors of a few FP32 roundings, and the FP32
sums round three times per 16 points: below 5e-7 rel-L2 at every size here, so 1e-6.
"""
import numpy as np
import pytest
import torch

import miscellaneous_amd as m
import oracle

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def cn01(rng, shape):
    return ((rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) / np.sqrt(2)).astype(np.complex64)


# the smallest; one pair more or less than a tile of 8 or 16; chunk edges (32 / 34, 96 / 98, 128 / 130);
# points at the edges of a 64-point stage and of 12 ranges; a long, narrow pair; the largest of the rule
@pytest.mark.parametrize("N1,N2,M", [(2, 2, 1), (2, 256, 63), (16, 18, 64), (34, 32, 65), (22, 46, 300), (88, 88, 1936),
                                     (96, 98, 767), (98, 96, 769), (126, 128, 2500), (130, 126, 700), (256, 22, 6144),
                                     (256, 254, 6000), (64, 256, 6145)])
def test_dropin_direct_sum(N1, N2, M):
    rng = np.random.default_rng(N1 + 1000 * N2 + M)
    x1 = (rng.uniform(-1.5 * N1, 1.5 * N1, M)).astype(np.float32)       # beyond one period: periodic
    x2 = (rng.uniform(-1.5 * N2, 1.5 * N2, M)).astype(np.float32)
    d = cn01(rng, M) * np.float32(1e-20 if M == 300 else 1.0)             # the block's scale
    out = torch.empty(N1 * N2, dtype=torch.complex64, device=DEV)
    m.NFFT2_2D_GPU(out, T(d), T(x1), T(x2), N1, N2, M)
    torch.cuda.synchronize()
    ref = oracle.ndft_type1(d.astype(np.complex128), x1, x2, N1, N2)
    e = oracle.rel_l2(out.cpu().numpy().reshape(N1, N2), ref)
    print(f"direct sum {N1}x{N2} M={M}: rel-L2 {e:.2e}", flush=True)
    assert e < 1e-6


def test_dropin_result_over_data():
    """The result array may overlap the samples: it is written after they were read."""
    rng = np.random.default_rng(5)
    N, M = 40, 1600
    x1, x2, d = (rng.random(M) - 0.5) * N, (rng.random(M) - 0.5) * N, cn01(rng, M)
    buf = T(d)
    m.NFFT2_2D_GPU(buf, buf, T(x1.astype(np.float32)), T(x2.astype(np.float32)), N, N, M)
    torch.cuda.synchronize()
    ref = oracle.ndft_type1(d.astype(np.complex128), x1.astype(np.float32), x2.astype(np.float32), N, N)
    assert oracle.rel_l2(buf.cpu().numpy().reshape(N, N), ref) < 1e-6


@pytest.mark.parametrize("bad", ["nan", "inf", "far"])
def test_dropin_direct_sum_not_finite(bad):
    """A sample or coordinate that is not finite, or a coordinate beyond 2^29, reaches every mode as NaN."""
    rng = np.random.default_rng(6)
    N, M = 44, 500
    x1, x2, d = (rng.random(M) - 0.5) * N, (rng.random(M) - 0.5) * N, cn01(rng, M)
    if bad == "nan":
        d[17] = np.nan
    else:
        x1[17] = np.inf if bad == "inf" else 2.0 ** 30
    out = torch.zeros(N * N, dtype=torch.complex64, device=DEV)
    m.NFFT2_2D_GPU(out, T(d), T(x1.astype(np.float32)), T(x2.astype(np.float32)), N, N, M)
    assert torch.isnan(out.real).all() and torch.isnan(out.imag).all()


# whole transforms per block, point ranges with partial sums, chunks of modes, uneven M with an empty one
@pytest.mark.parametrize("N1,N2,Ms", [(88, 88, [1936] * 40), (22, 22, [400] * 3), (126, 126, [2500, 0, 64, 65, 1] * 52),
                                      (64, 90, [1200] * 20), (130, 88, [1000, 2000])])
def test_batch_direct_sum(N1, N2, Ms):
    """setpts_type1 by the direct sums; type1 and type2 after it find the points sorted."""
    rng = np.random.default_rng(N1 + len(Ms))
    xs = [T(((rng.random(k) - 0.5) * N1).astype(np.float32)) for k in Ms]
    ys = [T(((rng.random(k) - 0.5) * N2).astype(np.float32)) for k in Ms]
    ds = [T(cn01(rng, k)) for k in Ms]
    outs = [torch.full((N1 * N2,), np.nan, dtype=torch.complex64, device=DEV) for _ in Ms]
    fs = [T(cn01(rng, (N1, N2))) for _ in Ms]
    t2 = [torch.empty(k, dtype=torch.complex64, device=DEV) for k in Ms]
    b = m.Batch([(N1, N2, k) for k in Ms], device=DEV).set_io_type1(ds, outs).set_points(xs, ys).set_io(fs, t2)
    b.setpts_type1()
    got = [o.cpu().numpy() for o in outs]
    b.type1()
    b.type2()
    torch.cuda.synchronize()
    for t in sorted({0, 1, len(Ms) // 2, len(Ms) - 1, *range(min(5, len(Ms)))}):
        if Ms[t] == 0:
            assert np.all(got[t] == 0)
            continue
        x1, x2 = xs[t].cpu().numpy(), ys[t].cpu().numpy()
        ref = oracle.ndft_type1(ds[t].cpu().numpy().astype(np.complex128), x1, x2, N1, N2)
        e = oracle.rel_l2(got[t].reshape(N1, N2), ref)
        print(f"batch direct sum {N1}x{N2} x{len(Ms)} transform {t} M={Ms[t]}: rel-L2 {e:.2e}", flush=True)
        assert e < 1e-6
        assert oracle.rel_l2(outs[t].cpu().numpy(), got[t]) < 2e-6
        r2 = oracle.ndft_type2(fs[t].cpu().numpy().astype(np.complex128), x1[:64], x2[:64])
        assert oracle.rel_l2(t2[t].cpu().numpy()[:64], r2) < 1e-5


# scaled in the sums' epilogue, in the addition of the partial sums, and after the passes of larger transforms
@pytest.mark.parametrize("P,N1,N2,M", [(250, 88, 88, 60), (3, 40, 54, 900), (2, 64, 300, 700)])
def test_batch_scaled(P, N1, N2, M):
    """setpts_type1(scale) is the unscaled result times the factors, bit for bit where the sums are direct."""
    g = torch.Generator(device=DEV).manual_seed(9)
    xs = [(torch.rand(M, generator=g, device=DEV) - 0.5) * N1 for _ in range(P)]
    ys = [(torch.rand(M, generator=g, device=DEV) - 0.5) * N2 for _ in range(P)]
    ds = [torch.randn(M, generator=g, dtype=torch.complex64, device=DEV) for _ in range(P)]
    outs = [torch.zeros(N1 * N2, dtype=torch.complex64, device=DEV) for _ in range(P)]
    b = m.Batch([(N1, N2, M)] * P, device=DEV).set_points(xs, ys).set_io_type1(ds, outs)
    scale = torch.rand(N1 * N2, generator=g, device=DEV) + 0.5
    b.setpts_type1()
    ref = torch.stack(outs) * scale
    b.setpts_type1(scale=scale)
    got = torch.stack(outs)
    if max(N1, N2) <= 256:
        assert torch.equal(got, ref)
    assert (got - ref).abs().max().item() < 1e-5 * ref.abs().max().item()
    with pytest.raises(ValueError):
        b.setpts_type1(scale=scale[1:])
