"""The fp32 product formed from bf16 planes (mirl_gemm_f32_abt) against float64: partial tiles,
the shortest reductions, spreads of magnitude, and the values that do not split (GPU)."""

import pytest
import torch

from rl_amd import _C

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _check(a, b):
    """Summing K products in fp32 errs by at most K 2^-24 of the sum of their magnitudes; the
    planes left out of a product are below 3 * 2^-25 of it."""
    M, K = a.shape
    out = torch.full((M, b.shape[0]), 7.0, device=DEV)
    _C.gemm_f32_abt(a.to(DEV), b.to(DEV), K, out)
    out = out.cpu().double()
    want = a.double() @ b.double().t()
    fine = torch.isfinite(want)
    assert torch.equal(torch.isnan(out), torch.isnan(want))
    assert torch.equal(out[torch.isinf(want)], want[torch.isinf(want)])
    size = a.abs().double().nan_to_num(0, 0, 0) @ b.abs().double().nan_to_num(0, 0, 0).t()
    bad = (out - want).abs()[fine] > ((K + 2) * 2.0**-24 * size)[fine]
    assert not bad.any(), int(bad.sum())
    # Root mean square over the outputs of random operands: 3 K / 8 roundings (six products of planes per 16 elements),
    # each uniform within half an ulp of a partial sum of half the final square on average, give
    # sqrt(K) / 4 times 2^-24 of the root of the sum of squared products; twice that and one
    # rounding are allowed.  Without the third planes it would be 2^-18 at any K.
    norm = (a.double().nan_to_num(0, 0, 0).square() @ b.double().nan_to_num(0, 0, 0).square().t()).sqrt()
    fine &= norm > 0
    if fine.any():
        rms = ((out - want)[fine] / norm[fine]).square().mean().sqrt().item()
        assert rms <= (K / 4 + 1) ** 0.5 * 2.0**-24, rms
    return out


@pytest.mark.parametrize("M,N,K", [(1, 1, 64), (255, 257, 64), (256, 256, 128), (513, 31, 192), (3, 300, 1024)])
def test_shapes(M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    _check(torch.randn(M, K, generator=g), torch.randn(N, K, generator=g) * 0.02)


@pytest.mark.parametrize("spread", [4.0, 12.0])
def test_magnitudes_far_apart(spread):
    g = torch.Generator().manual_seed(3)
    a = torch.randn(257, 256, generator=g) * torch.exp(spread * torch.randn(257, 256, generator=g))
    _check(a, torch.randn(64, 256, generator=g))


@pytest.mark.parametrize("scale", [1e-38, 1e-36, 2.0**-109, 1e-30, 1e18])
def test_small_and_large_values(scale):
    """Below 2^-109 the third plane of an unscaled value would lose bits."""
    g = torch.Generator().manual_seed(5)
    a = torch.randn(300, 128, generator=g) * scale
    b = torch.randn(260, 128, generator=g) * (1e20 if scale < 1 else 1.0)
    a[:, ::7] = 0.0
    _check(a, b)
    a[5, 3] = 1.5 * 2.0**-110  # one such value among ordinary ones
    _check(a, torch.randn(260, 128, generator=g))


def test_values_that_do_not_split():
    g = torch.Generator().manual_seed(7)
    a, b = torch.randn(600, 64, generator=g), torch.randn(520, 64, generator=g)
    _check(a, b)
    a[3, 5], a[4, 6], a[300, 0] = float("inf"), float("-inf"), float("nan")
    b[7, 9], b[8, 1] = float("-inf"), 0.0
    a[290] = 0.0
    a[290, 1] = torch.finfo(torch.float32).max  # rounds to infinity as a bf16
    b[:, 1] = b[:, 1].clamp(-0.5, 0.5)
    _check(a, b)


@pytest.mark.parametrize("a,b", [(2.0**-140, 2.0**100), (1.25 * 2.0**-134, 3.0 * 2.0**90), (1.7 * 2.0**-126, 5.0),
                                 (1e32, 1e-10), (1e25, 1e9)])
def test_ends_of_the_range(a, b):
    """Subnormal values against large ones, and values and sums that the first operand's scale
    takes past the largest fp32: every product is there, whichever operand holds which."""
    g = torch.Generator().manual_seed(11)
    A, B = torch.randn(257, 64, generator=g) * a, torch.randn(260, 64, generator=g) * b
    A[:, ::5] = 0.0
    _check(A, B)
    _check(B, A)


@pytest.mark.parametrize("value", [1.5 * 2.0**-110, 1e-35, 1e-41])
def test_small_value_leaves_other_rows_alone(value):
    """One value below 2^-109 among ordinary ones of the first operand (the logits gradient of
    dH and dW) changes no bit of another row: its tile takes the arithmetic it takes without it."""
    g = torch.Generator().manual_seed(9)
    a, b = torch.randn(256, 128, generator=g), torch.randn(256, 128, generator=g)
    a[5, 3] = 0.0
    out = [torch.empty(256, 256, device=DEV) for _ in range(2)]
    _C.gemm_f32_abt(a.to(DEV), b.to(DEV), 128, out[0])
    a[5, 3] = value
    _C.gemm_f32_abt(a.to(DEV), b.to(DEV), 128, out[1])
    others = torch.arange(256, device=DEV) != 5
    assert torch.equal(out[0][others], out[1][others])
