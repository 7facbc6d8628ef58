"""The logits gradient over rows that start at any offset (V not a multiple of a vector):
the flat pieces give the bits of the row-per-workgroup kernel (GPU)."""

import pytest
import torch

from rl_amd import _C

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("dtype,V", [(torch.bfloat16, 2047), (torch.bfloat16, 2049), (torch.bfloat16, 6151),
                                     (torch.bfloat16, 100003), (torch.float16, 2051), (torch.float32, 1023),
                                     (torch.float32, 1025), (torch.float32, 4098)])
@pytest.mark.parametrize("B,S,R", [(1, 1, 1), (3, 7, 6), (2, 40, 40), (2, 5, 0)])
def test_flat_pieces_equal_rows(dtype, V, B, S, R):
    g = torch.Generator().manual_seed(V + S)
    x = (torch.randn(B, S, V, generator=g) * 2).to(dtype).to(DEV)
    target = torch.randint(0, V, (B, max(R, 1)), generator=g)[:, :R]
    if R > 3:
        target[0, :4] = torch.tensor([0, V - 1, V, V // 2])  # a row's ends, and one outside
    up = torch.randn(B, R, generator=g) * (torch.rand(B, R, generator=g) < 0.6)
    target, up = target.to(DEV), up.to(DEV)
    stats = torch.empty((B, R, 2), device=DEV)
    _C.logprob_fwd(x, target, 0, V, torch.empty((B, R), device=DEV), stats)
    wide = torch.empty((B, S, V + 5), dtype=dtype, device=DEV)  # rows of another stride: row kernels
    wide[..., :V] = x
    want = torch.empty_like(wide)[..., :V]
    _C.logprob_bwd(wide[..., :V], target, 0, V, stats, up, want)
    got = torch.full_like(x, 9.0)
    _C.logprob_bwd(x, target, 0, V, stats, up, got)
    bits = {2: torch.int16, 4: torch.int32}[x.element_size()]
    nonzero = want != 0  # a zero may carry either sign
    assert torch.equal(got[nonzero].view(bits), want[nonzero].view(bits)) and not got[~nonzero].any()
    # starting 16 bytes into a 4 KB page, and in place
    store = torch.empty(x.numel() + 64, dtype=dtype, device=DEV)
    own = store[16 // x.element_size():][: x.numel()].view(B, S, V)
    own.copy_(x)
    _C.logprob_bwd(own, target, 0, V, stats, up, own)
    assert torch.equal(own, got)


@pytest.mark.parametrize("dtype,V", [(torch.bfloat16, 2049), (torch.float16, 6151), (torch.float32, 1027)])
@pytest.mark.parametrize("B,S,R", [(1, 3, 1), (1, 4, 3), (2, 5, 3)])
def test_logits_end_with_the_last_row(dtype, V, B, S, R):
    """Logits that end with row R - 1 of the last sample under a gradient of S > R rows: the
    vector that holds their end also holds elements of a row without logits."""
    g = torch.Generator().manual_seed(V + S)
    flat = (torch.randn((B - 1) * S * V + R * V, generator=g) * 2).to(dtype).to(DEV)
    x = flat.as_strided((B, R, V), (S * V, V, 1))
    target = torch.randint(0, V, (B, R), generator=g).to(DEV)
    target[-1, -1] = V - 1
    up = torch.randn(B, R, generator=g).to(DEV)
    stats = torch.empty((B, R, 2), device=DEV)
    _C.logprob_fwd(x, target, 0, V, torch.empty((B, R), device=DEV), stats)
    want = torch.empty((B, S, V + 5), dtype=dtype, device=DEV)[..., :V]  # rows of another stride: row kernels
    _C.logprob_bwd(x, target, 0, V, stats, up, want)
    got = torch.full((B, S, V), 9.0, dtype=dtype, device=DEV)
    _C.logprob_bwd(x, target, 0, V, stats, up, got)
    assert torch.equal(got, want)
    assert not got[:, R:].any()
