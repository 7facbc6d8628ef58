"""The divergences' logits gradient over rows that start at any offset (V not a multiple of
a vector): the flat pieces give the bits of the row-per-workgroup kernel (GPU)."""

import pytest
import torch

from rl_amd import _C

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("dtype,V", [(torch.bfloat16, 2047), (torch.bfloat16, 2049), (torch.bfloat16, 6151),
                                     (torch.bfloat16, 100003), (torch.float16, 2051), (torch.float32, 1023),
                                     (torch.float32, 1025), (torch.float32, 4098)])
@pytest.mark.parametrize("B,S", [(1, 1), (3, 7), (2, 40)])
@pytest.mark.parametrize("kind", ["reverse_kl", "cross_entropy", "entropy"])
def test_flat_pieces_equal_rows(kind, dtype, V, B, S):
    g = torch.Generator().manual_seed(V + S)
    x, t = ((torch.randn(B, S, V, generator=g) * 2).to(dtype).to(DEV) for _ in range(2))
    if kind == "entropy":
        t = None
    up = (torch.randn(B, S, generator=g) * (torch.rand(B, S, generator=g) < 0.6)).to(DEV)
    out, stats = torch.empty((B, S), device=DEV), torch.empty((B, S, 4), device=DEV)
    _C.divergence_fwd(kind, x, t, out, stats)
    wide = torch.empty((B, S, V + 5), dtype=dtype, device=DEV)  # rows of another stride: the row kernel
    want = torch.empty_like(wide)[..., :V]
    _C.divergence_bwd(kind, x, t, out, stats, up, want)
    got = torch.full_like(x, 9.0)
    _C.divergence_bwd(kind, x, t, out, stats, up, got)
    bits = {2: torch.int16, 4: torch.int32}[x.element_size()]
    nonzero = want != 0  # a zero may carry either sign
    assert torch.equal(got[nonzero].view(bits), want[nonzero].view(bits)) and not got[~nonzero].any()
    # starting 16 bytes into a 4 KB page, and in place
    store = torch.empty(x.numel() + 64, dtype=dtype, device=DEV)
    own = store[16 // x.element_size():][: x.numel()].view(B, S, V)
    own.copy_(x)
    _C.divergence_bwd(kind, own, t, out, stats, up, own)
    assert torch.equal(own, got)
