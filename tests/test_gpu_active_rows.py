"""The rows of the hidden-state backward with a non-zero upstream gradient, moved to the front,
against torch on the CPU (GPU)."""

import pytest
import torch

from rl_amd import _C

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("S,B,H,pad", [(1, 1, 8, 0), (63, 1, 5, 0), (1023, 1, 16, 0), (512, 2, 24, 8), (205, 5, 7, 1),
                                       (8192, 1, 8, 0), (2731, 3, 4, 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("share", [0.0, 0.3, 1.0])
def test_active_rows(S, B, H, pad, dtype, share):
    g = torch.Generator().manual_seed(S + B)
    up = torch.randn(B, S + 1, generator=g) * (torch.rand(B, S + 1, generator=g) < share)
    up = up[:, 1:]  # strided
    if share > 0:
        up[0, 0], up[-1, -1] = float("nan"), -0.0
    target = torch.randint(-5, 1000, (B, S), generator=g)
    T = S * B
    stats = torch.randn(T, 2, generator=g)
    wide = torch.randn(T, H + pad, generator=g).to(dtype)
    hidden = wide.to(DEV)[:, :H]
    perm, count, h, tgt, st, ga = (x.cpu() for x in _C.lce_active_rows(up.to(DEV), target.to(DEV), stats.to(DEV),
                                                                       hidden))
    rows = up.t().reshape(T)
    active = (rows != 0).nonzero()[:, 0]
    n = int(count)
    assert n == active.numel()
    assert torch.equal(perm[:n], active) and torch.equal(perm.sort().values, torch.arange(T))
    assert torch.equal(h[:n], wide[:, :H][active])
    assert torch.equal(tgt[0], target.t().reshape(T)[perm]) and torch.equal(st, stats[perm])
    torch.testing.assert_close(ga[0], rows[perm], rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("T", [(1 << 20) + 5, (1 << 24) + 5])
def test_more_rows_than_a_launch_holds_workgroups_for(T):
    """2^24 rows of 256 threads each would be 2^32 threads, more than a launch takes."""
    g = torch.Generator(device=DEV).manual_seed(T)
    up = torch.randn(1, T, generator=g, device=DEV) * (torch.rand(1, T, generator=g, device=DEV) < 0.5)
    target = torch.randint(0, 1000, (1, T), generator=g, device=DEV)
    stats = torch.randn(T, 2, generator=g, device=DEV)
    hidden = torch.randn(T, 8, generator=g, device=DEV).to(torch.bfloat16)
    perm, count, h, tgt, st, ga = _C.lce_active_rows(up, target, stats, hidden)
    active = (up[0] != 0).nonzero()[:, 0]
    n = int(count)
    assert n == active.numel()
    assert torch.equal(perm[:n], active)
    assert torch.equal(perm[n:], (up[0] == 0).nonzero()[:, 0].flip(0))
    assert torch.equal(h[:n], hidden[active])
    assert torch.equal(tgt[0], target[0][perm]) and torch.equal(st, stats[perm]) and torch.equal(ga[0], up[0][perm])
