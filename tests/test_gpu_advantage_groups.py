"""Grouping of prompt rows for the GRPO advantages: hashed rows, rows compared directly and
scalar ids give the same bits, at the edges of a wave, a scan step and a workgroup (GPU)."""

import pytest
import torch

from oracle.advantage import baseline_and_std_per_prompt
from rl_amd import _C

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
STEP = 0x9E3779B97F4A7C15 - (1 << 64)  # the hash adds (k + 1) * STEP to element k, as int64


def _rows(groups, K, g):
    """[groups, K] keys that agree in their first element; group 1 differs from group 0 in
    the last one only, and groups 2 and 3 are different rows of one hash: element 0 and 1 of
    the one are elements 1 and 0 of the other, moved by what their positions add."""
    base = torch.randint(0, 50000, (groups, K), generator=g)
    base[:, 0] = 7
    if groups > 1:
        base[1] = base[0]
        base[1, -1] += 1
    if groups > 3:
        base[3] = base[2]
        base[3, 0] = base[2, 1] + STEP
        base[3, 1] = base[2, 0] - STEP
    return base


@pytest.mark.parametrize("loo", [False, True])
@pytest.mark.parametrize("B,groups,K", [(17, 4, 2), (63, 5, 3), (64, 8, 256), (65, 9, 257), (255, 1, 5),
                                        (256, 4, 64), (257, 16, 65), (1025, 100, 33)])
def test_rows_of_equal_hash_stay_apart(B, groups, K, loo):
    g = torch.Generator().manual_seed(B + K)
    gid = torch.randint(0, groups, (B,), generator=g)
    wide = torch.zeros((B, K + 3), dtype=torch.int64)
    wide[:, :K] = _rows(groups, K, g)[gid]
    rows = wide.to(DEV)[:, :K]  # a row stride of its own
    rewards = torch.rand(B, generator=g)
    valid = (torch.rand(B, generator=g) > 0.1).float()
    r, v = rewards.to(DEV), valid.to(DEV)
    want = baseline_and_std_per_prompt(gid[:, None], rewards, valid, loo)
    ids = _C.grpo_advantage(gid[:, None].to(DEV), r, v, loo, True, want_stats=True)
    for limit in (0, 1 << 40):  # hashed; compared directly
        keep = _C._ADV_DIRECT_ROWS
        _C._ADV_DIRECT_ROWS = limit
        try:
            got = _C.grpo_advantage(rows, r, v, loo, True, want_stats=True)
        finally:
            _C._ADV_DIRECT_ROWS = keep
        for a, b in zip(got, ids):
            assert torch.equal(a, b)
        # fp32 rounding of the oracle's sums of up to n rewards in [0, 1): n * 2^-24
        torch.testing.assert_close(got[1].cpu(), want[0], rtol=1e-5, atol=1e-6)
        assert torch.equal(got[3].cpu(), want[2])
