"""Which prompt rows are compared pair by pair and which are hashed (CPU)."""

import pytest

from rl_amd._C import _adv_direct


@pytest.mark.parametrize("B,K,direct", [(1, 1 << 20, True), (2, 16384, True), (4096, 1, True), (24, 64, True),
                                        (32, 2, True), (3, 4096, True), (16, 512, True), (8, 1024, True), (24, 512, False),
                                        (64, 2, False), (4, 4096, False), (16, 1024, False), (8, 16384, False)])
def test_route_follows_the_work(B, K, direct):
    """Few or short rows in one launch, many or long ones hashed: the comparison of a pair
    grows with the row's length, the three launches of the other route hardly."""
    assert _adv_direct(B, K) == direct
