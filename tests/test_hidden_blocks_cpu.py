"""The hidden-state path's rows per block and the splits of dH's reduction (CPU)."""

import pytest

from rl_amd.distributed.linear_ce import _block_rows, _dh_splits


@pytest.mark.parametrize("n", [1, 255, 257, 2048, 16384])
@pytest.mark.parametrize("H", [64, 300, 4096])
@pytest.mark.parametrize("K", [128, 1024, 1408, 9984, 32000, 151936])
def test_splits_give_whole_ranges(n, H, K):
    """Every split count leaves that many ranges of whole 128-element steps, none shorter than
    1024, as the GEMM requires; few tiles never ask for more workgroups than CUs."""
    tiles = -(-n // 256) * -(-H // 256)
    for known in (True, False):
        s = _dh_splits(n, H, K, known)
        assert s >= 1
        if s > 1:
            kb = -(-(-(-K // s)) // 128) * 128
            assert kb >= 1024 and -(-K // kb) == s
        assert s <= 8 or tiles * s <= 256


@pytest.mark.parametrize("T,chunk,per,V", [(1, 1, 1, 5), (100, 4, 3, 3001), (512, 64, 1, 32000), (16384, 256, 8, 151936),
                                           (16384, None, 8, 151936)])
def test_blocks_hold_a_chunk_and_fill_the_chip(T, chunk, per, V):
    rows = _block_rows(T, chunk, per, V)
    assert rows == T or (rows % 256 == 0 and rows >= chunk * per and rows // 256 * -(-V // 256) >= 512)
    if chunk is not None:
        # beyond a chunk: at most 512 tiles and one strip of the logits
        assert rows <= -(-chunk * per // 256) * 256 or rows * V <= 512 * 256 * 256 + 256 * V


@pytest.mark.parametrize("V", [300, 1000, 2047, 4000, 9973, 32000, 151936])
@pytest.mark.parametrize("H", [64, 1024, 4096, 8192])
def test_scratch_of_a_block(V, H):
    """The fp32 backward's scratch for a block of a tiny chunk: logits, their transpose and dH's
    partial products stay within what _block_rows states."""
    rows = _block_rows(1 << 24, 1, 1, V)
    K = -(-V // 64) * 64
    part = _dh_splits(rows, H, K, count_known=False) * rows * H
    assert rows * V <= 512 * 65536 + 256 * V
    assert part <= max(1 << 24, -(-V // 1024) * rows * H)
    if (V, H) == (4000, 4096):
        assert rows == 8192 and part * 4 == 268435456
