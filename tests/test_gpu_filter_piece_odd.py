"""The filtered backward's 8 KB pieces over rows that each start at another offset from a
16-byte boundary (V not a multiple of a vector), against the row-per-workgroup walk (GPU).

The sizes put the last piece's end around a piece's 512 vectors: rows of one launch with a
last piece that holds vectors and with one that holds only the elements after them.
"""

import pytest
import torch

from rl_amd import _C

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("dtype,V", [(torch.bfloat16, 5), (torch.bfloat16, 13), (torch.bfloat16, 4095),
                                     (torch.bfloat16, 4099), (torch.bfloat16, 4105), (torch.bfloat16, 4107),
                                     (torch.bfloat16, 38931), (torch.float16, 4107), (torch.float32, 2047),
                                     (torch.float32, 2053), (torch.float32, 20002),
                                     # whole vectors: pieces on lines would be one more
                                     (torch.bfloat16, 4088), (torch.float16, 8184), (torch.float32, 2044)])
@pytest.mark.parametrize("tied", [1, 8, 400])  # elements per distinct value: listed ties, and lists that overflow
@pytest.mark.parametrize("T", [1.0, 0.7])
def test_pieces_equal_walk(dtype, V, tied, T):
    B, S = 2, 17
    g = torch.Generator().manual_seed(V + tied)
    x = torch.randn(B, S, V, generator=g)
    if tied > 1:
        step = 8.0 * tied / V
        x = (x / step).round() * step
    x = x.to(dtype).to(DEV)
    tgt = torch.randint(0, V, (B, S - 1), generator=g)
    tgt[0, :2] = torch.tensor([0, V - 1])
    up = torch.randn(B, S - 1, generator=g)
    up[:, 3:6] = 0.0
    tgt, up = tgt.to(DEV), up.to(DEV)
    decision = torch.float32 if dtype != torch.float32 else None
    for p in (0.9, 0.4):
        info, kidx, kp = _C.filtered_fwd(x, tgt, T, 0, p, None, decision)
        out = []
        for pieces in (True, False):
            store = torch.full((B * S * V + 64,), 7.0, dtype=dtype, device=DEV)
            grad = store[:B * S * V].view(B, S, V)
            _C.filtered_bwd(x, tgt, T, info, kidx, kp, up, grad, top_k=0, pieces=pieces)
            assert torch.all(store[B * S * V:] == 7.0)
            out.append(grad)
        assert torch.equal(out[0], out[1])
        assert not out[0][:, -1].any() and not out[0][:, 3:6].any()
        # rows of another stride at the same offsets
        wide = torch.full((B, S, V + 16), 7.0, dtype=dtype, device=DEV)[..., :V]
        _C.filtered_bwd(x, tgt, T, info, kidx, kp, up, wide, top_k=0)
        assert torch.equal(wide, out[0])


@pytest.mark.parametrize("dtype,V", [(torch.bfloat16, 4099), (torch.bfloat16, 12290), (torch.float16, 8200),
                                     (torch.float32, 6149)])
@pytest.mark.parametrize("p", [0.97, 0.7, 0.45, 0.2])
def test_rank_cut_in_each_part_of_a_piece(dtype, V, p):
    """Rows of one value: every list overflows and the cut's rank falls into another part of
    another piece for each p."""
    B, S = 1, 9
    x = torch.zeros(B, S, V, dtype=dtype, device=DEV)
    tgt = torch.full((B, S - 1), V - 1, dtype=torch.int64, device=DEV)
    up = torch.ones(B, S - 1, device=DEV)
    info, kidx, kp = _C.filtered_fwd(x, tgt, 1.0, 0, p, None, torch.float32 if dtype != torch.float32 else None)
    out = []
    for pieces in (True, False):
        grad = torch.full((B, S, V), 7.0, dtype=dtype, device=DEV)
        _C.filtered_bwd(x, tgt, 1.0, info, kidx, kp, up, grad, top_k=0, pieces=pieces)
        out.append(grad)
    assert torch.equal(out[0], out[1])
    kept = (out[0][0, :-1] != 0).sum(-1)
    assert (kept >= int(p * V) - 8).all() and (kept <= int(p * V) + 8).all()
