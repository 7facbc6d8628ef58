"""Top-k / top-p over rows with a chosen number of distinct 16-bit values (GPU).

The entry-list kernel gives each thread an equal share of the row's distinct values and its
phases stop at the shares' length; the numbers here lie around whole shares and whole groups
of them (512 threads for bf16, 1024 for fp16).  The same values as fp32 logits go through
the fp32 kernels, which hold no such list: the kept counts must be equal, the same targets
kept, and the logprobs agree to the fp32 rounding of the sums (1e-6 relative, 1e-5 absolute
on values up to 20).  (The recorded cut value is not compared: a cut between two values may
be named by either, with all or none of its ties kept.)
"""

import pytest
import torch

from rl_amd import _C

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
V = 20000


@pytest.mark.parametrize("dtype,distinct", [(torch.bfloat16, n) for n in (1, 2, 511, 512, 513, 1536, 1537, 3073)]
                         + [(torch.float16, n) for n in (1, 1023, 1025, 3072, 3073, 9217, 18000)])
@pytest.mark.parametrize("k,p", [(0, 0.9), (0, 0.2), (0, 0.999), (3000, 0.9), (1500, 1.0)])
@pytest.mark.parametrize("T", [1.0, 0.7])
def test_share_lengths(dtype, distinct, k, p, T):
    B, S = 1, 6
    g = torch.Generator().manual_seed(distinct + k)
    pool = torch.arange(0x10000, dtype=torch.int32).to(torch.int16).view(dtype)
    pool = pool[(pool.float().abs() < 9) & (pool.float().abs() > 2.0 ** -14)]
    rows = []
    for _ in range(B * S):
        vals = pool[torch.randperm(pool.numel(), generator=g)[:distinct]]
        row = vals[torch.randint(0, distinct, (V,), generator=g)]
        row[torch.randperm(V, generator=g)[:distinct]] = vals  # each at least once
        rows.append(row)
    x = torch.stack(rows).view(B, S, V).to(DEV)
    y = (x.float() * torch.tensor(1.0 / T, dtype=torch.float32, device=DEV)).to(dtype) if T != 1.0 else x
    tgt = torch.randint(0, V, (B, S), generator=g).to(DEV)
    out, ref = torch.empty((B, S), device=DEV), torch.empty((B, S), device=DEV)
    info, _, _ = _C.filtered_fwd(x, tgt, T, k, p, out, torch.float32)
    want, _, _ = _C.filtered_fwd(y.float(), tgt, 1.0, k, p, ref)
    a, b = (t.cpu().view(torch.int32).view(-1, 6) for t in (info, want))
    assert torch.equal(a[:, 4], b[:, 4]), "kept count"
    # a tie at the cut is kept from a rank (here) or an index (fp32) on: the same elements
    assert torch.equal(torch.isinf(out), torch.isinf(ref))
    fin = ~torch.isinf(out)
    assert torch.allclose(out[fin], ref[fin], rtol=1e-6, atol=1e-5)
