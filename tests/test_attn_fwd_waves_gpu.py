"""The bf16 forward where a grid's last round decides its workgroup shape: a
batch that runs 4-wave workgroups gives the bits of its halves, which run
8-wave ones (a query's arithmetic does not depend on the shape).  On 256 CUs
the 4-wave grids' last rounds are exactly one workgroup per CU, a few less, and
(the last two) a few more, which stay 8-wave."""
import pytest
import torch

from foundry_attn import attn_fwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("B,S,H,D", [(4, 1024, 24, 128), (4, 900, 24, 64), (6, 600, 25, 128), (2, 1795, 25, 64),
                                     (2, 1921, 25, 128), (2, 2048, 25, 64)])
def test_batch_matches_halves(B, S, H, D, masked):
    torch.manual_seed(S + H)
    q, k, v = (torch.randn(B, S, H, D, device="cuda").to(torch.bfloat16) for _ in range(3))
    keep = None
    if masked:
        keep = torch.ones(B, S, dtype=torch.uint8, device="cuda")
        keep[::2, S // 4:S // 2] = 0
    o, lse = attn_fwd(q, k, v, key_keep=keep)
    n = B // 2
    for h in (slice(0, n), slice(n, B)):
        oh, lh = attn_fwd(q[h], k[h], v[h], key_keep=None if keep is None else keep[h])
        assert torch.equal(o[h], oh) and torch.equal(lse[h], lh)
