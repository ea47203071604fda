"""The one-grid dK/dV + dQ of the 4-wave bf16 backward: the bits of the two
kernels issued as separate phases, over tile remainders, masks, D = 64 on
grids where D = 128 takes 8 waves, grids the range split leaves alone, and
both ends of the sizes whose workgroups are reordered."""
import pytest
import torch

from foundry_attn import _abi, attn_bwd, attn_fwd
from foundry_attn.ops import attn_bwd_workspace_bytes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("B,S,H,D", [(1, 1, 1, 128), (2, 129, 3, 128), (1, 511, 5, 64), (1, 700, 24, 128),
                                     (1, 1100, 44, 64), (1, 1100, 4, 128), (1, 1024, 24, 64),
                                     (1, 128, 512, 128), (1, 100, 513, 128), (1, 128, 608, 128),
                                     (1, 70, 609, 128), (2, 1400, 24, 128), (1, 100, 520, 64)])
def test_pair_matches_phases(B, S, H, D, masked):
    torch.manual_seed(S + H)
    q, k, v, do = (torch.randn(B, S, H, D, device="cuda").to(torch.bfloat16) for _ in range(4))
    keep = None
    if masked:
        keep = torch.ones(B, S, dtype=torch.uint8, device="cuda")
        keep[0, S // 4:S // 2] = 0
    o, lse = attn_fwd(q, k, v, key_keep=keep)
    got = attn_bwd(q, k, v, o, do, lse, key_keep=keep)
    ws = torch.empty(attn_bwd_workspace_bytes(B, S, H, D, minimum=True), dtype=torch.uint8, device="cuda")
    phases = [(p, None) for p in (_abi.FA_BWD_PREPASS, _abi.FA_BWD_DQ, _abi.FA_BWD_DKDV)]
    want = attn_bwd(q, k, v, o, do, lse, key_keep=keep, workspace=ws, phases=phases)
    for name, a, b in zip(("dq", "dk", "dv"), got, want):
        assert torch.equal(a, b), name
