"""Calls whose kernels would hold 2^32 threads or more in one launch, past
which a grid wraps without an error and runs only what is left of it."""
import pytest
import torch

from foundry_attn import attn_bwd, attn_fwd, lora_bwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,B,H,masked", [(torch.bfloat16, 2, (1 << 22) + 1, False),
                                              (torch.bfloat16, (1 << 22) + 1, 2, True),
                                              (torch.float32, 2, (1 << 23) + 1, False)])
def test_attention_over_many_heads(dtype, B, H, masked):
    """One token per (batch, head), 64 features: O = V, dV = dO, dQ = dK = 0
    (the softmax of one score is 1), and zeros where the mask excludes it."""
    S, D = 1, 64
    gen = torch.Generator(device="cuda").manual_seed(H)
    # rows of a head D apart (bf16 operands span less than 2 GiB per head)
    x, do = (torch.randn(B, H, S, D, device="cuda", generator=gen, dtype=dtype).transpose(1, 2) for _ in range(2))
    keep = None
    if masked:
        keep = torch.ones(B, S, dtype=torch.uint8, device="cuda")
        keep[::3] = 0
    o, lse = attn_fwd(x, x, x, key_keep=keep)
    dq, dk, dv = attn_bwd(x, x, x, o, do, lse, key_keep=keep)
    torch.cuda.synchronize()
    kept = torch.ones(B, dtype=torch.bool, device="cuda") if keep is None else keep[:, 0].bool()
    assert bool(torch.isfinite(lse).all(-1).all(-1).eq(kept).all())
    # bf16 rounds P to 1.  f32: O = P V / P to three roundings; the backward's P = 2^(s c - lse2), whose two terms
    # (below 64) each carry three roundings
    for got, want, rel in ((o, x, 2.0 ** -22), (dv, do, 6 * 64 * 2.0 ** -24)):
        rel = 0.0 if dtype == torch.bfloat16 else rel
        assert bool(((got[kept] - want[kept]).abs() <= rel * want[kept].abs()).all())
        assert float(got[~kept].abs().sum()) == 0
    # dS is the rounding of two 64-term sums of dO V (|dO V| sums below 200), dQ and dK 0.125 dS |x| (below 6.5)
    for g in (dq, dk):
        assert float(g.abs().max()) <= 0.125 * 6.5 * 128 * 200 * 2.0 ** -24


def test_lora_gradient_of_2_26_features():
    """dA of one token and rank 1 is that token: C x 32 partial sums, 2^31."""
    K = 1 << 26
    x = torch.randn(1, K, device="cuda", dtype=torch.bfloat16)
    a = torch.zeros(1, K, device="cuda", dtype=torch.bfloat16)
    b, dy = (torch.zeros(*s, device="cuda", dtype=torch.bfloat16) for s in ((16, 1), (1, 16)))
    b[3, 0] = dy[0, 3] = 1
    da, db = lora_bwd(x, a, b, torch.full((1, 1), 2.0, device="cuda"), dy, 1.0)
    assert torch.equal(da, x.float())
    assert torch.equal(db, 2 * dy.float().t())


def test_lora_f32_gradient_of_2_29_tokens():
    """du of the last tokens, which a wrapped grid of the down product would
    leave out, reaches dA: all other tokens are zero."""
    N, K, M = (1 << 29) + 5, 4, 4
    x, dy = torch.zeros(N, K, device="cuda"), torch.zeros(N, M, device="cuda")
    u = torch.zeros(N, 1, device="cuda")
    x[-3:, 1] = torch.tensor([1.0, 2.0, 3.0], device="cuda")
    dy[-3:, 0] = 1
    u[-3:] = 1
    a, b = torch.ones(1, K, device="cuda"), torch.tensor([[2.0], [1.0], [1.0], [1.0]], device="cuda")
    da, db = lora_bwd(x, a, b, u, dy, 1.0)
    assert da.tolist() == [[0.0, 12.0, 0.0, 0.0]] and db.tolist() == [[3.0], [0.0], [0.0], [0.0]]
