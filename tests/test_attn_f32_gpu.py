"""The f32 attention kernels (csrc/attn_f32.hip) at their workgroup shapes'
edges, against the oracle.  The bound: every output is a chain of f32 sums
and products over at most S + 2 D terms, each rounded to 2^-24, in the kernel
and in the oracle."""
import numpy as np
import pytest
import torch

import oracle
from foundry_attn import _abi, attn_bwd, attn_fwd
from foundry_attn.ops import attn_bwd_workspace_bytes
from helpers import rel_l2

pytestmark = pytest.mark.gpu


def check(q, k, v, do, keep, o, lse, grads):
    B, S, H, D = q.shape
    scale = 1 / np.sqrt(D)
    wo, wl = oracle.attn_fwd(q, k, v, scale=scale, key_keep=keep, bf16=False)
    want = (wo,) + oracle.attn_bwd(q, k, v, do, scale=scale, key_keep=keep, bf16=False)
    bound = 2 * (S + 2 * D) * 2.0 ** -24
    for name, g, w in zip(("o", "dq", "dk", "dv"), (o,) + grads, want):
        r = rel_l2(g.cpu().numpy(), w)
        assert r <= bound, (name, r, bound)
    np.testing.assert_allclose(lse.cpu().numpy(), wl, rtol=1e-5, atol=1e-5)


# One, two and four streaming groups per workgroup (the launcher's choice for
# these grids on 256 CUs); sequence lengths that leave a partial last row tile,
# a partial last block, and groups with no block at all.
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,S,H", [(1, 500, 60), (1, 300, 48), (1, 97, 5), (2, 33, 3), (1, 130, 2)])
def test_groups_and_remainders(B, S, H, D):
    rng = np.random.default_rng(S + D)
    q, k, v, do = (rng.standard_normal((B, S, H, D)).astype(np.float32) for _ in range(4))
    keep = np.ones((B, S), np.uint8)
    keep[0, S // 3:S // 2] = 0
    t = [torch.from_numpy(a).cuda() for a in (q, k, v, do)]
    tk = torch.from_numpy(keep).cuda()
    o, lse = attn_fwd(*t[:3], key_keep=tk)
    grads = attn_bwd(*t[:3], o, t[3], lse, key_keep=tk)
    check(q, k, v, do, keep, o, lse, grads)
    # the recomputing dQ (minimum workspace, or separate phases with any) gives the same bits
    full = torch.empty(attn_bwd_workspace_bytes(B, S, H, D, torch.float32), dtype=torch.uint8, device="cuda")
    least = full[:attn_bwd_workspace_bytes(B, S, H, D, torch.float32, minimum=True)]
    phases = [(p, None) for p in (_abi.FA_BWD_PREPASS, _abi.FA_BWD_DQ, _abi.FA_BWD_DKDV)]
    for ws, ph in ((least, None), (full, phases)):
        for a, b in zip(attn_bwd(*t[:3], o, t[3], lse, key_keep=tk, workspace=ws, phases=ph), grads):
            assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,S,H", [(torch.float32, 300, 4), (torch.bfloat16, 4608, 24)])
def test_backward_without_room_for_ds(monkeypatch, dtype, S, H):
    """Where memory has no room for the stored dS, the recomputing dQ runs: the same bits."""
    gen = torch.Generator(device="cuda").manual_seed(S)
    q, k, v, do = (torch.randn(1, S, H, 128, device="cuda", generator=gen).to(dtype) for _ in range(4))
    o, lse = attn_fwd(q, k, v)
    want = attn_bwd(q, k, v, o, do, lse)
    least = attn_bwd_workspace_bytes(1, S, H, 128, dtype, minimum=True)
    assert attn_bwd_workspace_bytes(1, S, H, 128, dtype) > least
    empty, refused = torch.empty, []

    def limited(*shape, **kw):
        if kw.get("dtype") == torch.uint8 and shape[0] > least:
            refused.append(shape[0])
            raise torch.cuda.OutOfMemoryError("no room")
        return empty(*shape, **kw)

    monkeypatch.setattr(torch, "empty", limited)
    got = attn_bwd(q, k, v, o, do, lse)
    assert refused
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_graph_and_phases_hold_no_ds(monkeypatch):
    """A captured f32 backward keeps no dS in its graph's memory, and separate
    phases (which do not use it) allocate none: the same bits, on replays too."""
    B, S, H, D = 1, 1056, 4, 128
    ds_bytes = 4 * H * S * S
    t = [torch.randn(B, S, H, D, device="cuda") for _ in range(4)]
    out = [torch.empty_like(t[0]) for _ in range(3)]
    o, lse = attn_fwd(*t[:3])
    want = attn_bwd(*t[:3], o, t[3], lse)
    sizes, empty = [], torch.empty

    def recorded(*shape, **kw):
        if kw.get("dtype") == torch.uint8:
            sizes.append(shape[0])
        return empty(*shape, **kw)

    monkeypatch.setattr(torch, "empty", recorded)
    phases = [(p, None) for p in (_abi.FA_BWD_PREPASS, _abi.FA_BWD_DKDV, _abi.FA_BWD_DQ)]
    for a, b in zip(attn_bwd(*t[:3], o, t[3], lse, phases=phases), want):
        assert torch.equal(a, b)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        attn_bwd(*t[:3], o, t[3], lse, out=out)
    assert len(sizes) == 2 and max(sizes) < ds_bytes, sizes
    for _ in range(3):
        for g in out:
            g.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, want):
            assert torch.equal(a, b)
    attn_bwd(*t[:3], o, t[3], lse)
    assert sizes[-1] > ds_bytes  # the eager call still takes it


@pytest.mark.parametrize("D", [64, 128])
def test_row_stride_past_32_bit_offsets(D):
    """Rows 2^25 elements apart: a 32-row tile spans 4 GiB and more."""
    S, stride = 3, 1 << 25
    rng = np.random.default_rng(D)
    host = [rng.standard_normal((1, S, 1, D)).astype(np.float32) for _ in range(4)]
    buf = torch.empty(2 * stride + 4 * D, device="cuda")
    views = []
    for i, a in enumerate(host):
        view = buf.as_strided((1, S, 1, D), (0, stride, D, 1), i * D)
        view.copy_(torch.from_numpy(a))
        views.append(view)
    o, lse = attn_fwd(*views[:3])
    check(*host, None, o, lse, attn_bwd(*views[:3], o, views[3], lse))


def test_reference_moves_after_small_scores():
    """Scores that grow along the keys move the exp2 reference in later
    blocks, after O and the row sum were accumulated under an earlier one."""
    rng = np.random.default_rng(5)
    q, k, v, do = (rng.standard_normal((1, 200, 2, 128)).astype(np.float32) for _ in range(4))
    k *= np.linspace(0.1, 12, 200, dtype=np.float32)[None, :, None, None]
    t = [torch.from_numpy(a).cuda() for a in (q, k, v, do)]
    o, lse = attn_fwd(*t[:3])
    wo, wl = oracle.attn_fwd(q, k, v, scale=128 ** -0.5, key_keep=None, bf16=False)
    # |score| reaches ~40: its f32 rounding, 40 * 2^-24 per product chain, is P's relative error
    assert rel_l2(o.cpu().numpy(), wo) <= 2 * (200 + 256) * 40 * 2.0 ** -24
    np.testing.assert_allclose(lse.cpu().numpy(), wl, rtol=1e-5, atol=1e-5)
