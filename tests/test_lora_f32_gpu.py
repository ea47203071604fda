"""The f32 LoRA kernels over the shapes that choose between them: rows on and
off 16-byte alignment, widths that are and are not multiples of 4, ranks at
and between the register sizes, token counts around a block, a split and
several splits.  Each result is a chain of at most max(N, K, M) + r f32 sums
and products, each rounded to 2^-24."""
import pytest
import torch

from foundry_attn import lora_bwd, lora_fwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K,M,r,ypad,dxpad", [
    (1, 2, 6, 1, 0, 0),            # the smallest; K off 4: the general down product
    (37, 256, 770, 4, 0, 0),       # M off 4: the general up product
    (130, 258, 512, 12, 2, 0),     # y rows off 16 bytes; two token splits' worth of rows
    (700, 768, 256, 32, 0, 1),     # dx rows off 16 bytes, the widest rank
    (100, 1056, 1540, 17, 4, 4),   # column tiles cut short, a k-step cut short
    (1000, 44, 44, 8, 0, 0),       # fewer columns than a tile, several splits
    (257, 3072, 300, 16, 0, 0),
])
def test_lora_f32_shapes(N, K, M, r, ypad, dxpad):
    torch.manual_seed(N + r)
    x = torch.randn(N, K + (-K) % 4, device="cuda")[:, :K]
    dy = torch.randn(N, M + (-M) % 4, device="cuda")[:, :M]
    a, b = torch.randn(r, K, device="cuda"), torch.randn(M, r, device="cuda")
    yf, dxf = torch.randn(N + 1, M + ypad, device="cuda"), torch.randn(N + 1, K + dxpad, device="cuda")
    y0, dx0 = yf.double().cpu(), dxf.double().cpu()
    u = lora_fwd(x, a, b, yf[:N, :M], 0.5)
    da, db = lora_bwd(x, a, b, u, dy, 0.5, dx=dxf[:N, :K])
    X, A, B, DY = (t.double().cpu() for t in (x, a, b, dy))
    U, DU = X @ A.t(), 0.5 * (DY @ B)
    wy, wdx = y0.clone(), dx0.clone()  # padding columns and the row past N stay as they were
    wy[:N, :M] += 0.5 * U @ B.t()
    wdx[:N, :K] += DU @ A
    bound = (max(N, K, M) + r) * 2.0 ** -24
    for name, got, want in (("u", u, U), ("y", yf, wy), ("da", da, DU.t() @ X), ("db", db, 0.5 * DY.t() @ U),
                            ("dx", dxf, wdx)):
        err = float((got.double().cpu() - want).norm() / want.norm())
        assert err <= bound, (name, err, bound)
    assert torch.equal(yf[N].cpu().double(), y0[N]) and torch.equal(dxf[N].cpu().double(), dx0[N])
