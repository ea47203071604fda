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


@pytest.mark.parametrize("N,K,M,r", [(1536, 3072, 3072, 32), (1536, 3072, 3072, 16), (1025, 1024, 512, 32),
                                     (257, 256, 260, 17), (37, 512, 256, 32), (5, 64, 128, 9), (1, 16, 16, 32)])
def test_lora_f32_vector_up_products_by_element(N, K, M, r):
    """y and dx with aligned rows, element by element: each within the rounding
    of its own sums (N % 4 == 1 leaves a wave's last group of four rows with
    one), and four rows past N untouched."""
    torch.manual_seed(N + 7 * r)
    x, dy = torch.randn(N, K, device="cuda"), torch.randn(N, M, device="cuda")
    a, b = torch.randn(r, K, device="cuda"), torch.randn(M, r, device="cuda")
    yf, dxf = torch.randn(N + 4, M, device="cuda"), torch.randn(N + 4, K, device="cuda")
    y0, dx0 = yf.clone(), dxf.clone()
    for _ in range(3):  # the same bits each time
        yf.copy_(y0)
        dxf.copy_(dx0)
        u = lora_fwd(x, a, b, yf[:N], 0.5)
        lora_bwd(x, a, b, u, dy, 0.5, dx=dxf[:N])
        X, A, B, DY, Y0, DX0 = (t.double() for t in (x, a, b, dy, y0[:N], dx0[:N]))
        for name, got, start, left, w1, w2, k in (("y", yf, Y0, X, A.t(), B.t(), K), ("dx", dxf, DX0, DY, B, A, M)):
            want = start + 0.5 * left @ w1 @ w2
            # k + r products and sums, the scale and the addition, each rounded to 2^-24
            bound = 2.0 ** -24 * ((k + r + 3) * 0.5 * left.abs() @ w1.abs() @ w2.abs() + start.abs() + want.abs())
            over = (got[:N].double() - want).abs() - bound
            assert bool((over <= 0).all()), (name, int((over > 0).sum()), float(over.max()))
        assert torch.equal(yf[N:], y0[N:]) and torch.equal(dxf[N:], dx0[N:])


@pytest.mark.parametrize("dtype,K,M", [(torch.float32, 44, 20), (torch.float32, 3076, 1028), (torch.bfloat16, 48, 16),
                                       (torch.bfloat16, 3088, 1040)])
def test_non_finite_factor_row_stays_in_its_rank(dtype, K, M):
    """A NaN or infinity in one rank's row of A reaches that column of u only,
    and one in B that row of dA only, where the last 64 bytes of a row are cut
    short by the next row's first values."""
    torch.manual_seed(K)
    N, r, bad = 70, 20, 7
    x, dy = torch.randn(N, K, device="cuda").to(dtype), torch.randn(N, M, device="cuda").to(dtype)
    a, b = torch.randn(r, K, device="cuda").to(dtype), torch.randn(M, r, device="cuda").to(dtype)
    y = torch.zeros(N, M, device="cuda", dtype=dtype)
    u = lora_fwd(x, a, b, y.clone(), 0.5)
    da, db = lora_bwd(x, a, b, u, dy, 0.5)
    others = [j for j in range(r) if j != bad]
    for value in (float("nan"), float("inf")):
        a2, b2 = a.clone(), b.clone()
        a2[bad, 0], b2[0, bad] = value, value
        u2 = lora_fwd(x, a2, b, y.clone(), 0.5)
        da2, db2 = lora_bwd(x, a, b2, u, dy, 0.5)
        assert torch.equal(u2[:, others], u[:, others]) and not bool(torch.isfinite(u2[:, bad]).any())
        assert torch.equal(da2[others], da[others]) and not bool(torch.isfinite(da2[bad]).any())
        assert torch.equal(db2, db)


@pytest.mark.parametrize("stride", [1 << 24, 1 << 26])
def test_lora_f32_row_strides_past_32_bit_offsets(stride):
    """Rows of x, dy, y and dx far apart: 64 of them past 4 GiB (the general
    down and up products), and 16 (the general gradient as well)."""
    N, K, M, r = 3, 8, 12, 5
    torch.manual_seed(stride >> 20)
    buf = torch.empty((N - 1) * stride + 128, device="cuda")
    x, dy, y, dx = (buf.as_strided((N, w), (stride, 1), at) for w, at in ((K, 0), (M, 16), (M, 32), (K, 48)))
    for t in (x, dy, y, dx):
        t.copy_(torch.randn(t.shape, device="cuda"))
    a, b = torch.randn(r, K, device="cuda"), torch.randn(M, r, device="cuda")
    X, DY, Y, DX, A, B = (t.double().cpu() for t in (x, dy, y, dx, a, b))
    u = lora_fwd(x, a, b, y, 0.5)
    da, db = lora_bwd(x, a, b, u, dy, 0.5, dx=dx)
    U, DU = X @ A.t(), 0.5 * (DY @ B)
    for name, got, want in (("u", u, U), ("y", y, Y + 0.5 * U @ B.t()), ("da", da, DU.t() @ X),
                            ("db", db, 0.5 * DY.t() @ U), ("dx", dx, DX + DU @ A)):
        err = float((got.double().cpu() - want).norm() / want.norm())
        assert err <= (max(N, K, M) + r) * 2.0 ** -24, (name, err)
    assert torch.equal(x.double().cpu(), X) and torch.equal(dy.double().cpu(), DY)
