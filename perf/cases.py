"""The work that programs have this framework do, as timed cases.

Every case is one pass through the public entry points of foundry_attn:

  attention  the joint text + image attention, forward and backward, through
             the plain calls (attn_fwd, attn_bwd) or the autograd wrapper
  prologue   QK-RMSNorm + axial RoPE of the text and image streams' Q and K
             into the joint buffers, and its gradient
  lora       one adapter beside a frozen linear: lora_fwd and lora_bwd
  mlp        the row-wise operators around a block's linears
  double     a double-stream LoRA block's forward and backward
  single     a single-stream LoRA block's forward and backward

listed() holds fixed cases, draw() further ones of the same ranges: the
sequence of a training bucket runs from a 64-pixel crop (tens of tokens) to
about 1.5 megapixels (6656 tokens), heads from one to the model's 24 (fewer
where a sequence-parallel group divides them), storage is bf16 or, for runs
that check the bf16 path, f32.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "foundry-trainer_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import foundry_attn as fa  # noqa: E402
from foundry_attn import block as fb  # noqa: E402

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
STREAMS = ("txt", "img")
AXES3, THETA3 = (16, 56, 56), 1e4           # (text index, row, column)
AXES4, THETA4 = (32, 32, 32, 32), 2000.0    # the single-stream block's (t, h, w, l)
EPS = 1e-6


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # The smallest op-level call: B1 H4 D64 S256 in f32 (64 text + 192 image
        # tokens), as a numerics check of the op runs it, through autograd.
        dict(name="attn_f32_256", kind="attention", dtype="f32", batch=1, heads=4, head_dim=64, seq=256, txt=64,
             valid=0, api="autograd"),
        # A 256-pixel preview bucket: 16 x 16 image tokens after 77 text slots of
        # which 41 hold the prompt, two samples, in a training step (autograd).
        dict(name="attn_bf16_333", kind="attention", dtype="bf16", batch=2, heads=24, head_dim=128, seq=333, txt=77,
             valid=41, api="autograd"),
        # 512 pixels, batch 4: 512 text + 32 x 32 image tokens.
        dict(name="attn_bf16_1536x4", kind="attention", dtype="bf16", batch=4, heads=24, head_dim=128, seq=1536,
             txt=512, valid=0, api="op"),
        # 1024 pixels, one sample: 512 text + 64 x 64 image tokens.
        dict(name="attn_bf16_4608", kind="attention", dtype="bf16", batch=1, heads=24, head_dim=128, seq=4608,
             txt=512, valid=0, api="op"),
        # 1024 x 1536 pixels, two samples of an aspect bucket, padded prompts
        # excluded by the key mask.
        dict(name="attn_bf16_6656x2", kind="attention", dtype="bf16", batch=2, heads=24, head_dim=128, seq=6656,
             txt=512, valid=77, api="op"),
        # One 512-pixel sample in f32: the run a bf16 one is checked against.
        dict(name="attn_f32_1536", kind="attention", dtype="f32", batch=1, heads=24, head_dim=128, seq=1536, txt=512,
             valid=0, api="op"),
        # Q and K of the 1024-pixel sample, normalised and rotated.
        dict(name="prologue_4608", kind="prologue", dtype="bf16", heads=24, head_dim=128, txt=512, rows=64, cols=64),
        # One rank-16 adapter on a frozen 3072 x 3072 projection, 1024 pixels.
        dict(name="lora_bf16_4096", kind="lora", dtype="bf16", tokens=4096, fin=3072, fout=3072, rank=16, dx=True),
        # The same adapter in f32 at 512 pixels.
        dict(name="lora_f32_1536", kind="lora", dtype="f32", tokens=1536, fin=3072, fout=3072, rank=16, dx=True),
        # The row-wise operators of the single-stream block at 1024 pixels.
        dict(name="mlp_swiglu_4608", kind="mlp", dtype="bf16", act="swiglu", tokens=4608, width=3072, ratio=3),
        # The whole double-stream block at 1024 pixels, with the input gradient.
        dict(name="double_4608", kind="double", dtype="bf16", heads=24, head_dim=128, txt=512, rows=64, cols=64,
             rank=16),
        # The whole single-stream block at 512 pixels, with the input gradient.
        dict(name="single_1536", kind="single", dtype="bf16", heads=24, head_dim=128, txt=512, rows=32, cols=32,
             rank=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _attention_flops(case):
    kept = sum(case["seq"] - (case["txt"] - v) for v in _valid(case))
    return 14.0 * case["heads"] * case["seq"] * kept * case["head_dim"]


def draw(rng):
    kind = rng.choice(["attention", "attention", "attention", "attention", "prologue", "lora", "lora", "mlp",
                       "double", "single"])
    if kind == "attention":
        dtype = rng.choice(["bf16", "bf16", "f32"])
        seq = _log_int(rng, 24, 6656 if dtype == "bf16" else 1536)
        txt = min(rng.choice([16, 77, 256, 512]), max(1, seq // 3))
        case = dict(kind=kind, dtype=dtype, batch=rng.randint(1, 4), heads=rng.choice([1, 2, 3, 4, 6, 8, 12, 24]),
                    head_dim=rng.choice([64, 128, 128, 128]), seq=seq, txt=txt,
                    valid=rng.choice([0, max(1, txt // 5), max(1, txt // 2)]), api=rng.choice(["op", "autograd"]))
        most = 3.6e12 if dtype == "bf16" else 1.0e11
        while _attention_flops(case) > most:
            if case["batch"] > 1:
                case["batch"] -= 1
            else:
                case["heads"] //= 2
        return case
    if kind == "prologue":
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "bf16", "f32"]), heads=rng.choice([2, 3, 6, 12, 24]),
                    head_dim=128, txt=rng.choice([16, 77, 256, 512]), rows=_log_int(rng, 4, 64),
                    cols=_log_int(rng, 4, 64))
    if kind == "lora":
        dtype = rng.choice(["bf16", "bf16", "f32"])
        return dict(kind=kind, dtype=dtype, tokens=_log_int(rng, 24, 4608 if dtype == "bf16" else 1536),
                    fin=rng.choice([256, 768, 1536, 3072]), fout=rng.choice([256, 768, 1536, 3072]),
                    rank=rng.choice([4, 8, 12, 16, 32]), dx=rng.random() < 0.75)
    if kind == "mlp":
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "bf16", "f32"]), act=rng.choice(["gelu", "swiglu"]),
                    tokens=_log_int(rng, 24, 4608), width=rng.choice([256, 768, 1536, 3072]), ratio=3)
    side = rng.choice([8, 16, 24, 32, 48])
    return dict(kind=kind, dtype="bf16", heads=24, head_dim=128, txt=rng.choice([77, 256, 512]), rows=side,
                cols=rng.choice([side, side * 3 // 4, side * 5 // 4]), rank=rng.choice([4, 16]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _valid(case):
    """Kept text tokens per sample: `valid` of the txt slots in every even
    sample, all of them in the odd ones; valid = 0 means no mask."""
    if not case["valid"]:
        return [case["txt"]] * case["batch"]
    return [case["valid"] if i % 2 == 0 else case["txt"] for i in range(case["batch"])]


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(gen, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=gen, device=DEV) * std).to(dtype)


def _unit_rows(gen, *shape, dtype):
    """Rows as they leave the QK-RMSNorm (unit root mean square times a learned
    scale near 1); the rotation that follows does not change their lengths."""
    x = torch.randn(*shape, generator=gen, device=DEV)
    w = 1 + 0.02 * torch.randn(shape[-1], generator=gen, device=DEV)
    return (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w).to(dtype)


def _positions(txt, rows, cols):
    pos = torch.zeros(txt + rows * cols, 3)
    pos[:txt, 0] = torch.arange(txt)
    i = torch.arange(rows * cols)
    pos[txt:, 1], pos[txt:, 2] = (i // cols).float(), (i % cols).float()
    return pos.numpy()


def _prepare_attention(case, gen):
    dt = DTYPES[case["dtype"]]
    shape = (case["batch"], case["seq"], case["heads"], case["head_dim"])
    st = dict(q=_unit_rows(gen, *shape, dtype=dt), k=_unit_rows(gen, *shape, dtype=dt),
              v=_randn(gen, *shape, dtype=dt), do=_randn(gen, *shape, dtype=dt), keep=None)
    if case["valid"]:
        keep = torch.ones(shape[:2], dtype=torch.uint8, device=DEV)
        for b, n in enumerate(_valid(case)):
            keep[b, n:case["txt"]] = 0
        st["keep"] = keep
    if case["api"] == "autograd":
        for t in "qkv":
            st[t].requires_grad_(True)
    return st


def _prepare_prologue(case, gen):
    dt = DTYPES[case["dtype"]]
    H, D = case["heads"], case["head_dim"]
    C, T, I = H * D, case["txt"], case["rows"] * case["cols"]
    cos, sin = fa.rope_tables(_positions(T, case["rows"], case["cols"]), AXES3, THETA3, dtype=dt, device=DEV)
    st = dict(qkv=_randn(gen, T + I, 3 * C, dtype=dt), dq=_randn(gen, 1, T + I, H, D, dtype=dt),
              dk=_randn(gen, 1, T + I, H, D, dtype=dt), dqkv=torch.zeros(T + I, 3 * C, dtype=dt, device=DEV),
              q=torch.empty(1, T + I, H, D, dtype=dt, device=DEV), k=torch.empty(1, T + I, H, D, dtype=dt, device=DEV))
    st["norm"] = {s + t: _randn(gen, D, std=0.02).add_(1).to(dt) for s in STREAMS for t in "qk"}
    st["rope"] = {"txt": (cos[:T].contiguous(), sin[:T].contiguous()),
                  "img": (cos[T:].contiguous(), sin[T:].contiguous())}
    fwd, bwd = [], []
    for s, off, n in (("txt", 0, T), ("img", T, I)):
        c, r = st["rope"][s]
        for j, t in enumerate("qk"):
            x = st["qkv"][off:off + n, j * C:(j + 1) * C].view(1, n, H, D)
            dx = st["dqkv"][off:off + n, j * C:(j + 1) * C].view(1, n, H, D)
            fwd.append((x, st["norm"][s + t], c, r, AXES3, st[t], off))
            bwd.append((x, st["norm"][s + t], c, r, AXES3, st["d" + t], off, dx))
    st["fwd"], st["bwd"] = fwd, bwd
    return st


def _prepare_lora(case, gen):
    dt = DTYPES[case["dtype"]]
    N, K, M, r = case["tokens"], case["fin"], case["fout"], case["rank"]
    st = dict(x=_randn(gen, N, K, dtype=dt), a=_randn(gen, r, K, std=1.0 / r, dtype=dt),
              b=_randn(gen, M, r, std=1e-2, dtype=dt), base=_randn(gen, N, M, dtype=dt),
              dy=_randn(gen, N, M, dtype=dt), y=torch.empty(N, M, dtype=dt, device=DEV), scale=16.0 / r)
    if case["dx"]:
        st["dbase"] = _randn(gen, N, K, dtype=dt)
        st["dx"] = torch.empty(N, K, dtype=dt, device=DEV)
    return st


def _prepare_mlp(case, gen):
    dt = DTYPES[case["dtype"]]
    N, C, M = case["tokens"], case["width"], case["ratio"] * case["width"]
    st = dict(x=_randn(gen, N, C, dtype=dt), out=_randn(gen, N, C, dtype=dt), dy=_randn(gen, N, C, dtype=dt),
              dh=_randn(gen, N, C, dtype=dt))
    for key in ("shift", "scale", "gate"):
        st[key] = _randn(gen, C, std=0.5, dtype=dt)
    new = lambda *shape: torch.empty(*shape, dtype=dt, device=DEV)
    for key in ("h", "sum", "dx", "dout", "res"):
        st["o_" + key] = new(N, C)
    if case["act"] == "swiglu":
        # gate and up are column slices of the fused projection's rows, the
        # activation goes into its slice of the out projection's input
        st["fused"] = _randn(gen, N, 3 * C + 2 * M, dtype=dt)
        st["djoined"] = _randn(gen, N, C + M, dtype=dt)
        st["joined"], st["dfused"] = new(N, C + M).zero_(), new(N, 3 * C + 2 * M).zero_()
    else:
        st["pre"], st["dact"] = _randn(gen, N, M, dtype=dt), _randn(gen, N, M, dtype=dt)
        st["o_act"], st["o_dpre"] = new(N, M), new(N, M)
    return st


def _lora_factors(w, gen, shapes, rank, dt):
    for t, (fin, fout) in shapes.items():
        w.lora_a[t] = _randn(gen, rank, fin, std=1.0 / rank, dtype=dt)
        w.lora_b[t] = _randn(gen, fout, rank, std=1e-3, dtype=dt)


def _block_weights(case, gen):
    """Random-init weights of the block and the conditioning vector."""
    dt = DTYPES[case["dtype"]]
    D = case["head_dim"]
    C = case["heads"] * D
    rn = lambda *shape: _randn(gen, *shape, std=0.02, dtype=dt)
    norm = lambda: _randn(gen, D, std=0.02).add_(1).to(dt)
    if case["kind"] == "double":
        ws = {}
        for s in STREAMS:
            ws[s] = fb.StreamWeights(w_qkv=rn(3 * C, C), w_out=rn(C, C), w1=rn(4 * C, C), w2=rn(C, 4 * C),
                                     q_norm=norm(), k_norm=norm(), w_mod=rn(6 * C, C))
            _lora_factors(ws[s], gen, {t: (C, C) for t in fb.LORA_TARGETS}, case["rank"], dt)
    else:
        M = 3 * C
        ws = fb.SingleWeights(w_in=rn(3 * C + 2 * M, C), w_out=rn(C, C + M), q_norm=norm(), k_norm=norm(),
                              w_mod=rn(3 * C, C))
        _lora_factors(ws, gen, {"to_in": (C, 3 * C + 2 * M), "to_out": (C + M, C)}, case["rank"], dt)
    return ws, _randn(gen, C, dtype=dt)


def _prepare_block(case, gen):
    dt = DTYPES[case["dtype"]]
    H, D, T, I = case["heads"], case["head_dim"], case["txt"], case["rows"] * case["cols"]
    ws, c = _block_weights(case, gen)
    args = (ws, H, D, T, case["rows"], case["cols"])
    if case["kind"] == "double":
        n = {"txt": T, "img": I}
        x = {s: _randn(gen, n[s], H * D, dtype=dt) for s in STREAMS}
        dy = {s: _randn(gen, n[s], H * D, dtype=dt) for s in STREAMS}
        blk = fb.DoubleBlockLoRA(*args, axes=AXES3, theta=THETA3, lora_scale=1.0)
    else:
        x, dy = _randn(gen, T + I, H * D, dtype=dt), _randn(gen, T + I, H * D, dtype=dt)
        blk = fb.SingleBlockLoRA(*args, axes=AXES4, theta=THETA4, lora_scale=1.0)
    blk.set_conditioning(c)
    return dict(block=blk, x=x, dy=dy)


_PREPARE = {"attention": _prepare_attention, "prologue": _prepare_prologue, "lora": _prepare_lora,
            "mlp": _prepare_mlp, "double": _prepare_block, "single": _prepare_block}


def prepare(case, seed):
    st = _PREPARE[case["kind"]](case, _generator(seed))
    st["case"] = case
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _run_attention(st):
    q, k, v, do = st["q"], st["k"], st["v"], st["do"]
    if st["case"]["api"] == "autograd":
        o = fa.attention(q, k, v, key_keep=st["keep"])
        dq, dk, dv = torch.autograd.grad(o, (q, k, v), do)
        return dict(o=o.detach(), dq=dq, dk=dk, dv=dv)
    o, lse = fa.attn_fwd(q, k, v, key_keep=st["keep"])
    dq, dk, dv = fa.attn_bwd(q, k, v, o, do, lse, key_keep=st["keep"])
    return dict(o=o, lse=lse, dq=dq, dk=dk, dv=dv)


def _run_prologue(st):
    fa.qk_prologue_multi(st["fwd"], EPS)
    fa.qk_prologue_bwd_multi(st["bwd"], EPS)
    return dict(q=st["q"], k=st["k"], dqkv=st["dqkv"])


def _run_lora(st):
    # y and dx arrive holding the frozen linear's own products, which the
    # adapter adds to in place: the copies put them there for each pass
    st["y"].copy_(st["base"])
    u = fa.lora_fwd(st["x"], st["a"], st["b"], st["y"], st["scale"])
    dx = st.get("dx")
    if dx is not None:
        dx.copy_(st["dbase"])
    da, db = fa.lora_bwd(st["x"], st["a"], st["b"], u, st["dy"], st["scale"], dx=dx)
    out = dict(y=st["y"], u=u, da=da, db=db)
    if dx is not None:
        out["dx"] = dx
    return out


def _run_mlp(st):
    case = st["case"]
    C = case["width"]
    M = case["ratio"] * C
    x, sh, sc, g = st["x"], st["shift"], st["scale"], st["gate"]
    if case["act"] == "swiglu":
        h, mean, rstd = fb.ln_mod_fwd(x, sh, sc, EPS, out=st["o_h"], stats=True)
        gate, up = st["fused"][:, 3 * C:3 * C + M], st["fused"][:, 3 * C + M:]
        fb.swiglu(gate, up, out=st["joined"][:, C:])
        res = fb.gated_residual(x, g, st["out"], out=st["o_res"])
        dout = fb.gated_residual(None, g, st["dy"], out=st["o_dout"])
        fb.swiglu_bwd(st["djoined"][:, C:], gate, up, dgate=st["dfused"][:, 3 * C:3 * C + M],
                      dup=st["dfused"][:, 3 * C + M:])
        dx = fb.ln_mod_bwd(x, st["dh"], sc, mean, rstd, EPS, dres=st["dy"], out=st["o_dx"])
        return dict(h=h, res=res, dout=dout, dx=dx, joined=st["joined"], dfused=st["dfused"], mean=mean, rstd=rstd)
    s, h, mean, rstd = fb.gated_ln_mod_fwd(x, g, st["out"], sh, sc, EPS, out=st["o_h"], sum_out=st["o_sum"])
    act = fb.gelu(st["pre"], out=st["o_act"])
    dpre = fb.gelu_bwd(st["dact"], st["pre"], out=st["o_dpre"])
    dx, dout = fb.ln_mod_bwd_gate(s, st["dh"], sc, mean, rstd, g, EPS, dres=st["dy"], out=st["o_dx"],
                                  gated_out=st["o_dout"])
    return dict(s=s, h=h, mean=mean, rstd=rstd, act=act, dpre=dpre, dx=dx, dout=dout)


def _run_double(st):
    y, grads = st["block"].forward_backward(st["x"], st["dy"], want_dx=True)
    out = {"y." + s: y[s] for s in STREAMS}
    for s in STREAMS:
        out["dx." + s] = grads[(s, "x")]
        for t in fb.LORA_TARGETS:
            out[f"da.{s}.{t}"], out[f"db.{s}.{t}"] = grads[(s, t)]
    return out


def _run_single(st):
    y, grads = st["block"].forward_backward(st["x"], st["dy"], want_dx=True)
    out = dict(y=y, dx=grads["x"])
    for t in fb.SINGLE_LORA_TARGETS:
        out["da." + t], out["db." + t] = grads[t]
    return out


_RUN = {"attention": _run_attention, "prologue": _run_prologue, "lora": _run_lora, "mlp": _run_mlp,
        "double": _run_double, "single": _run_single}


def run(state):
    return _RUN[state["case"]["kind"]](state)


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how far correct results may differ
# ---------------------------------------------------------------------------
def work(case):
    e = 2 if case["dtype"] == "bf16" else 4
    kind = case["kind"]
    if kind == "attention":
        n = case["batch"] * case["seq"] * case["heads"] * case["head_dim"]
        # q, k, v, do read; o, dq, dk, dv written
        return dict(bytes=8.0 * n * e, flops=_attention_flops(case))
    if kind == "prologue":
        n = 2.0 * (case["txt"] + case["rows"] * case["cols"]) * case["heads"] * case["head_dim"]
        # forward: x read, y written; backward: x and dy read, dx written
        return dict(bytes=5.0 * n * e, flops=30.0 * n)
    if kind == "lora":
        N, K, M, r = case["tokens"], case["fin"], case["fout"], case["rank"]
        rows = N * (K + 3.0 * M + (2.0 * K if case["dx"] else 0.0)) * e  # x, dy, y twice, dx twice
        fac = r * (K + M) * (e + 4.0) + 4.0 * N * r
        return dict(bytes=rows + fac, flops=2.0 * N * r * (2 * K + 3 * M + (K if case["dx"] else 0)))
    if kind == "mlp":
        N, C, M = case["tokens"], case["width"], case["ratio"] * case["width"]
        if case["act"] == "swiglu":
            # x, out, dy, dh and gate, up, dact read; h, res, dout, dx, act, dgate, dup written
            return dict(bytes=float(N) * (8 * C + 6 * M) * e, flops=float(N) * (40 * C + 40 * M))
        return dict(bytes=float(N) * (8 * C + 4 * M) * e, flops=float(N) * (40 * C + 40 * M))
    C = case["heads"] * case["head_dim"]
    S, r = case["txt"] + case["rows"] * case["cols"], case["rank"]
    attn = 14.0 * S * S * C
    if kind == "double":
        linears, factors, streams = 12.0 * C * C, 8.0 * C * r, 2
    else:
        linears, factors, streams = 9.0 * C * C + 4.0 * C * C, (1 + 9 + 4 + 1) * C * float(r), 1
    # every frozen linear once forward and once for its input gradient; each
    # adapter factor three products (forward, gradient, input gradient)
    flops = 4.0 * S * linears + 6.0 * S * factors + attn
    return dict(bytes=streams * (linears * e + factors * (e + 4)) + 4.0 * S * C * e, flops=flops)


def tolerance(case):
    return _TOLERANCE[(case["kind"], case["dtype"])]


# Four times the 2-norm errors that passes show against exact(): bf16 results
# 1.7e-3 to 2.7e-3 (one rounding), f32 sums up to 2.2e-6 (1536 keys), the
# blocks up to 1.2e-2 (double: the gradients of the q and k factors, whose
# scores have a standard deviation near 11) and 6e-3 (single).
_TOLERANCE = {
    ("attention", "bf16"): {"rel": 1e-2},
    ("attention", "f32"): {"rel": 1e-5},
    ("prologue", "bf16"): {"rel": 1e-2},
    ("prologue", "f32"): {"rel": 1e-5},
    ("lora", "bf16"): {"rel": 1e-2},
    ("lora", "f32"): {"rel": 1e-5},
    ("mlp", "bf16"): {"rel": 1e-2},
    ("mlp", "f32"): {"rel": 1e-5},
    ("double", "bf16"): {"rel": 4e-2},
    ("single", "bf16"): {"rel": 2.5e-2},
}


# ---------------------------------------------------------------------------
# the same results in 64 bits, by plain torch
# ---------------------------------------------------------------------------
def _attention64(q, k, v, keep, do=None):
    """q, k, v, do [S, D] of one head: o, lse and, with do, dq, dk, dv."""
    scale = 1.0 / math.sqrt(q.shape[1])
    s = q @ k.t() * scale
    if keep is not None:
        s.masked_fill_(~keep[None, :], -math.inf)
    lse = torch.logsumexp(s, 1)
    p = s.sub_(lse[:, None]).exp_()
    o = p @ v
    if do is None:
        return o, lse
    dv = p.t() @ do
    dp = do @ v.t()
    ds = dp.sub_((do * o).sum(1, keepdim=True)).mul_(p).mul_(scale)
    return o, lse, ds @ k, ds.t() @ q, dv


class _JointAttention64(torch.autograd.Function):
    """[S, H, D] attention in 64 bits, one head at a time."""

    @staticmethod
    def forward(ctx, q, k, v):
        ctx.save_for_backward(q, k, v)
        return torch.stack([_attention64(q[:, h], k[:, h], v[:, h], None)[0] for h in range(q.shape[1])], 1)

    @staticmethod
    def backward(ctx, do):
        q, k, v = ctx.saved_tensors
        g = [_attention64(q[:, h], k[:, h], v[:, h], None, do[:, h])[2:] for h in range(q.shape[1])]
        return tuple(torch.stack([gh[i] for gh in g], 1) for i in range(3))


def _rope_tables64(pos, axes, theta):
    cols = []
    for a, d in enumerate(axes):
        inv = theta ** (-torch.arange(0, d, 2, dtype=torch.float64) / d)
        f = torch.as_tensor(pos[:, a], dtype=torch.float64)[:, None] * inv
        cols.append(torch.cat([f, f], 1))
    f = torch.cat(cols, 1).to(DEV)
    return f.cos(), f.sin()


def _rotate64(x, cos, sin, axes):
    parts, o = [], 0
    for d in axes:
        a, b = x[..., o:o + d // 2], x[..., o + d // 2:o + d]
        parts += [-b, a]
        o += d
    return x * cos[:, None] + torch.cat(parts, -1) * sin[:, None]


def _qk64(x, w, cos, sin, axes):
    n = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w
    return _rotate64(n, cos, sin, axes)


def _ln_mod64(x, shift, scale):
    d = x - x.mean(1, keepdim=True)
    return d * torch.rsqrt(d.square().mean(1, keepdim=True) + EPS) * (1 + scale) + shift


def _gelu64(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _silu64(x):
    return x * torch.sigmoid(x)


def _exact_attention(case, st):
    B, H = case["batch"], case["heads"]
    names = ("o", "dq", "dk", "dv")
    out = {n: torch.empty(st["q"].shape, dtype=torch.float64, device=DEV) for n in names}
    lse = torch.empty(B, H, case["seq"], dtype=torch.float64, device=DEV)
    for b in range(B):
        keep = None if st["keep"] is None else st["keep"][b].bool()
        for h in range(H):
            q, k, v, do = (st[t][b, :, h].detach().double() for t in ("q", "k", "v", "do"))
            o, l, dq, dk, dv = _attention64(q, k, v, keep, do)
            for n, t in zip(names, (o, dq, dk, dv)):
                out[n][b, :, h] = t
            lse[b, h] = l
    if case["api"] == "op":
        out = dict(o=out["o"], lse=lse, dq=out["dq"], dk=out["dk"], dv=out["dv"])
    return out


def _exact_prologue(case, st):
    H, D, T = case["heads"], case["head_dim"], case["txt"]
    C, S = H * D, case["txt"] + case["rows"] * case["cols"]
    out = dict(q=torch.empty(1, S, H, D, dtype=torch.float64, device=DEV),
               k=torch.empty(1, S, H, D, dtype=torch.float64, device=DEV),
               dqkv=torch.zeros(S, 3 * C, dtype=torch.float64, device=DEV))
    for s, sl in (("txt", slice(0, T)), ("img", slice(T, S))):
        cos, sin = (t.double() for t in st["rope"][s])
        for j, t in enumerate("qk"):
            cols = slice(j * C, (j + 1) * C)
            x = st["qkv"][sl, cols].double().reshape(-1, H, D).requires_grad_(True)
            y = _qk64(x, st["norm"][s + t].double(), cos, sin, AXES3)
            (dx,) = torch.autograd.grad(y, x, st["d" + t][0, sl].double())
            out[t][0, sl] = y.detach()
            out["dqkv"][sl, cols] = dx.reshape(-1, C)
    return out


def _exact_lora(case, st):
    d = {k: st[k].double() for k in ("x", "a", "b", "base", "dy")}
    s = st["scale"]
    u = d["x"] @ d["a"].t()
    du = s * (d["dy"] @ d["b"])
    out = dict(y=d["base"] + s * (u @ d["b"].t()), u=u, da=du.t() @ d["x"], db=s * (d["dy"].t() @ u))
    if case["dx"]:
        out["dx"] = st["dbase"].double() + du @ d["a"]
    return out


def _exact_mlp(case, st):
    C = case["width"]
    M = case["ratio"] * C
    d = {k: v.double() for k, v in st.items() if torch.is_tensor(v) and not k.startswith("o_")}
    x, g = d["x"], d["gate"]
    s = x if case["act"] == "swiglu" else x + g * d["out"]
    xs = s.clone().requires_grad_(True)
    h = _ln_mod64(xs, d["shift"], d["scale"])
    (dln,) = torch.autograd.grad(h, xs, d["dh"])
    dx = d["dy"] + dln
    mean = s.mean(1)
    rstd = torch.rsqrt((s - mean[:, None]).square().mean(1) + EPS)
    h = h.detach()
    if case["act"] == "swiglu":
        gate = d["fused"][:, 3 * C:3 * C + M].clone().requires_grad_(True)
        up = d["fused"][:, 3 * C + M:].clone().requires_grad_(True)
        act = _silu64(gate) * up
        dgate, dup = torch.autograd.grad(act, (gate, up), d["djoined"][:, C:])
        zero = torch.zeros(x.shape[0], 3 * C, dtype=torch.float64, device=DEV)
        return dict(h=h, res=x + g * d["out"], dout=g * d["dy"], dx=dx, joined=torch.cat([zero[:, :C], act.detach()], 1),
                    dfused=torch.cat([zero, dgate, dup], 1), mean=mean, rstd=rstd)
    pre = d["pre"].clone().requires_grad_(True)
    act = _gelu64(pre)
    (dpre,) = torch.autograd.grad(act, pre, d["dact"])
    return dict(s=s, h=h, mean=mean, rstd=rstd, act=act.detach(), dpre=dpre, dx=dx, dout=g * dx)


def _lora_linear64(x, w, a, b):
    return x @ w.t() + (x @ a.t()) @ b.t()


def _exact_double(case, st):
    blk, H, D, T = st["block"], case["heads"], case["head_dim"], case["txt"]
    C = H * D
    ws, c = _block_weights(case, _generator(st["seed"]))
    cos, sin = _rope_tables64(_positions(T, case["rows"], case["cols"]), AXES3, THETA3)
    part = {"txt": slice(0, T), "img": slice(T, T + case["rows"] * case["cols"])}
    x = {s: st["x"][s].double().requires_grad_(True) for s in STREAMS}
    leaf = {(s, t, f): getattr(ws[s], "lora_" + f)[t].double().requires_grad_(True)
            for s in STREAMS for t in fb.LORA_TARGETS for f in "ab"}
    mod, qkv = {}, {t: [] for t in "qkv"}
    for s in STREAMS:
        w = ws[s]
        mod[s] = (_silu64(c.double()) @ w.w_mod.double().t()).split(C)
        h = _ln_mod64(x[s], mod[s][0], mod[s][1])
        for j, t in enumerate("qkv"):
            z = _lora_linear64(h, w.w_qkv[j * C:(j + 1) * C].double(), leaf[s, t, "a"], leaf[s, t, "b"])
            z = z.reshape(-1, H, D)
            if t != "v":
                norm = w.q_norm if t == "q" else w.k_norm
                z = _qk64(z, norm.double(), cos[part[s]], sin[part[s]], AXES3)
            qkv[t].append(z)
    o = _JointAttention64.apply(*(torch.cat(qkv[t]) for t in "qkv")).reshape(-1, C)
    y = {}
    for s in STREAMS:
        w, m = ws[s], mod[s]
        x1 = x[s] + m[2] * _lora_linear64(o[part[s]], w.w_out.double(), leaf[s, "out", "a"], leaf[s, "out", "b"])
        act = _gelu64(_ln_mod64(x1, m[3], m[4]) @ w.w1.double().t())
        y[s] = x1 + m[5] * (act @ w.w2.double().t())
    wrt = [x[s] for s in STREAMS] + list(leaf.values())
    grads = torch.autograd.grad([y[s] for s in STREAMS], wrt, [st["dy"][s].double() for s in STREAMS])
    by = dict(zip(leaf, grads[2:]))
    out = {"y." + s: y[s].detach() for s in STREAMS}
    for i, s in enumerate(STREAMS):
        out["dx." + s] = grads[i]
        for t in fb.LORA_TARGETS:
            out[f"da.{s}.{t}"], out[f"db.{s}.{t}"] = by[s, t, "a"], by[s, t, "b"]
    return out


def _exact_single(case, st):
    H, D, T = case["heads"], case["head_dim"], case["txt"]
    C = H * D
    M = 3 * C
    w, c = _block_weights(case, _generator(st["seed"]))
    pos = fb.klein_positions(T, case["rows"], case["cols"])
    cos, sin = _rope_tables64(pos, AXES4, THETA4)
    x = st["x"].double().requires_grad_(True)
    leaf = {(t, f): getattr(w, "lora_" + f)[t].double().requires_grad_(True)
            for t in fb.SINGLE_LORA_TARGETS for f in "ab"}
    sh, sc, g = (_silu64(c.double()) @ w.w_mod.double().t()).split(C)
    z = _lora_linear64(_ln_mod64(x, sh, sc), w.w_in.double(), leaf["to_in", "a"], leaf["to_in", "b"])
    q, k, v = (z[:, j * C:(j + 1) * C].reshape(-1, H, D) for j in range(3))
    q = _qk64(q, w.q_norm.double(), cos, sin, AXES4)
    k = _qk64(k, w.k_norm.double(), cos, sin, AXES4)
    o = _JointAttention64.apply(q, k, v).reshape(-1, C)
    joined = torch.cat([o, _silu64(z[:, 3 * C:3 * C + M]) * z[:, 3 * C + M:]], 1)
    y = x + g * _lora_linear64(joined, w.w_out.double(), leaf["to_out", "a"], leaf["to_out", "b"])
    grads = torch.autograd.grad(y, [x] + list(leaf.values()), st["dy"].double())
    by = dict(zip(leaf, grads[1:]))
    out = dict(y=y.detach(), dx=grads[0])
    for t in fb.SINGLE_LORA_TARGETS:
        out["da." + t], out["db." + t] = by[t, "a"], by[t, "b"]
    return out


_EXACT = {"attention": _exact_attention, "prologue": _exact_prologue, "lora": _exact_lora, "mlp": _exact_mlp,
          "double": _exact_double, "single": _exact_single}


def exact(case, seed):
    st = prepare(case, seed)
    st["seed"] = seed
    return _EXACT[case["kind"]](case, st)
