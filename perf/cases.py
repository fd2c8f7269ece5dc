"""The calls a user of this library makes, as cases that can be timed and compared: every attention path of
include/lr_attn.h through the torch-facing entry points (localrouter_amd.ops, localrouter_amd.mmdit), over the sizes of
the engines' own calls, the repository's workloads and tests.

  listed()             the named cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  the inputs and what a program keeps between calls (tables, output and workspace buffers)
  run(state)           one pass; returns its outputs
  work(case)           the bytes and floating-point operations the pass cannot do without
  tolerance(case)      how far another correct implementation at the same precision may be off
  exact(case, seed)    the outputs in 64 bits, from plain torch
"""
from __future__ import annotations

import math

import numpy as np
import torch

from localrouter_amd import mmdit, ops, rope_host

D = 128
EPS = 1e-6                       # QK-RMSNorm epsilon of the joint calls
H3_EPS, H3_ROT = 1e-5, 96        # MiniMax H3's rmsRope
THETA = 10000.0


# ---------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest fused call in use: a 256 x 256 preview of a small model (64 text + 16 x 16 image tokens, 4 heads)
        dict(name="joint-320x4", kind="joint", text=64, gh=16, gw=16, frames=1, heads=4, kv_heads=4, prefix=0),
        # a 512 x 512 image step: 256 text + 32 x 32 image tokens, 24 heads
        dict(name="joint-1280x24", kind="joint", text=256, gh=32, gw=32, frames=1, heads=24, kv_heads=24, prefix=0),
        # the 1024 x 1024 image step: 512 text + 64 x 64 image tokens, 24 heads
        dict(name="joint-4608x24", kind="joint", text=512, gh=64, gw=64, frames=1, heads=24, kv_heads=24, prefix=0),
        # an image edit: 512 text + the target and two reference latents of 64 x 64 tokens
        dict(name="joint-edit-12800x24", kind="joint", text=512, gh=64, gw=64, frames=3, heads=24, kv_heads=24,
             prefix=0),
        # an engine that binds the launches one by one (rope of q, rope of k behind the cached text prefix, value rows
        # copied behind it, attention): a 512 x 512 step of Qwen-Image 2.1, 32 x 32 image queries over 80 + 1,024 keys
        dict(name="launches-1024x1104x32", kind="launches", prefix=80, gh=32, gw=32, heads=32),
        # a text encoder's causal prefill chunk, 32 query heads over 8 key heads, 77 positions already cached
        dict(name="causal-1500x32g8", kind="rows", queries=1500, keys=1577, heads=32, kv_heads=8, causal=1, p0=77),
        # Kandinsky-6: 218 audio queries over the 50,220 video tokens
        dict(name="audio-from-video-218x50220", kind="ws", queries=218, keys=50220, heads=16, kv_heads=16),
        # Kandinsky-6: the visual self-attention, the largest call (50,220 tokens x 32 heads)
        dict(name="visual-self-50220x32", kind="ws", queries=50220, keys=50220, heads=32, kv_heads=32),
        # Kandinsky-6: cross-attention to padded text, 700 of 1,024 text keys kept
        dict(name="kmask-3000x1024x32", kind="kmask", queries=3000, keys=1024, valid=700, heads=32),
        # MiniMax H3: rmsRope + INT8 prep, then the INT8 attention, at its headline length
        dict(name="int8-5967x56", kind="int8", tokens=5967, heads=56),
        # the INT8 attention at head dim 64, the shape of the reference's own gate
        dict(name="int8-d64-1797x32", kind="int8_64", tokens=1797, heads=32),
        # a whole MMDiT double-stream block: 512 text + 4,096 image rows, hidden 3072, MLP 12288
        dict(name="mmdit-512+4096", kind="mmdit", text=512, image=4096, hidden=3072, mlp=12288),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["joint", "joint", "joint", "launches", "rows", "rows", "ws", "kmask", "int8", "int8_64", "mmdit"])
    if kind == "joint":
        frames = rng.choice([1, 1, 1, 2, 3])
        gh, gw = _log_int(rng, 12, 64), _log_int(rng, 12, 64)
        kv = rng.choice([1, 1, 1, 2, 4])           # query heads per key head
        heads = rng.choice([4, 12, 16, 24, 32])
        text = _log_int(rng, 16, 600)
        # a cached text prefix is for the keys of a single image's step
        prefix = text if frames == 1 and rng.random() < 0.3 else 0
        return dict(kind="joint", text=text, gh=gh, gw=gw, frames=frames, heads=heads, kv_heads=heads // kv,
                    prefix=prefix)
    if kind == "launches":
        return dict(kind="launches", prefix=_log_int(rng, 16, 512), gh=_log_int(rng, 12, 64), gw=_log_int(rng, 12, 64),
                    heads=rng.choice([16, 24, 32]))
    if kind == "rows":
        w = _log_int(rng, 32, 4608)
        p0 = rng.choice([0, 0, 77, _log_int(rng, 1, 2000)])
        heads = rng.choice([16, 24, 32])
        if rng.random() < 0.6:
            return dict(kind="rows", queries=w, keys=w + p0, heads=heads, kv_heads=heads // rng.choice([1, 4]),
                        causal=1, p0=p0)
        return dict(kind="rows", queries=w, keys=_log_int(rng, 64, 6000), heads=heads, kv_heads=heads, causal=0, p0=0)
    if kind == "ws":
        q, k = _log_int(rng, 100, 24000), _log_int(rng, 200, 50220)
        heads = rng.choice([16, 24, 32])
        return dict(kind="ws", queries=q, keys=k, heads=heads, kv_heads=heads)
    if kind == "kmask":
        k = _log_int(rng, 64, 4000)
        return dict(kind="kmask", queries=_log_int(rng, 100, 12000), keys=k, valid=max(1, int(k * rng.uniform(0.2, 1))),
                    heads=rng.choice([16, 32]))
    if kind == "int8":
        return dict(kind="int8", tokens=_log_int(rng, 200, 13000), heads=rng.choice([24, 40, 56]))
    if kind == "int8_64":
        return dict(kind="int8_64", tokens=_log_int(rng, 80, 6000), heads=rng.choice([16, 32, 56]))
    return dict(kind="mmdit", text=_log_int(rng, 32, 1024), image=_log_int(rng, 256, 4500), hidden=3072, mlp=12288)


# --------------------------------------------------------------------------------------------------- the inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _bf(g, *shape):
    return _randn(g, *shape).to(torch.bfloat16)


def _weight(g):
    """A trained norm weight: around 1."""
    return 1.0 + 0.1 * _randn(g, D)


def _grid_table(text, gh, gw, frames):
    """cos / sin [rows, 64] of the text rows, then the frames' image rows (frames > 1: the edit table)."""
    if frames > 1:
        cos, sin = rope_host.edit_table(text, frames, gh, gw)
    else:
        cos, sin = rope_host.grid2d_table(text, gh, gw, THETA)
    return torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()


def _h3_table(tokens):
    """H3's bf16 table [tokens, 192] ([48 pairs][2][2]): 16 frequencies on each of three axes, of a text + video
    layout's positions, repeated to the number of tokens."""
    pos = rope_host.h3_positions(24, 3, 8, 12, 15)
    inv = (1.0 / np.power(THETA, np.arange(16) / 16.0)).astype(np.float32)
    tab = torch.from_numpy(rope_host.h3_rope_table(pos, inv).reshape(-1, 192).view(np.int16)).view(torch.bfloat16)
    return tab.repeat(-(-tokens // tab.shape[0]), 1)[:tokens].contiguous().cuda()


def _sizes(case):
    """(queries, keys) of an attention case."""
    kind = case["kind"]
    if kind == "joint":
        img = case["gh"] * case["gw"] * case["frames"]
        return (img, case["prefix"] + img) if case["prefix"] else (case["text"] + img,) * 2
    if kind == "launches":
        img = case["gh"] * case["gw"]
        return img, case["prefix"] + img
    if kind in ("rows", "ws"):
        return case["queries"], case["keys"]
    if kind == "kmask":
        return case["queries"], case["valid"]
    return case["tokens"], case["tokens"]


def _inputs(case, seed):
    """The tensors that come from the seed."""
    g, kind = _gen(seed), case["kind"]
    x = {}
    if kind in ("joint", "launches"):
        sq, sk = _sizes(case)
        h, hk = case["heads"], case.get("kv_heads", case["heads"])
        n_pre = case["prefix"]
        x["q"], x["k"], x["v"] = _bf(g, sq, h, D), _bf(g, sk - n_pre, hk, D), _bf(g, sk, hk, D)
        x["q_norm"], x["k_norm"] = _weight(g), _weight(g)
        # the cached prefix: normalised, rotated keys
        x["k_pre"] = _bf(g, n_pre, hk, D)
        cos, sin = _grid_table(0 if n_pre else case["text"], case["gh"], case["gw"], case.get("frames", 1))
        x["cos"], x["sin"] = cos, sin
    elif kind in ("rows", "ws", "kmask"):
        w, sk = case["queries"], case["keys"]
        h, hk = case["heads"], case.get("kv_heads", case["heads"])
        x["q"], x["k"], x["v"] = _bf(g, w, h, D), _bf(g, sk, hk, D), _bf(g, sk, hk, D)
        if kind == "kmask":
            keep = torch.randperm(sk, generator=g, device="cuda")[:case["valid"]]
            x["mask"] = torch.zeros(sk, dtype=torch.uint8, device="cuda")
            x["mask"][keep] = 1
    elif kind == "int8":
        s, h = case["tokens"], case["heads"]
        x["qkv"] = _bf(g, s, 3 * h * D)
        x["q_norm"], x["k_norm"] = _weight(g).to(torch.bfloat16), _weight(g).to(torch.bfloat16)
        x["freqs"] = _h3_table(s)
    elif kind == "int8_64":
        s, h = case["tokens"], case["heads"]
        x["q"], x["k"], x["v"] = (_bf(g, 1, h, s, 64) for _ in range(3))
    else:
        d = case["hidden"]
        x["txt"], x["img"] = _bf(g, case["text"], d), _bf(g, case["image"], d)
        x["t"] = torch.rand(1, generator=g, device="cuda")
        x["weights"] = mmdit.make_weights(d, case["mlp"], torch.device("cuda", torch.cuda.current_device()), seed=seed)
        pos = torch.arange(case["text"] + case["image"], device="cuda", dtype=torch.float64)
        pos = (pos - case["text"]).clamp(min=0)      # text rows un-rotated
        ang = pos[:, None] * torch.pow(THETA, -torch.arange(64, device="cuda", dtype=torch.float64) / 64)
        x["cos"], x["sin"] = ang.cos().float(), ang.sin().float()
    return x


def prepare(case, seed):
    s = dict(case=case, **_inputs(case, seed))
    kind = case["kind"]
    if kind == "joint":
        sq, sk = _sizes(case)
        if case["prefix"]:           # the key buffer of a step: the cached prefix in front of the step's raw keys
            s["k"] = torch.cat([s["k_pre"], s["k"]])
        s["out"] = torch.empty((sq, case["heads"], D), dtype=torch.bfloat16, device="cuda")
        s["ws"] = torch.empty(ops.workspace_bytes(sk, case["kv_heads"]), dtype=torch.uint8, device="cuda")
    elif kind == "launches":
        sq, sk = _sizes(case)
        h, p = case["heads"], case["prefix"]
        # the step's key and value buffers hold the cached prefix; each step writes behind it
        s["kbuf"], s["vbuf"] = (torch.empty((sk, h, D), dtype=torch.bfloat16, device="cuda") for _ in range(2))
        s["kbuf"][:p], s["vbuf"][:p] = s["k_pre"], s["v"][:p]
        s["v_img"] = s["v"][p:].contiguous()
        s["qbuf"], s["out"] = (torch.empty((sq, h, D), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    elif kind in ("rows", "ws", "kmask"):
        s["out"] = torch.empty((case["queries"], case["heads"], D), dtype=torch.bfloat16, device="cuda")
        if kind == "ws":
            n = ops.attention_ws_bytes(case["queries"], case["heads"], case["keys"])
        elif kind == "kmask":
            n = int(ops._lib.load().lr_attention_kmask_workspace_bytes(case["valid"], case["heads"]))
        else:
            n = 0
        s["ws"] = torch.empty(n, dtype=torch.uint8, device="cuda") if n else None
    elif kind == "int8":
        t, h = case["tokens"], case["heads"]
        s["out"] = torch.empty((t, h * D), dtype=torch.bfloat16, device="cuda")
        s["ws"] = torch.empty(ops.int8_workspace_bytes(h, t), dtype=torch.uint8, device="cuda")
    elif kind == "int8_64":
        t, h = case["tokens"], case["heads"]
        s["out"] = torch.empty((1, h, t, 64), dtype=torch.bfloat16, device="cuda")
        s["ws"] = torch.empty(ops.int8_workspace_bytes(h, t, head_dim=64), dtype=torch.uint8, device="cuda")
    else:
        s["block"] = mmdit.MMDiTBlock(s["weights"])
        s["block"].workspace(case["text"], case["image"])
        s["block"].plan(case["text"], case["image"])
        s["x_txt"], s["x_img"] = torch.empty_like(s["txt"]), torch.empty_like(s["img"])
    return s


# ------------------------------------------------------------------------------------------------------ one pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "joint":
        return ops.joint_attention(s["q"], s["k"], s["v"], s["out"], q_norm=s["q_norm"], k_norm=s["k_norm"],
                                   q_table=(s["cos"], s["sin"]), n_pre=case["prefix"], workspace=s["ws"])
    if kind == "launches":
        h, p = case["heads"], case["prefix"]
        n, rs = s["q"].shape[0], h * D
        tab = dict(n=n, heads=h, src_row_stride=rs, dst_row_stride=rs, table_a=s["cos"], table_b=s["sin"])
        ops.rms_rope(s["q"], s["qbuf"], s["q_norm"], **tab)
        ops.rms_rope(s["k"], s["kbuf"][p:], s["k_norm"], **tab)
        s["vbuf"][p:].copy_(s["v_img"])
        return ops.attention(s["qbuf"], s["kbuf"], s["vbuf"], s["out"])
    if kind == "rows":
        return ops.attention(s["q"], s["k"], s["v"], s["out"], causal=bool(case["causal"]), p0=case["p0"])
    if kind == "ws":
        return ops.attention_ws(s["q"], s["k"], s["v"], s["out"], workspace=s["ws"])
    if kind == "kmask":
        return ops.attention_kmask(s["q"], s["k"], s["v"], s["mask"], s["out"], n_valid=case["valid"],
                                   workspace=s["ws"])
    if kind == "int8":
        h = case["heads"]
        ops.kitchen_attention_prep_rope(s["qkv"], s["ws"], h, s["freqs"], s["q_norm"], s["k_norm"], rot=H3_ROT,
                                        eps=H3_EPS)
        return ops.kitchen_attention_kernel(s["out"], s["ws"], h, case["tokens"], True)
    if kind == "int8_64":
        return ops.int8_attention(s["q"], s["k"], s["v"], s["out"], workspace=s["ws"])
    # the block updates its rows in place: they are the step's hidden states, new in every step
    s["x_txt"].copy_(s["txt"])
    s["x_img"].copy_(s["img"])
    s["block"](s["x_txt"], s["x_img"], s["t"], s["cos"], s["sin"])
    return s["x_txt"], s["x_img"]


# ---------------------------------------------------------------------------------------------------- its work
def work(case):
    kind = case["kind"]
    if kind == "mmdit":
        d, f, st, si = case["hidden"], case["mlp"], case["text"], case["image"]
        rows = st + si
        flops = 2 * rows * (4 * d * d + 2 * d * f) + 4 * rows * rows * d + 2 * (256 * d + d * d + 12 * d * d)
        weights = 2 * (2 * (4 * d * d + 2 * d * f + 6 * d * d) + 256 * d + d * d)
        return {"bytes": weights + 2 * 2 * rows * d + 2 * rows * 64 * 4, "flops": flops}
    sq, sk = _sizes(case)
    h, hk = case["heads"], case.get("kv_heads", case["heads"])
    d = 64 if kind == "int8_64" else D
    pairs = sq * sk
    if kind == "rows" and case["causal"]:
        pairs = sum(min(sk, case["p0"] + i + 1) for i in range(sq))
    nbytes = 2 * d * (2 * sq * h + 2 * sk * hk)
    if kind in ("joint", "launches"):
        nbytes += 2 * 64 * 4 * (sk - case["prefix"])
    elif kind == "kmask":
        nbytes += case["keys"]
    elif kind == "int8":
        nbytes += 192 * 2 * sq
    return {"bytes": nbytes, "flops": 4 * pairs * d * h}


def tolerance(case):
    # measured against exact(): 2.3e-3 for bf16 attention (bf16 probabilities and outputs), 3.3e-3 with the norm and
    # rotation in front (bf16 queries and keys), 2.2e-3 for the block, 1.6e-2 / 1.4e-2 for INT8 at 128 / 64 dims. Two
    # implementations that round alike share the inputs' roundings (all of the int8 operands'), and differ by those of
    # the probabilities and of the output.
    if case["kind"] in ("int8", "int8_64"):
        return {"rel": 1e-2, "max": 0.3}
    if case["kind"] == "mmdit":
        return {"rel": 5e-3, "max": 0.1}
    return {"rel": 5e-3, "max": 0.1}


# --------------------------------------------------------------------------------------------- the same in 64 bits
def _norm_rope64(x, w, cos, sin):
    """[rows, heads, 128] in 64 bits: RMSNorm, then the interleaved pairs rotated."""
    x = x.double()
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()
    a, b = y[..., 0::2], y[..., 1::2]
    c, s = cos.double()[:, None, :], sin.double()[:, None, :]
    return torch.stack((c * a - s * b, s * a + c * b), -1).flatten(-2)


def _rms_rope_h3_64(x, w, tab):
    """[heads, rows, 128]: RMSNorm, then the split-half pairs (i, i + 48) of the first 96 dims by the table's matrices."""
    x = x.double()
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + H3_EPS) * w.double()
    m = tab.double().view(-1, H3_ROT // 2, 2, 2)
    a, b = y[..., :H3_ROT // 2], y[..., H3_ROT // 2:H3_ROT]
    r = torch.cat((m[:, :, 0, 0] * a + m[:, :, 0, 1] * b, m[:, :, 1, 0] * a + m[:, :, 1, 1] * b, y[..., H3_ROT:]), -1)
    return r


def _attention64(q, k, v, scale, causal=False, p0=0):
    """[rows, heads, d] in 64 bits (k, v: [keys, kv heads, d]), by blocks of query rows."""
    w, h = q.shape[0], q.shape[1]
    out = torch.empty((w, h, q.shape[2]), dtype=torch.float64, device=q.device)
    group = h // k.shape[1]
    step = max(64, min(w, (1 << 28) // max(1, k.shape[0])))
    for i in range(h):
        kh = k[:, i // group].double().t().contiguous()
        vh = v[:, i // group].double().contiguous()
        for r in range(0, w, step):
            s = (q[r:r + step, i].double() * scale) @ kh
            if causal:
                pos = p0 + torch.arange(r, min(w, r + step), device=q.device)
                s.masked_fill_(torch.arange(k.shape[0], device=q.device)[None, :] > pos[:, None], -math.inf)
            s -= s.amax(1, keepdim=True)
            s.exp_()
            out[r:r + step, i] = (s @ vh) / s.sum(1, keepdim=True)
    return out


def exact(case, seed):
    x, kind = _inputs(case, seed), case["kind"]
    if kind in ("joint", "launches"):
        p = case["prefix"]
        q = _norm_rope64(x["q"], x["q_norm"], x["cos"], x["sin"])
        k = torch.cat([x["k_pre"].double(), _norm_rope64(x["k"], x["k_norm"], x["cos"], x["sin"])])
        return _attention64(q, k, x["v"], D ** -0.5)
    if kind in ("rows", "ws"):
        return _attention64(x["q"], x["k"], x["v"], D ** -0.5, bool(case.get("causal")), case.get("p0", 0))
    if kind == "kmask":
        keep = x["mask"].nonzero()[:, 0]
        return _attention64(x["q"], x["k"][keep], x["v"][keep], D ** -0.5)
    if kind == "int8":
        q, k, v = ops.qkv_views(x["qkv"], case["heads"])
        q = _rms_rope_h3_64(q[0], x["q_norm"], x["freqs"]).transpose(0, 1)
        k = _rms_rope_h3_64(k[0], x["k_norm"], x["freqs"]).transpose(0, 1)
        return _attention64(q, k, v[0].transpose(0, 1), D ** -0.5).reshape(case["tokens"], -1)
    if kind == "int8_64":
        q, k, v = (t[0].transpose(0, 1) for t in (x["q"], x["k"], x["v"]))
        return _attention64(q, k, v, 64 ** -0.5).transpose(0, 1)[None].contiguous()
    return _block64(case, x)


def _block64(case, x):
    """The double-stream block of include/lr_mmdit.h in 64 bits."""
    w = {k: v.double() for k, v in x["weights"].items()}
    n_txt, d = case["text"], case["hidden"]
    heads = d // D
    t = (x["t"] * 1000).to(torch.bfloat16).float() * (1 / 1000)
    t = t.to(torch.bfloat16).double() * 1000         # the sinusoid's argument passes through bf16, by definition
    freq = torch.exp(-math.log(10000.0) * torch.arange(128, device=t.device, dtype=torch.float64) / 128)
    emb = torch.cat((torch.cos(t * freq), torch.sin(t * freq)))
    silu = torch.nn.functional.silu
    temb = silu(silu(emb @ w["t1"].t()) @ w["t2"].t())
    mod = {s: (temb @ w[f"{s}.mod"].t()).view(6, d) for s in ("txt", "img")}
    rows = {"txt": x["txt"].double(), "img": x["img"].double()}

    def norm(s, which):
        m = mod[s]
        return torch.nn.functional.layer_norm(rows[s], (d,), eps=1e-6) * (1 + m[3 * which + 1]) + m[3 * which]

    qkv = torch.cat([norm(s, 0) @ w[f"{s}.qkv"].t() for s in ("txt", "img")]).view(-1, 3, heads, D)
    q = _norm_rope64(qkv[:, 0], w["q_norm"], x["cos"], x["sin"])
    k = _norm_rope64(qkv[:, 1], w["k_norm"], x["cos"], x["sin"])
    att = _attention64(q, k, qkv[:, 2], D ** -0.5).reshape(-1, d)
    part = {"txt": att[:n_txt], "img": att[n_txt:]}
    for s in ("txt", "img"):
        rows[s] = rows[s] + mod[s][2] * (part[s] @ w[f"{s}.out"].t())
        h = torch.nn.functional.gelu(norm(s, 1) @ w[f"{s}.mlp_up"].t(), approximate="tanh")
        rows[s] = rows[s] + mod[s][5] * (h @ w[f"{s}.mlp_down"].t())
    return rows["txt"], rows["img"]
