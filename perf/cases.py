"""Performance cases of the framework: the device work of one image's generation (text encoder, DiT steps,
VAE decode), each piece through the entry points that a program calls, over the range of image sizes,
batch sizes, weight formats and precisions that such programs use.

A case is a plain dict: `kind` names the piece, the rest its sizes and options.

  block      one DiT block: self-attention, cross-attention and MLP sublayers (28 of these are a step)
  self       the self-attention sublayer: LayerNorm + adaLN, QKV projection, attention, output projection
  cross      the cross-attention sublayer against 512 prepared text tokens
  mlp        the MLP sublayer (2048 -> 8192 -> 2048, GELU)
  attn       the fused attention op alone (q/k RMSNorm + 3D RoPE + softmax(QK^T)V) on fp32 q/k/v
  text       the text encoder's layers (1024 wide, 16 / 8 heads, MLP 3072, bf16 weights), replayed from a graph
  vae_stage  a residual block of the VAE decoder, optionally followed by its 2x upsampling convolution
  vae_attn   the VAE decoder's single-head 384-dim spatial attention
  time_cond  the adaLN modulation vectors of all 28 blocks for one sigma, optionally with LoRAs

`hp`, `wp`: token grid of the DiT (image size / 16); `h`, `w`: the latent grid (image size / 8) or, for a
VAE stage, its input resolution.
"""

import importlib
import math

import numpy as np
import torch

anima = importlib.import_module("anima-studio_amd")

D, HEADS, HD, MLP, CTX, LK = 2048, 16, 128, 8192, 1024, 512
RANK_MOD, BLOCKS = 256, 28
TE_D, TE_H, TE_KH, TE_MLP, TE_THETA = 1024, 16, 8, 3072, 1e6
VAE_C = 384
CODEBOOK = [-0.980602, -0.794529, -0.638165, -0.500986, -0.377321, -0.263187, -0.155210, -0.050720,
            0.052541, 0.156985, 0.265284, 0.379533, 0.502636, 0.638953, 0.794876, 0.980671]
PRECISION = {"bf16": anima.PREC_BF16, "fp32": anima.PREC_FP32}


def listed():
    return [
        # a step of the default image, 1024 x 1024 with classifier-free guidance, is 28 of these
        {"name": "block_1024_cfg", "kind": "block", "b": 2, "hp": 64, "wp": 64, "weight": "w4", "kv_len": 0},
        # a draft at 512 x 512 without guidance: the smallest image in common use
        {"name": "block_512", "kind": "block", "b": 1, "hp": 32, "wp": 32, "weight": "w4", "kv_len": 0},
        # a portrait of 832 x 1216 with guidance: 52 x 76 tokens, not a multiple of 64; the first and
        # last blocks of a mixed checkpoint are int8
        {"name": "self_832x1216_cfg", "kind": "self", "b": 2, "hp": 52, "wp": 76, "weight": "i8", "lora": 0},
        # 768 x 768 with guidance, prompts shorter than the 512-token context masked
        {"name": "cross_768_cfg", "kind": "cross", "b": 2, "hp": 48, "wp": 48, "weight": "w4", "kv_len": 77},
        # a fine-tuned style (rank-32 LoRA) at 640 x 896 without guidance
        {"name": "mlp_640x896_lora", "kind": "mlp", "b": 1, "hp": 40, "wp": 56, "weight": "w4", "lora": 32},
        # the attention op of the default image by itself, from fp32 q/k/v
        {"name": "attn_1024_cfg", "kind": "attn", "b": 2, "hp": 64, "wp": 64, "precision": "bf16"},
        # the full-precision option, at 512 x 512
        {"name": "attn_512_fp32", "kind": "attn", "b": 1, "hp": 32, "wp": 32, "precision": "fp32"},
        # a prompt padded to the context length, and an ordinary short prompt
        {"name": "text_512", "kind": "text", "tokens": 512, "layers": 4, "precision": "bf16"},
        {"name": "text_43", "kind": "text", "tokens": 43, "layers": 4, "precision": "bf16"},
        # decoding a 1024 x 1024 image: the 192-channel level with its upsampling to full resolution,
        # and the attention over 128 x 128 latents, at the decoder's default precision
        {"name": "vae_stage_512_192", "kind": "vae_stage", "h": 512, "w": 512, "c": 192, "up": True, "precision": "fp32"},
        {"name": "vae_attn_1024", "kind": "vae_attn", "h": 128, "w": 128, "precision": "fp32"},
        # once per step and sigma: matrix-vector products over 350 MB of weights
        {"name": "time_cond", "kind": "time_cond", "lora": 0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi):
    """A token grid (hp, wp) of lo to hi tokens, aspect ratios up to about 2:1."""
    n, r = math.exp(rng.uniform(math.log(lo), math.log(hi))), math.exp(rng.uniform(-0.35, 0.35))
    hp = max(8, int(round(math.sqrt(n) * r)))
    return hp, max(8, min(int(hi // hp), int(round(n / hp))))


def draw(rng):
    kind = rng.choice(["block", "self", "cross", "mlp", "attn", "text", "vae_stage", "vae_attn", "time_cond"])
    if kind in ("block", "self", "cross", "mlp"):
        b = rng.choice([1, 2])
        hp, wp = _grid(rng, 256, 4096)  # 256 x 256 to 1024 x 1024 pixels and what has their area
        c = {"kind": kind, "b": b, "hp": hp, "wp": wp, "weight": rng.choice(["w4", "w4", "i8"])}
        if kind in ("block", "cross"):
            c["kv_len"] = rng.choice([0, _log_int(rng, 8, LK)])
        else:
            c["lora"] = rng.choice([0, 0, 16, 32, 64])
        return c
    if kind == "attn":
        precision = rng.choice(["bf16", "bf16", "fp32"])
        b = rng.choice([1, 2])
        hp, wp = _grid(rng, 256, 4096 if precision == "bf16" else 2048)
        return {"kind": kind, "b": b, "hp": hp, "wp": wp, "precision": precision}
    if kind == "text":
        return {"kind": kind, "tokens": _log_int(rng, 8, 512), "layers": 4, "precision": rng.choice(["bf16", "bf16", "fp32"])}
    if kind == "vae_stage":
        c = rng.choice([96, 192, 384])
        scale = {384: 1, 192: 4, 96: 8}[c]  # the level's resolution over the latent's
        if c == 384:
            scale = rng.choice([1, 2])
        h, w = 8 * rng.randint(4, 16), 8 * rng.randint(4, 16)
        return {"kind": kind, "h": h * scale, "w": w * scale, "c": c, "up": c > 96 and rng.choice([True, False]),
                "precision": rng.choice(["fp32", "fp32", "bf16"])}
    if kind == "vae_attn":
        return {"kind": kind, "h": 2 * rng.randint(16, 64), "w": 2 * rng.randint(16, 64),
                "precision": rng.choice(["fp32", "fp32", "bf16"])}
    return {"kind": kind, "lora": 4 * rng.randint(1, 32)}


# ---------------------------------------------------------------- inputs

_context = None


def _ctx():
    """The program's one context."""
    global _context
    if _context is None:
        _context = anima.Context(0)
    return _context


class _Inputs:
    """Seeded device tensors, in the order they are asked for."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, shape, std=1.0, mean=0.0):
        return torch.randn(shape, generator=self.g, device="cuda") * std + mean

    def uniform(self, shape, lo, hi):
        return torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def integers(self, shape, lo, hi):
        return torch.randint(lo, hi + 1, shape, generator=self.g, device="cuda")

    def linear(self, kind, n, k):
        """A quantized linear [n, k] in the checkpoint formats, as a dict of tensors."""
        scale = self.uniform((n,), 0.5, 1.5) / (127 * math.sqrt(k))
        if kind == "i8":
            return {"kind": kind, "n": n, "k": k, "scale": scale,
                    "w": self.normal((n, k), 40.0).round_().clamp_(-127, 127).to(torch.int8)}
        return {"kind": kind, "n": n, "k": k, "scale": scale,
                "w": self.integers((n, k // 2), 0, 255).to(torch.uint8),
                "srel": self.integers((n, k // 16), 0x60, 0x6F).to(torch.uint8),
                "codebook": torch.tensor(CODEBOOK, device="cuda")}

    def bf16(self, n, k, gain=1.0):
        """A bf16 matrix [n, k], uniform with a variance of gain^2 / k."""
        a = gain * math.sqrt(3.0 / k)
        return self.uniform((n, k), -a, a).to(torch.bfloat16)

    def lora(self, n, k, r, parts=1):
        """LoRA factors of a linear [n, k] whose `parts` column blocks have ranks of their own: A stacked
        [parts * r, k] (in the rotated input's basis) and B [n, r], as fp32."""
        return {"a": self.normal((parts * r, k), 1.0 / math.sqrt(k)), "b": self.normal((n, r), 0.5 / math.sqrt(r)),
                "r": r, "cols": n // parts if parts > 1 else 0}


def _empty(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda")


def _ptr(t):
    return None if t is None else t.data_ptr()


def _weight(d):
    kind = {"i8": anima.W_I8, "w4": anima.W_W4}[d["kind"]]
    return anima.weight(kind, d["n"], d["k"], _ptr(d["w"]), scale=_ptr(d["scale"]),
                        srel=_ptr(d.get("srel")), codebook=_ptr(d.get("codebook")))


def _split3(t):
    """The three bf16 planes of an fp32 matrix that the LoRA products read."""
    out = _empty(3, *t.shape, dtype=torch.bfloat16)
    torch.cuda.synchronize()
    _ctx().split3_bf16(_ptr(t), _ptr(out), t.numel())
    return out


class _Lora:
    """A LoRA as a program keeps it beside its linear: A and B as split planes, the A product's buffer."""

    def __init__(self, d, m):
        self.a, self.b, self.r, self.cols = _split3(d["a"]), _split3(d["b"]), d["r"], d["cols"]
        self.rows = d["a"].shape[0]
        self.xa = _empty(m, self.rows)
        self.weight = anima.weight(anima.W_F32S3, self.rows, d["a"].shape[1], _ptr(self.a))

    def args(self, m, xq, xs):
        """Runs the A product over the int8 rows; the arguments of the linear that adds B times it."""
        _ctx().linear(self.weight, m, _ptr(self.xa), xq=_ptr(xq), xs=_ptr(xs))
        return {"lora_xa": _ptr(self.xa), "ld_lora_xa": self.rows, "lora_b": _ptr(self.b), "lora_r": self.r,
                "lora_cols": self.cols}


def _rope3d(hp, wp):
    return torch.from_numpy(anima.dit_rope_table(hp, wp)).cuda()


def _kv_len(case):
    """Valid context tokens of each prompt: all of them, or the case's count and (with guidance) a shorter
    negative prompt."""
    n = case["kv_len"]
    return [LK] * case["b"] if not n else [n, max(1, n // 2)][: case["b"]]


def _dit_inputs(case, seed):
    """The tensors of a DiT sublayer or block, as made from the seed (exact() makes the same)."""
    kind, b = case["kind"], case["b"]
    m = b * case["hp"] * case["wp"]
    g, t = _Inputs(seed), {}
    t["x"] = g.normal((m, D))
    w, lora = case["weight"], case.get("lora", 0)
    for part in ("self", "cross", "mlp"):
        if kind not in ("block", part):
            continue
        mod = g.normal((3 * D,), 0.3)  # shift, scale, gate
        mod[2 * D:] = mod[2 * D:] * 2
        t["mod_" + part] = mod
        if part == "self":
            t["qkv"], t["o"] = g.linear(w, 3 * D, D), g.linear(w, D, D)
            t["qn"], t["kn"] = g.normal((HD,), 0.02, 1.0), g.normal((HD,), 0.02, 1.0)
            if lora:
                t["lora_qkv"], t["lora_o"] = g.lora(3 * D, D, lora, 3), g.lora(D, D, lora)
        elif part == "cross":
            t["cq"], t["co"] = g.linear(w, D, D), g.linear(w, D, D)
            t["cqn"] = g.normal((HD,), 0.02, 1.0)
            t["ck"], t["cv"] = g.normal((b * LK, D)), g.normal((b * LK, D))
        else:
            t["l1"], t["l2"] = g.linear(w, MLP, D), g.linear(w, D, MLP)
            if lora:
                t["lora_l1"], t["lora_l2"] = g.lora(MLP, D, lora), g.lora(D, MLP, lora)
    return t


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = case
    make, s.run = {"block": (_prepare_block, _run_block), "self": (_prepare_block, _run_block),
                   "cross": (_prepare_block, _run_block), "mlp": (_prepare_block, _run_block),
                   "attn": (_prepare_attn, _run_attn), "text": (_prepare_text, _run_text),
                   "vae_stage": (_prepare_vae_stage, _run_vae_stage), "vae_attn": (_prepare_vae_attn, _run_vae_attn),
                   "time_cond": (_prepare_time_cond, _run_time_cond)}[case["kind"]]
    make(s, case, seed)
    torch.cuda.synchronize()  # the context's stream and torch's are two
    return s


def run(state):
    return state.run(state)


# ---------------------------------------------------------------- DiT block and its sublayers


def _prepare_block(s, case, seed):
    ctx, t = _ctx(), _dit_inputs(case, seed)
    b, l = case["b"], case["hp"] * case["wp"]
    m = b * l
    s.t, s.b, s.l, s.m = t, b, l, m
    s.x = t["x"]
    s.parts = ["self", "cross", "mlp"] if case["kind"] == "block" else [case["kind"]]
    s.w = {k: _weight(v) for k, v in t.items() if isinstance(v, dict) and "kind" in v}
    s.lora = {k[5:]: _Lora(v, m) for k, v in t.items() if k.startswith("lora_")}
    s.xq, s.xs = _empty(m, D, dtype=torch.int8), _empty(m)
    s.aligned = l % 64 == 0  # the projections can write the attention's operands
    if "self" in s.parts:
        s.cs = _rope3d(case["hp"], case["wp"])
        if s.aligned:
            s.kv = _empty(ctx.attention_kv_bytes(b, HEADS, l), dtype=torch.uint8)
        else:
            s.qkv = _empty(m, 3 * D)
    if "cross" in s.parts:
        # once per prompt: the context's keys and values in the attention's operand layout
        s.kv_len = _kv_len(case)
        s.ckv = _empty(ctx.attention_kv_bytes(b, HEADS, LK), dtype=torch.uint8)
        torch.cuda.synchronize()
        ctx.attention(q=_ptr(t["ck"]), k=_ptr(t["ck"]), v=_ptr(t["cv"]), o=_ptr(s.ckv), B=b, Lq=LK, Lk=LK, H=HEADS, D=HD,
                      ldq=D, ldk=D, ldv=D, prepare_into=_ptr(s.ckv))
        if not s.aligned:
            s.q = _empty(m, D)
    if s.aligned:
        s.qp = _empty(m, D, dtype=torch.bfloat16)
    s.a = _empty(m, D, dtype=torch.bfloat16)
    s.aq, s.as_ = _empty(m, D, dtype=torch.int8), _empty(m)
    if "mlp" in s.parts:
        s.pre = _empty(m, MLP)
        s.hq, s.hs = _empty(m, MLP, dtype=torch.int8), _empty(m)


def _norm(ctx, s, mod):
    ctx.layernorm_mod(_ptr(s.x), _ptr(mod), 0, D, s.m, D, rotate=True, q=_ptr(s.xq), s=_ptr(s.xs))


def _lora_args(s, name, xq, xs):
    return s.lora[name].args(s.m, xq, xs) if name in s.lora else {}


def _out_projection(ctx, s, name, mod):
    """x += gate * linear(attention output), from the attention's bf16 rows."""
    ctx.quant_rows_bf16(_ptr(s.a), s.m, D, True, _ptr(s.aq), _ptr(s.as_))
    ctx.linear(s.w[name], s.m, _ptr(s.x), xq=_ptr(s.aq), xs=_ptr(s.as_), epilogue=anima.EPI_GATED, gate=_ptr(mod),
               gate_off=2 * D, **_lora_args(s, name, s.aq, s.as_))


def _run_self(ctx, s):
    t, mod = s.t, s.t["mod_self"]
    _norm(ctx, s, mod)
    lora = _lora_args(s, "qkv", s.xq, s.xs)
    if s.aligned:
        ctx.linear_qkv(s.w["qkv"], s.m, None, B=s.b, L=s.l, H=HEADS, k_norm=_ptr(t["kn"]), rope_cs=_ptr(s.cs),
                       rope_sin_off=s.l * 64, kv_prep=_ptr(s.kv), xq=_ptr(s.xq), xs=_ptr(s.xs), q_norm=_ptr(t["qn"]),
                       q_prep=_ptr(s.qp), **lora)
        ctx.attention(q=None, k=None, v=None, o=_ptr(s.a), B=s.b, Lq=s.l, Lk=s.l, H=HEADS, D=HD, ldq=D, ldk=D, ldv=D,
                      kv_prep=_ptr(s.kv), q_prep=_ptr(s.qp), o_bf16=True)
    else:
        ctx.linear(s.w["qkv"], s.m, _ptr(s.qkv), xq=_ptr(s.xq), xs=_ptr(s.xs), **lora)
        ctx.attention(q=_ptr(s.qkv), k=_ptr(s.qkv), v=_ptr(s.qkv), o=_ptr(s.a), B=s.b, Lq=s.l, Lk=s.l, H=HEADS, D=HD,
                      ldq=3 * D, ldk=3 * D, ldv=3 * D, k_off=D, v_off=2 * D, q_norm=_ptr(t["qn"]), k_norm=_ptr(t["kn"]),
                      rope_cs=_ptr(s.cs), rope_sin_off=s.l * 64, o_bf16=True)
    _out_projection(ctx, s, "o", mod)


def _run_cross(ctx, s):
    t, mod = s.t, s.t["mod_cross"]
    _norm(ctx, s, mod)
    if s.aligned:
        ctx.linear_qkv(s.w["cq"], s.m, None, B=s.b, L=s.l, H=HEADS, xq=_ptr(s.xq), xs=_ptr(s.xs), q_norm=_ptr(t["cqn"]),
                       q_prep=_ptr(s.qp))
        ctx.attention(q=None, k=None, v=None, o=_ptr(s.a), B=s.b, Lq=s.l, Lk=LK, H=HEADS, D=HD, ldq=D, ldk=D, ldv=D,
                      kv_prep=_ptr(s.ckv), q_prep=_ptr(s.qp), kv_len=s.kv_len, o_bf16=True)
    else:
        ctx.linear(s.w["cq"], s.m, _ptr(s.q), xq=_ptr(s.xq), xs=_ptr(s.xs))
        ctx.attention(q=_ptr(s.q), k=None, v=None, o=_ptr(s.a), B=s.b, Lq=s.l, Lk=LK, H=HEADS, D=HD, ldq=D, ldk=D, ldv=D,
                      kv_prep=_ptr(s.ckv), q_norm=_ptr(t["cqn"]), kv_len=s.kv_len, o_bf16=True)
    _out_projection(ctx, s, "co", mod)


def _run_mlp(ctx, s):
    mod = s.t["mod_mlp"]
    _norm(ctx, s, mod)
    ctx.linear(s.w["l1"], s.m, _ptr(s.pre), xq=_ptr(s.xq), xs=_ptr(s.xs), **_lora_args(s, "l1", s.xq, s.xs))
    ctx.quant_rows(_ptr(s.pre), s.m, MLP, True, _ptr(s.hq), _ptr(s.hs), act="gelu")
    ctx.linear(s.w["l2"], s.m, _ptr(s.x), xq=_ptr(s.hq), xs=_ptr(s.hs), epilogue=anima.EPI_GATED, gate=_ptr(mod),
               gate_off=2 * D, **_lora_args(s, "l2", s.hq, s.hs))


def _run_block(s):
    ctx = _ctx()
    for part in s.parts:
        {"self": _run_self, "cross": _run_cross, "mlp": _run_mlp}[part](ctx, s)
    return s.x  # the residual stream, updated in place


# ---------------------------------------------------------------- attention op


def _attn_inputs(case, seed):
    g, l = _Inputs(seed), case["hp"] * case["wp"]
    return {"qkv": g.normal((case["b"], l, 3 * D)), "qn": g.normal((HD,), 0.02, 1.0), "kn": g.normal((HD,), 0.02, 1.0)}


def _prepare_attn(s, case, seed):
    s.t, s.b, s.l = _attn_inputs(case, seed), case["b"], case["hp"] * case["wp"]
    s.cs, s.o = _rope3d(case["hp"], case["wp"]), _empty(s.b, s.l, D)


def _run_attn(s):
    t, q = s.t, _ptr(s.t["qkv"])
    _ctx().attention(q=q, k=q, v=q, o=_ptr(s.o), B=s.b, Lq=s.l, Lk=s.l, H=HEADS, D=HD, ldq=3 * D, ldk=3 * D, ldv=3 * D,
                     k_off=D, v_off=2 * D, precision=PRECISION[s.case["precision"]], q_norm=_ptr(t["qn"]),
                     k_norm=_ptr(t["kn"]), rope_cs=_ptr(s.cs), rope_sin_off=s.l * 64)
    return s.o


# ---------------------------------------------------------------- text encoder


def _text_inputs(case, seed):
    g, layers = _Inputs(seed), []
    x = g.normal((case["tokens"], TE_D), 0.5)
    for _ in range(case["layers"]):
        layers.append({"ln1": g.uniform((TE_D,), 0.9, 1.1), "ln2": g.uniform((TE_D,), 0.9, 1.1),
                       "qn": g.uniform((HD,), 0.9, 1.1), "kn": g.uniform((HD,), 0.9, 1.1),
                       "qkv": g.bf16((TE_H + 2 * TE_KH) * HD, TE_D), "o": g.bf16(TE_D, TE_H * HD),
                       "gate": g.bf16(TE_MLP, TE_D), "up": g.bf16(TE_MLP, TE_D), "down": g.bf16(TE_D, TE_MLP)})
    return {"x": x, "layers": layers, "norm": g.uniform((TE_D,), 0.9, 1.1)}


def _rope1d_angles(n):
    inv = np.array([np.float32(1.0 / TE_THETA ** (2 * i / HD)) for i in range(HD // 2)], np.float64)
    return (np.arange(n, dtype=np.float64)[:, None] * inv[None, :]).astype(np.float32)


class _TextState:
    """The encoder's buffers for one token count and the graph of its layers over them."""

    graph = None

    def __del__(self):
        if self.graph is not None:
            _ctx().graph_destroy(self.graph)


def _text_layers(s):
    ctx, n = _ctx(), s.n
    for p in s.layers:
        w = p["w"]
        ctx.rmsnorm(_ptr(s.x), p["ln1"], _ptr(s.h), n, TE_D)
        ctx.linear(w["qkv"], n, _ptr(s.qkv), x=_ptr(s.h))
        ld = (TE_H + 2 * TE_KH) * HD
        ctx.attention(q=_ptr(s.qkv), k=_ptr(s.qkv), v=_ptr(s.qkv), o=_ptr(s.a), B=1, Lq=n, Lk=n, H=TE_H, D=HD, ldq=ld,
                      ldk=ld, ldv=ld, k_off=TE_H * HD, v_off=(TE_H + TE_KH) * HD, group=TE_H // TE_KH, causal=1,
                      q_norm=p["qn"], k_norm=p["kn"], rope_cs=_ptr(s.cs), rope_sin_off=n * (HD // 2), precision=s.precision)
        ctx.linear(w["o"], n, _ptr(s.x), x=_ptr(s.a), epilogue=anima.EPI_RESID)
        ctx.rmsnorm(_ptr(s.x), p["ln2"], _ptr(s.h), n, TE_D)
        ctx.linear(w["gate"], n, _ptr(s.g), x=_ptr(s.h))
        ctx.linear(w["up"], n, _ptr(s.u), x=_ptr(s.h))
        ctx.elementwise("silu_mul", _ptr(s.g), _ptr(s.u), _ptr(s.g), n * TE_MLP)
        ctx.linear(w["down"], n, _ptr(s.x), x=_ptr(s.g), epilogue=anima.EPI_RESID)
    ctx.rmsnorm(_ptr(s.x), _ptr(s.t["norm"]), _ptr(s.out), n, TE_D)


def _prepare_text(state, case, seed):
    s = state.s = _TextState()
    s.t, s.n, s.precision = _text_inputs(case, seed), case["tokens"], PRECISION[case["precision"]]
    s.layers = []
    for l in s.t["layers"]:
        w = {k: anima.weight(anima.W_BF16, v.shape[0], v.shape[1], _ptr(v)) for k, v in l.items() if v.dim() == 2}
        s.layers.append({"w": w, **{k: _ptr(v) for k, v in l.items() if v.dim() == 1}})
    s.x, s.h, s.out, s.a = (_empty(s.n, k) for k in (TE_D, TE_D, TE_D, TE_H * HD))
    s.qkv, s.g, s.u = _empty(s.n, (TE_H + 2 * TE_KH) * HD), _empty(s.n, TE_MLP), _empty(s.n, TE_MLP)
    s.cs = torch.from_numpy(anima.rope_table(_rope1d_angles(s.n))).cuda()
    torch.cuda.synchronize()
    ctx = _ctx()
    ctx.elementwise("copy", _ptr(s.t["x"]), None, _ptr(s.x), s.n * TE_D)
    _text_layers(s)  # one eager pass first: the pool then holds what the capture asks for
    ctx.sync()
    ctx.graph_begin()
    _text_layers(s)
    s.graph = ctx.graph_end()


def _run_text(state):
    ctx, s = _ctx(), state.s
    ctx.elementwise("copy", _ptr(s.t["x"]), None, _ptr(s.x), s.n * TE_D)  # the prompt's embedding rows
    ctx.graph_launch(s.graph)
    return s.out, s.x


# ---------------------------------------------------------------- VAE decoder


def _vae_stage_inputs(case, seed):
    g, c = _Inputs(seed), case["c"]
    t = {"x": g.normal((case["h"] * case["w"], c)), "n1": g.uniform((c,), 0.9, 1.1), "n2": g.uniform((c,), 0.9, 1.1),
         "c1": g.bf16(c, 9 * c), "b1": g.uniform((c,), -0.05, 0.05), "c2": g.bf16(c, 9 * c, 0.5),
         "b2": g.uniform((c,), -0.05, 0.05)}
    if case["up"]:
        t["cu"], t["bu"] = g.bf16(c // 2, 9 * c), g.uniform((c // 2,), -0.05, 0.05)
    return t


def _prepare_vae_stage(s, case, seed):
    s.t = _vae_stage_inputs(case, seed)
    n, c = case["h"] * case["w"], case["c"]
    s.x, s.h, s.a = s.t["x"], _empty(n, c), _empty(n, c)
    s.y = _empty(4 * n, c // 2) if case["up"] else None


def _run_vae_stage(s):
    ctx, t, case = _ctx(), s.t, s.case
    h, w, c, prec = case["h"], case["w"], case["c"], PRECISION[case["precision"]]
    ctx.channel_norm(_ptr(s.x), _ptr(t["n1"]), _ptr(s.h), h * w, c, silu=True)
    ctx.conv3x3(_ptr(s.h), _ptr(t["c1"]), _ptr(s.a), B=1, H=h, W=w, cin=c, cout=c, bias=_ptr(t["b1"]), precision=prec)
    ctx.channel_norm(_ptr(s.a), _ptr(t["n2"]), _ptr(s.h), h * w, c, silu=True)
    ctx.conv3x3(_ptr(s.h), _ptr(t["c2"]), _ptr(s.x), B=1, H=h, W=w, cin=c, cout=c, bias=_ptr(t["b2"]), resid=True,
                precision=prec)
    if not case["up"]:
        return s.x
    ctx.conv3x3(_ptr(s.x), _ptr(t["cu"]), _ptr(s.y), B=1, H=2 * h, W=2 * w, cin=c, cout=c // 2, up=True,
                bias=_ptr(t["bu"]), precision=prec)
    return s.x, s.y


def _vae_attn_inputs(case, seed):
    # the projections' outputs: scores of a few units
    return {"qkv": _Inputs(seed).normal((case["h"] * case["w"], 3 * VAE_C))}


def _prepare_vae_attn(s, case, seed):
    s.t, s.n = _vae_attn_inputs(case, seed), case["h"] * case["w"]
    s.o = _empty(s.n, VAE_C)


def _run_vae_attn(s):
    q = _ptr(s.t["qkv"])
    _ctx().attention(q=q, k=q, v=q, o=_ptr(s.o), B=1, Lq=s.n, Lk=s.n, H=1, D=VAE_C, ldq=3 * VAE_C, ldk=3 * VAE_C,
                     ldv=3 * VAE_C, k_off=VAE_C, v_off=2 * VAE_C, precision=PRECISION[s.case["precision"]])
    return s.o


# ---------------------------------------------------------------- modulation vectors


def _time_cond_inputs(case, seed):
    g, parts, r = _Inputs(seed), 3 * BLOCKS, case["lora"]
    t = {"t": g.normal((1, D)), "t1": g.bf16(D, D), "t2": g.bf16(3 * D, D), "tn": g.uniform((D,), 0.9, 1.1),
         "w1": g.bf16((parts + 1) * RANK_MOD, D), "w2": g.bf16(parts * 3 * D, RANK_MOD, 0.1),
         "wf": g.bf16(2 * D, RANK_MOD, 0.1)}
    if r:
        # one LoRA per modulation linear, stacked; the scales folded into the second factors
        t["a1"], t["b1"] = g.normal(((parts + 1) * r, D), 1 / math.sqrt(D)), g.normal(((parts + 1) * RANK_MOD, r), 0.1)
        t["a2"], t["b2"] = g.normal((parts * r, RANK_MOD), 1 / math.sqrt(RANK_MOD)), g.normal((parts * 3 * D, r), 0.1)
    return t


def _prepare_time_cond(s, case, seed):
    s.t = t = _time_cond_inputs(case, seed)
    parts, r = 3 * BLOCKS, case["lora"]
    s.w = {k: anima.weight(anima.W_BF16, t[k].shape[0], t[k].shape[1], _ptr(t[k])) for k in ("t1", "t2", "w1")}
    s.hid, s.low, s.emb, s.semb = _empty(1, D), _empty(1, 3 * D), _empty(1, D), _empty(1, D)
    s.h1, s.all, s.final = _empty(1, (parts + 1) * RANK_MOD), _empty(parts, 3 * D), _empty(1, 2 * D)
    s.la = _empty((parts + 1) * r) if r else None


def _run_time_cond(s):
    ctx, t, r, parts = _ctx(), s.t, s.case["lora"], 3 * BLOCKS
    ctx.linear(s.w["t1"], 1, _ptr(s.hid), x=_ptr(t["t"]), act="silu")
    ctx.linear(s.w["t2"], 1, _ptr(s.low), x=_ptr(s.hid))
    ctx.rmsnorm(_ptr(t["t"]), _ptr(t["tn"]), _ptr(s.emb), 1, D)
    ctx.elementwise("silu", _ptr(s.emb), None, _ptr(s.semb), D)
    ctx.linear(s.w["w1"], 1, _ptr(s.h1), x=_ptr(s.semb))
    if r:
        ctx.gemv_grouped_f32(1, (parts + 1) * r, D, _ptr(s.semb), 0, _ptr(t["a1"]), 0, _ptr(s.la), 0)
        ctx.gemv_grouped_f32(parts + 1, RANK_MOD, r, _ptr(s.la), r, _ptr(t["b1"]), RANK_MOD * r, _ptr(s.h1), RANK_MOD,
                             accumulate=True)
    ctx.linear_grouped_bf16(parts, 1, 3 * D, RANK_MOD, _ptr(s.h1), (parts + 1) * RANK_MOD, RANK_MOD, _ptr(t["w2"]),
                            3 * D * RANK_MOD, _ptr(s.low), 0, _ptr(s.all), 3 * D, 3 * D)
    ctx.linear_grouped_bf16(1, 1, 2 * D, RANK_MOD, _ptr(s.h1) + 4 * parts * RANK_MOD, RANK_MOD, 0, _ptr(t["wf"]), 0,
                            _ptr(s.low), 0, _ptr(s.final), 2 * D, 0)
    if r:
        ctx.gemv_grouped_f32(parts, r, RANK_MOD, _ptr(s.h1), RANK_MOD, _ptr(t["a2"]), r * RANK_MOD, _ptr(s.la), r)
        ctx.gemv_grouped_f32(parts, 3 * D, r, _ptr(s.la), r, _ptr(t["b2"]), 3 * D * r, _ptr(s.all), 3 * D, accumulate=True)
    return s.all, s.final


# ---------------------------------------------------------------- what a pass cannot do without


def _sublayer_work(case, part):
    """Weights, the residual stream in and out, and the products."""
    b, l = case["b"], case["hp"] * case["wp"]
    m = b * l
    per = 1.0 if case["weight"] == "i8" else 0.5 + 1 / 16
    if part == "self":
        macs, extra = m * 4 * D * D + 2 * b * l * l * D, 0
        weights = 4 * D * D
    elif part == "cross":
        keys = sum(_kv_len(case))
        macs, extra = m * 2 * D * D + 2 * l * keys * D, 2 * 2 * keys * D
        weights = 2 * D * D
    else:
        macs, extra = 2 * m * D * MLP, 0
        weights = 2 * D * MLP
    r = case.get("lora", 0)
    if r:
        n = {"self": (4 * D, 4 * D), "mlp": (D + MLP, D + MLP)}[part]
        macs += m * r * (n[0] + n[1])
        extra += 4 * r * (n[0] + n[1])
    return weights * per + extra, 2 * macs


def work(case):
    kind = case["kind"]
    if kind in ("block", "self", "cross", "mlp"):
        m = case["b"] * case["hp"] * case["wp"]
        parts = ["self", "cross", "mlp"] if kind == "block" else [kind]
        each = [_sublayer_work(case, p) for p in parts]
        return {"bytes": 2 * 4 * m * D + sum(e[0] for e in each), "flops": sum(e[1] for e in each)}
    if kind == "attn":
        b, l = case["b"], case["hp"] * case["wp"]
        return {"bytes": 4 * 4 * b * l * D, "flops": 4 * b * l * l * D}
    if kind == "text":
        n, k = case["tokens"], case["layers"]
        per = TE_D * (TE_H + 2 * TE_KH) * HD + TE_D * TE_H * HD + 3 * TE_D * TE_MLP
        return {"bytes": 2 * per * k + 3 * 4 * n * TE_D, "flops": k * (2 * n * per + 2 * n * (n + 1) * TE_H * HD)}
    if kind == "vae_stage":
        n, c, up = case["h"] * case["w"], case["c"], case["up"]
        return {"bytes": 2 * 4 * n * c + (8 * n * c if up else 0) + 2 * 9 * c * c * (2.5 if up else 2),
                "flops": 2 * 9 * n * c * c * (2 + (2 if up else 0))}
    if kind == "vae_attn":
        n = case["h"] * case["w"]
        return {"bytes": 4 * 4 * n * VAE_C, "flops": 4 * n * n * VAE_C}
    parts, r = 3 * BLOCKS, case["lora"]
    weights = 4 * D * D + (parts + 1) * RANK_MOD * D + parts * 3 * D * RANK_MOD + 2 * D * RANK_MOD
    lora = r * ((parts + 1) * (D + RANK_MOD) + parts * (RANK_MOD + 3 * D))
    return {"bytes": 2 * weights + 4 * lora + 4 * parts * 3 * D, "flops": 2 * (weights + lora)}


def tolerance(case):
    """About four times what the path differs from the 64-bit result by: bf16 attention operands 3.3e-3 (in
    a sublayer the residual stream dilutes them to 7e-4 and below), fp32-level sums up to 6e-6 over a
    16384-term row and 1e-6 otherwise."""
    kind = case["kind"]
    if kind in ("block", "self", "cross", "mlp"):
        return {"rel": 3e-3, "max": 0.1}
    if kind in ("attn", "text", "vae_stage", "vae_attn") and case["precision"] == "bf16":
        return {"rel": 1.3e-2, "max": 0.3}
    if kind in ("vae_stage", "vae_attn"):
        return {"rel": 3e-5, "max": 2e-3}
    return {"rel": 1e-5, "max": 4e-4}


# ---------------------------------------------------------------- the same in 64 bits


def _f64(t):
    return t.to(torch.float64)


_hadamard = None


def _rotate(x):
    """The ConvRot rotation: x times the 256 x 256 regular Hadamard matrix per group of 256 columns."""
    global _hadamard
    if _hadamard is None:
        h4 = torch.tensor([[1, 1, 1, -1], [1, 1, -1, 1], [1, -1, 1, 1], [-1, 1, 1, 1]], dtype=torch.float64, device="cuda")
        _hadamard = torch.kron(torch.kron(h4, h4), torch.kron(h4, h4)) / 16
    return (x.reshape(-1, 256) @ _hadamard).reshape(x.shape)


def _quantize(x):
    """Rows rounded to 127 steps of their largest value, as (integers, steps)."""
    step = x.abs().amax(1, keepdim=True) / 127
    return torch.round(x / torch.where(step > 0, step, torch.ones_like(step))), step


def _dequantize(d):
    """The weight matrix of a quantized linear, in the rotated basis."""
    if d["kind"] == "i8":
        grid = _f64(d["w"])
    else:
        codes = torch.stack([d["w"] & 15, d["w"] >> 4], -1).reshape(d["n"], d["k"]).long()
        rel = _f64(d["srel"].view(torch.float8_e4m3fn).float()).repeat_interleave(16, 1)
        grid = torch.round(_f64(d["codebook"])[codes] * rel).clamp(-127, 127)
    return grid * _f64(d["scale"])[:, None]


def _linear64(x, d, lora):
    """The quantized linear (and its LoRA) on rotated rows."""
    q, step = _quantize(x)
    x = q * step
    y = x @ _dequantize(d).T
    if lora is not None:
        parts = max(1, lora["a"].shape[0] // lora["r"])
        xa = (x @ _f64(lora["a"]).T).reshape(x.shape[0], parts, lora["r"])
        b = _f64(lora["b"]).reshape(parts, -1, lora["r"])
        y = y + torch.cat([xa[:, i] @ b[i].T for i in range(parts)], 1)
    return y


def _norm64(x, mod):
    mod = _f64(mod)
    mean = x.mean(1, keepdim=True)
    var = ((x - mean) ** 2).mean(1, keepdim=True)
    return _rotate((x - mean) / torch.sqrt(var + 1e-6) * (1 + mod[D:2 * D]) + mod[:D])


def _rms64(x, w, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * _f64(w)


def _angles3d(hp, wp):
    """The DiT's rotary angles [hp * wp, 64]: 22 temporal slots at time 0, 21 for the row, 21 for the column."""
    f = np.float32(1.0 / (1e4 * 4.0 ** (42 / 40)) ** (np.arange(21) * 2 / 42).astype(np.float32).astype(np.float64))
    a = np.zeros((hp, wp, 64), np.float32)
    a[:, :, 22:43] = np.arange(hp)[:, None, None] * f.astype(np.float64)
    a[:, :, 43:] = np.arange(wp)[None, :, None] * f.astype(np.float64)
    return a.reshape(hp * wp, 64)


def _rope64(x, angles):
    """x [..., tokens, heads, dims] with its halves rotated by `angles` [tokens, dims / 2]."""
    angles = torch.from_numpy(angles).cuda().double()[:, None]
    c, s = torch.cos(angles), torch.sin(angles)
    a, b = x.chunk(2, -1)
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attention64(q, k, v, valid=None, causal=False):
    """q [b, lq, h, d], k and v [b, lk, h / group, d]."""
    b, lq, h, d = q.shape
    group = h // k.shape[2]
    o = torch.empty_like(q)
    for i in range(b):
        n = k.shape[1] if valid is None else valid[i]
        for j in range(h):
            kk, vv = k[i, :n, j // group], v[i, :n, j // group]
            for r in range(0, lq, 4096):
                s = q[i, r:r + 4096, j] @ kk.T / math.sqrt(d)
                if causal:
                    at = torch.arange(r, r + s.shape[0], device=s.device)
                    s = s.masked_fill(torch.arange(n, device=s.device)[None, :] > at[:, None], -math.inf)
                o[i, r:r + 4096, j] = torch.softmax(s, -1) @ vv
    return o


def _exact_block(case, seed):
    t = _dit_inputs(case, seed)
    b, l = case["b"], case["hp"] * case["wp"]
    x = _f64(t["x"])
    parts = ["self", "cross", "mlp"] if case["kind"] == "block" else [case["kind"]]
    if "self" in parts:
        qkv = _linear64(_norm64(x, t["mod_self"]), t["qkv"], t.get("lora_qkv")).reshape(b, l, 3, HEADS, HD)
        cs = _angles3d(case["hp"], case["wp"])
        o = _attention64(_rope64(_rms64(qkv[:, :, 0], t["qn"]), cs), _rope64(_rms64(qkv[:, :, 1], t["kn"]), cs), qkv[:, :, 2])
        x = x + _f64(t["mod_self"])[2 * D:] * _linear64(_rotate(o.reshape(-1, D)), t["o"], t.get("lora_o"))
    if "cross" in parts:
        q = _linear64(_norm64(x, t["mod_cross"]), t["cq"], None).reshape(b, l, HEADS, HD)
        k, v = (_f64(t[n]).reshape(b, LK, HEADS, HD) for n in ("ck", "cv"))
        o = _attention64(_rms64(q, t["cqn"]), k, v, valid=_kv_len(case))
        x = x + _f64(t["mod_cross"])[2 * D:] * _linear64(_rotate(o.reshape(-1, D)), t["co"], None)
    if "mlp" in parts:
        y = _linear64(_norm64(x, t["mod_mlp"]), t["l1"], t.get("lora_l1"))
        y = 0.5 * y * (1 + torch.erf(y / math.sqrt(2)))
        x = x + _f64(t["mod_mlp"])[2 * D:] * _linear64(_rotate(y), t["l2"], t.get("lora_l2"))
    return x


def _exact_attn(case, seed):
    t = _attn_inputs(case, seed)
    b, l = case["b"], case["hp"] * case["wp"]
    qkv, cs = _f64(t["qkv"]).reshape(b, l, 3, HEADS, HD), _angles3d(case["hp"], case["wp"])
    o = _attention64(_rope64(_rms64(qkv[:, :, 0], t["qn"]), cs), _rope64(_rms64(qkv[:, :, 1], t["kn"]), cs), qkv[:, :, 2])
    return o.reshape(b, l, D)


def _exact_text(case, seed):
    t, n = _text_inputs(case, seed), case["tokens"]
    x, cs = _f64(t["x"]), _rope1d_angles(n)
    for p in t["layers"]:
        qkv = _rms64(x, p["ln1"]) @ _f64(p["qkv"]).T
        q, k, v = (a.reshape(1, n, -1, HD) for a in qkv.split([TE_H * HD, TE_KH * HD, TE_KH * HD], 1))
        o = _attention64(_rope64(_rms64(q, p["qn"]), cs), _rope64(_rms64(k, p["kn"]), cs), v, causal=True)
        x = x + o.reshape(n, TE_H * HD) @ _f64(p["o"]).T
        h = _rms64(x, p["ln2"])
        gate = h @ _f64(p["gate"]).T
        x = x + (gate * torch.sigmoid(gate) * (h @ _f64(p["up"]).T)) @ _f64(p["down"]).T
    return _rms64(x, t["norm"]), x


def _conv64(x, w, bias):
    """3 x 3 convolution with zero padding: x [h, w, cin], w [cout, 9 * cin]."""
    h, wd, cin = x.shape
    pad = torch.zeros((h + 2, wd + 2, cin), dtype=torch.float64, device=x.device)
    pad[1:-1, 1:-1] = x
    w = _f64(w).reshape(-1, 9, cin)
    y = _f64(bias).expand(h, wd, -1).clone()
    for tap in range(9):
        y += pad[tap // 3:tap // 3 + h, tap % 3:tap % 3 + wd] @ w[:, tap].T
    return y


def _channel_norm64(x, gamma):
    y = x * math.sqrt(x.shape[-1]) / x.norm(dim=-1, keepdim=True).clamp_min(1e-12) * _f64(gamma)
    return y * torch.sigmoid(y)


def _exact_vae_stage(case, seed):
    t = _vae_stage_inputs(case, seed)
    x = _f64(t["x"]).reshape(case["h"], case["w"], case["c"])
    a = _conv64(_channel_norm64(x, t["n1"]), t["c1"], t["b1"])
    x = x + _conv64(_channel_norm64(a, t["n2"]), t["c2"], t["b2"])
    out = x.reshape(-1, case["c"])
    if not case["up"]:
        return out
    y = _conv64(x.repeat_interleave(2, 0).repeat_interleave(2, 1), t["cu"], t["bu"])
    return out, y.reshape(-1, case["c"] // 2)


def _exact_vae_attn(case, seed):
    n = case["h"] * case["w"]
    q, k, v = _f64(_vae_attn_inputs(case, seed)["qkv"]).reshape(1, n, 3, 1, VAE_C).unbind(2)
    return _attention64(q, k, v).reshape(n, VAE_C)


def _exact_time_cond(case, seed):
    t, r, parts = _time_cond_inputs(case, seed), case["lora"], 3 * BLOCKS
    x = _f64(t["t"])
    h = x @ _f64(t["t1"]).T
    low = (h * torch.sigmoid(h)) @ _f64(t["t2"]).T
    e = _rms64(x, t["tn"])
    e = e * torch.sigmoid(e)
    h1 = (e @ _f64(t["w1"]).T).reshape(parts + 1, RANK_MOD, 1)
    if r:
        a = (_f64(t["a1"]) @ e.T).reshape(parts + 1, r, 1)
        h1 = h1 + _f64(t["b1"]).reshape(parts + 1, RANK_MOD, r) @ a
    every = (_f64(t["w2"]).reshape(parts, 3 * D, RANK_MOD) @ h1[:parts])[..., 0] + low
    final = (_f64(t["wf"]) @ h1[parts]).T + low[:, :2 * D]
    if r:
        a = _f64(t["a2"]).reshape(parts, r, RANK_MOD) @ h1[:parts]
        every = every + (_f64(t["b2"]).reshape(parts, 3 * D, r) @ a)[..., 0]
    return every, final


def exact(case, seed):
    kind = case["kind"]
    return {"block": _exact_block, "self": _exact_block, "cross": _exact_block, "mlp": _exact_block, "attn": _exact_attn,
            "text": _exact_text, "vae_stage": _exact_vae_stage, "vae_attn": _exact_vae_attn,
            "time_cond": _exact_time_cond}[kind](case, seed)
