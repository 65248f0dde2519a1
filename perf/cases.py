"""Performance cases of the DiT hot path, one call of the package's public entry points each.

The work a program has this package do: the linears of Flux and Z-Image blocks
(GGUF Q4_K / Q8_0 weights times f32 / f16 / bf16 activations), non-causal
attention, LoRA-adapted linears, and the composed Z-Image block and Flux
denoising step. Shapes are the models' (hidden 3072 or 3840, head_dim 128) at
image sizes from 256 x 256 to 1024 x 1024 with the text tokens in front, so
token counts run from one (the modulation projections) to 4608 and are ragged
wherever the prompt is.

A case is a dict of plain values; `prepare` makes its inputs on the GPU from
the seed alone, `run` is one pass, `exact` the same result in 64 bits by plain
torch.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llm-runner_amd"))

from llmr_amd import dit, glue, ops  # noqa: E402
from llmr_amd.gguf import GGML_Q4_K, GGML_Q8_0, row_bytes  # noqa: E402

DEV = "cuda"
HEAD = 128
WTYPES = {"q4_k": GGML_Q4_K, "q8_0": GGML_Q8_0}
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}

# (out_dim, in_dim) of the models' linears
FLUX = [(3072, 3072), (9216, 3072), (12288, 3072), (21504, 3072), (3072, 12288), (3072, 15360), (3072, 4096)]
ZIMAGE = [(3840, 3840), (11520, 3840), (10240, 3840), (3840, 10240)]


def listed():
    return [
        # a block's modulation vectors: one token through a whole weight, once per block and step
        {"name": "modulation", "kind": "linear", "w": "q4_k", "x": "f32", "tokens": 1, "out": 18432, "in": 3072},
        # a short prompt's text projection into the residual stream
        {"name": "text_in_77", "kind": "linear", "w": "q4_k", "x": "bf16", "tokens": 77, "out": 3072, "in": 4096},
        # the single Q8_0 linear of 256 tokens with the reference's f32 activations
        {"name": "q8_linear_256", "kind": "linear", "w": "q8_0", "x": "f32", "tokens": 256, "out": 3072, "in": 3072},
        # a Z-Image output projection at 512 x 512 (1024 image tokens and a prompt of 77), f32 buffers as a C caller has
        {"name": "o_proj_1101", "kind": "linear", "w": "q8_0", "x": "f32", "tokens": 1101, "out": 3840, "in": 3840},
        # Flux linear1 (Q | K | V | MLP-in) at 512 x 512 with 512 text tokens, and at 1024 x 1024
        {"name": "linear1_1536", "kind": "linear", "w": "q4_k", "x": "bf16", "tokens": 1536, "out": 21504, "in": 3072},
        {"name": "linear1_4608", "kind": "linear", "w": "q4_k", "x": "bf16", "tokens": 4608, "out": 21504, "in": 3072},
        # a Z-Image FFN's gate and up projections at 512 x 512
        {"name": "swiglu_1101", "kind": "swiglu", "x": "bf16", "tokens": 1101, "out": 10240, "in": 3840},
        # attention of a Z-Image block at 512 x 512 from f32 buffers, and of a Flux block at 1024 x 1024
        {"name": "attention_1101", "kind": "attention", "x": "f32", "heads": 30, "tokens": 1101},
        {"name": "attention_4608", "kind": "attention", "x": "f16", "heads": 24, "tokens": 4608},
        # a QKV projection with a LoRA adapter at 512 x 512
        {"name": "lora_1536", "kind": "lora", "w": "q4_k", "x": "bf16", "tokens": 1536, "out": 9216, "in": 3072,
         "rank": 32},
        # a whole Z-Image block at 512 x 512
        {"name": "zimage_block_1101", "kind": "zimage", "tokens": 1101},
        # one whole denoising step of the full Flux model at 1024 x 1024, 512 text tokens
        {"name": "flux_step_1024", "kind": "flux", "latent_h": 128, "latent_w": 128, "text": 512},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "vector", "swiglu", "attention", "attention", "lora", "zimage",
                       "flux"])
    x = rng.choice(["f32", "f16", "bf16", "bf16"])
    if kind == "vector":  # the modulation and timestep projections
        n, k = rng.choice([(18432, 3072), (9216, 3072), (6144, 3072), (3072, 3072), (3072, 256), (11520, 3840)])
        return {"kind": "linear", "w": "q4_k" if k % 256 == 0 and rng.random() < 0.75 else "q8_0", "x": "f32",
                "tokens": rng.randint(1, 4), "out": n, "in": k}
    if kind == "linear":
        w = rng.choice(["q4_k", "q8_0"])
        n, k = rng.choice(FLUX if w == "q4_k" else FLUX + ZIMAGE)
        return {"kind": "linear", "w": w, "x": x, "tokens": _log(rng, 5, 4608), "out": n, "in": k}
    if kind == "swiglu":
        return {"kind": "swiglu", "x": x, "tokens": _log(rng, 77, 4352), "out": 10240, "in": 3840}
    if kind == "attention":
        return {"kind": "attention", "x": x, "heads": rng.choice([24, 30]), "tokens": _log(rng, 77, 4608)}
    if kind == "lora":
        n, k = rng.choice(FLUX[:4])
        return {"kind": "lora", "w": rng.choice(["q4_k", "q8_0"]), "x": x, "tokens": _log(rng, 256, 4608), "out": n,
                "in": k, "rank": rng.choice([4, 8, 16, 32, 64, 128])}
    if kind == "zimage":
        return {"kind": "zimage", "tokens": _log(rng, 333, 4352)}
    return {"kind": "flux", "latent_h": 2 * rng.randint(16, 64), "latent_w": 2 * rng.randint(16, 64),
            "text": 4 * rng.randint(19, 128)}


# ---- inputs -------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, std=1.0, mean=0.0, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device=DEV).mul_(std).add_(mean).to(dtype)


def _q8_0(g, rows, cols, std=0.02):
    """Raw Q8_0 blocks of a random [rows, cols] weight: f16 scale amax / 127, then 32 int8 (halves away from zero)."""
    v = _randn(g, rows * cols // 32, 32, std=std)
    d = v.abs().amax(dim=1, keepdim=True) / 127.0
    q = (v / d).abs().add_(0.5).floor_().clamp_(max=127).mul_(v.sign()).to(torch.int8)
    return torch.cat([d.half().view(torch.uint8), q.view(torch.uint8)], dim=1).reshape(-1)


def _weight(g, seed, stream, w, rows, cols):
    if w == "q8_0":
        return _q8_0(g, rows, cols)
    return glue.synth_q4k(rows, cols, stream, 0.02, seed, DEV)


def _tensor(blocks, w, rows, cols):
    return ops.Tensor.quantized(blocks, WTYPES[w], rows, cols)


def _rope(g_positions, axes, theta):
    """cos, sin f32 [S, 64] of per-token positions [S, 3]."""
    cos, sin = [], []
    for a, dims in enumerate(axes):
        freq = theta ** (-torch.arange(0, dims, 2, device=DEV, dtype=torch.float64) / dims)
        ang = g_positions[:, a].double()[:, None] * freq[None, :]
        cos.append(ang.cos())
        sin.append(ang.sin())
    return torch.cat(cos, 1).float().contiguous(), torch.cat(sin, 1).float().contiguous()


def _inputs(case, seed):
    """The tensors of a case (no output buffers)."""
    g, kind, s = _gen(seed), case["kind"], {}
    if kind in ("linear", "lora", "swiglu"):
        M, N, K = case["tokens"], case["out"], case["in"]
        s["x"] = _randn(g, M, K, dtype=DTYPES[case["x"]])
        if kind == "swiglu":
            s["w"], s["w2"] = _q8_0(g, N, K), _q8_0(g, N, K)
        else:
            s["w"] = _weight(g, seed, 7, case["w"], N, K)
        if kind == "lora":
            s["a"] = _randn(g, case["rank"], K, std=0.02)
            s["b"] = _randn(g, N, case["rank"], std=0.02)
    elif kind == "attention":
        # head-normed Q and K have rows of unit mean square; a rotation leaves them so
        for n in "qkv":
            s[n] = _randn(g, case["heads"], case["tokens"], HEAD, dtype=DTYPES[case["x"]])
    elif kind == "zimage":
        S, d, f = case["tokens"], 3840, 10240
        gu = torch.cat([_q8_0(g, f, d), _q8_0(g, f, d)])
        half = gu.numel() // 2

        def vec(n, mean=1.0, std=0.1):
            return _randn(g, n, std=std, mean=mean)

        s["weights"] = dit.ZImageLayerWeights(
            wqkv=_q8_0(g, 3 * d, d), wo=_q8_0(g, d, d), w_gate=gu[:half], w_up=gu[half:], w_down=_q8_0(g, d, f),
            attn_norm1=vec(d), attn_norm2=vec(d), ffn_norm1=vec(d), ffn_norm2=vec(d), q_norm=vec(HEAD),
            k_norm=vec(HEAD), adaln=vec(4 * d, 0.0, 0.5).reshape(4, d), w_gate_up=gu)
        s["hidden0"] = _randn(g, S, d)
        # text tokens first, then image rows 32 wide
        i = torch.arange(S, device=DEV)
        img = (i - (S % 256)).clamp(min=0)
        s["cos"], s["sin"] = _rope(torch.stack([i, img // 32, img % 32], 1), (32, 48, 48), 256.0)
    else:
        cfg = dit.FluxConfig(n_txt=case["text"], latent_h=case["latent_h"], latent_w=case["latent_w"])
        s["cfg"] = cfg
        s["weights"] = dit.flux_weights(cfg, DEV, seed)
        s["latent"] = _randn(g, cfg.latent_ch, cfg.latent_h, cfg.latent_w)
        s["txt"] = _randn(g, cfg.n_txt, cfg.text_dim, dtype=torch.bfloat16)
        s["sigma"] = 0.25 + (seed % 97) / 200.0
    return s


def prepare(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    g = s["g"] = ops.default_graph()
    s["case"] = case
    if kind in ("linear", "lora", "swiglu"):
        M, N, K = case["tokens"], case["out"], case["in"]
        s["y"] = torch.empty(M, N, dtype=torch.float32, device=DEV)
        s["X"], s["Y"] = ops.Tensor.from_torch(s["x"]), ops.Tensor.from_torch(s["y"])
        s["W"] = _tensor(s["w"], case.get("w", "q8_0"), N, K)
        if kind == "swiglu":
            s["W2"] = _tensor(s["w2"], "q8_0", N, K)
        if kind == "lora":
            s["lora"] = ops.LoraTensor(s["a"], s["b"], case["rank"], 1.0)
            s["scratch"] = torch.empty(M * case["rank"], dtype=torch.float32, device=DEV)
    elif kind == "attention":
        H, S = case["heads"], case["tokens"]
        s["Q"], s["K"], s["V"] = (ops.Tensor.from_torch(s[n]) for n in "qkv")
        s["y"] = torch.empty(S, H * HEAD, dtype=torch.float32, device=DEV)
        s["Y"] = ops.Tensor.from_torch(s["y"])
        s["pc"] = ops.FlashAttentionPC(HEAD, H, S, 1.0 / math.sqrt(HEAD))
    elif kind == "zimage":
        s["block"] = dit.ZImageBlock(3840, 30, 10240, case["tokens"], torch.bfloat16, DEV, g)
        s["hidden"] = torch.empty_like(s["hidden0"])
    else:
        s["model"] = dit.FluxDiT(s["cfg"], *s["weights"], act_dtype=torch.bfloat16, device=DEV, g=g)
    return s


def run(s):
    case = s["case"]
    kind, g = case["kind"], s["g"]
    if kind == "linear":
        ops.dispatch_batch_matmul(g, s["W"], s["X"], s["Y"], case["out"], case["in"], case["tokens"], 0)
        return s["y"]
    if kind == "swiglu":
        ops.dispatch_batch_matmul_swiglu(g, s["W"], s["W2"], s["X"], s["Y"], case["out"], case["in"], case["tokens"])
        return s["y"]
    if kind == "lora":
        ops.dispatch_batch_matmul(g, s["W"], s["X"], s["Y"], case["out"], case["in"], case["tokens"], 0, s["lora"],
                                  s["scratch"])
        return s["y"]
    if kind == "attention":
        ops.dispatch_flash_attention(g, s["Q"], s["K"], s["V"], s["Y"], s["pc"])
        return s["y"]
    if kind == "zimage":  # the block updates the residual stream in place
        s["hidden"].copy_(s["hidden0"])
        return s["block"].forward(s["weights"], s["hidden"], s["cos"], s["sin"])
    return s["model"].forward(s["latent"], s["txt"], s["sigma"])


# ---- what a pass cannot do without ----------------------------------------------


def work(case):
    kind = case["kind"]
    if kind in ("linear", "lora", "swiglu"):
        M, N, K = case["tokens"], case["out"], case["in"]
        n = 2 if kind == "swiglu" else 1
        b = n * N * row_bytes(WTYPES[case.get("w", "q8_0")], K) + M * K * SIZE[case["x"]] + 4 * M * N
        f = 2.0 * n * M * N * K
        if kind == "lora":
            b += 4 * case["rank"] * (N + K)
            f += 2.0 * M * case["rank"] * (N + K)
        return {"bytes": b, "flops": f}
    if kind == "attention":
        H, S = case["heads"], case["tokens"]
        return {"bytes": H * S * HEAD * (3 * SIZE[case["x"]] + 4), "flops": 4.0 * H * S * S * HEAD}
    if kind == "zimage":
        S, d, f = case["tokens"], 3840, 10240
        elems = 4 * d * d + 3 * d * f
        return {"bytes": elems // 32 * 34 + 2 * 4 * S * d, "flops": 2.0 * S * elems + 4.0 * 30 * S * S * HEAD}
    cfg = dit.FluxConfig(n_txt=case["text"], latent_h=case["latent_h"], latent_w=case["latent_w"])
    d, m = cfg.dim, cfg.mlp
    double = 2 * (6 * d * d + 4 * d * d + 2 * m * d)
    single = 3 * d * d + (3 * d + m) * d + d * (d + m)
    elems = cfg.n_double * double + cfg.n_single * single + cfg.text_dim * d + 3 * d * d
    mods = 2.0 * d * d * (12 * cfg.n_double + 3 * cfg.n_single)
    return {"bytes": elems // 256 * 144 + 2 * cfg.n_txt * cfg.text_dim, "flops": cfg.gemm_flops() + mods}


def tolerance(case):
    """About four times the relative error against 64 bits that the operand
    types give: weights and activations rounded to bf16 (2^-9 / sqrt 3 each)
    or fp16 (2^-12 / sqrt 3), sums in f32."""
    kind = case["kind"]
    if kind == "attention":
        # Q, K, V and the softmax weights in fp16
        return {"rel": 2e-3}
    if kind in ("zimage", "flux"):
        # bf16 activations through a block / 57 blocks
        return {"rel": 1e-2 if kind == "zimage" else 2.5e-2}
    if kind == "linear" and case["w"] == "q4_k" and case["tokens"] <= 4:
        return {"rel": 1e-5}  # the weight and the f32 activations are not rounded
    half = case["x"] == "f16" or (case["x"] == "f32" and kind != "swiglu" and case["w"] == "q8_0")
    return {"rel": 2e-3 if half else 1e-2}


# ---- the same in 64 bits --------------------------------------------------------


def _dequant(blocks, w, rows, cols):
    """f64 [rows, cols] of raw GGUF blocks."""
    if w == "q8_0":
        b = blocks.view(-1, 34)
        d = b[:, :2].contiguous().view(torch.float16).double()
        return (b[:, 2:].contiguous().view(torch.int8).double() * d).view(rows, cols)
    out = torch.empty(rows, cols, dtype=torch.float64, device=DEV)
    step = max(1, (1 << 27) // cols)
    rb = cols // 256 * 144
    for r in range(0, rows, step):
        b = blocks.view(rows, rb)[r:r + step].reshape(-1, 144)
        d = b[:, 0:2].contiguous().view(torch.float16).double()
        dmin = b[:, 2:4].contiguous().view(torch.float16).double()
        s = b[:, 4:16].to(torch.int32)
        lo, mid, hi = s[:, 0:4], s[:, 4:8], s[:, 8:12]
        sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1).double()
        mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1).double()
        q = b[:, 16:].reshape(-1, 4, 32)
        q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()  # sub-blocks 2j (low) and 2j + 1 (high)
        out[r:r + step] = (q * (d * sc)[:, :, None] - (dmin * mn)[:, :, None]).view(-1, cols)
    return out


def _mm(x, blocks, w, rows, cols):
    return x.double() @ _dequant(blocks, w, rows, cols).t()


def _attention(q, k, v):
    """[H, S, 128] -> [S, H * 128] in 64 bits."""
    H, S, D = q.shape
    out = torch.empty(S, H * D, dtype=torch.float64, device=DEV)
    for h in range(H):
        p = torch.softmax((q[h].double() @ k[h].double().t()) / math.sqrt(D), dim=-1)
        out[:, h * D:(h + 1) * D] = p @ v[h].double()
    return out


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _layernorm(x, shift, scale, eps=1e-6):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * (1 + scale) + shift


def _heads(x, norm, H, eps, rope=None):
    """Rows [S, H * 128] -> head-normed, rotated [H, S, 128]."""
    x = x.view(x.shape[0], H, HEAD).transpose(0, 1)
    if norm is not None:
        x = _rms(x, norm.double(), eps)
    if rope is not None:
        c, s = rope[0].double(), rope[1].double()
        a, b = x[..., 0::2], x[..., 1::2]
        x = torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)
    return x


def _silu(x):
    return x / (1 + torch.exp(-x))


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(0.7978845608 * (x + 0.044715 * x ** 3)))


def _exact_zimage(s):
    w, h, eps, d, f, H = s["weights"], s["hidden0"].double(), 1e-5, 3840, 10240, 30
    rope = (s["cos"], s["sin"])
    ad = w.adaln.double()
    qkv = _mm(_rms(h, w.attn_norm1.double(), eps) * (1 + ad[0]), w.wqkv, "q8_0", 3 * d, d)
    o = _attention(_heads(qkv[:, :d], w.q_norm, H, eps, rope), _heads(qkv[:, d:2 * d], w.k_norm, H, eps, rope),
                   _heads(qkv[:, 2 * d:], None, H, eps))
    h = h + torch.tanh(ad[1]) * _rms(_mm(o, w.wo, "q8_0", d, d), w.attn_norm2.double(), eps)
    a = _rms(h, w.ffn_norm1.double(), eps) * (1 + ad[2])
    t = _silu(_mm(a, w.w_gate, "q8_0", f, d)) * _mm(a, w.w_up, "q8_0", f, d)
    return h + torch.tanh(ad[3]) * _rms(_mm(t, w.w_down, "q8_0", d, f), w.ffn_norm2.double(), eps)


def _exact_flux(s):
    cfg, (glob, doubles, singles) = s["cfg"], s["weights"]
    d, m, H, nt, p, C = cfg.dim, cfg.mlp, cfg.n_heads, cfg.n_txt, cfg.patch, cfg.latent_ch
    gh, gw, eps = cfg.latent_h // p, cfg.latent_w // p, 1e-6

    def mm(x, w, n, k, wt="q4_k"):
        return _mm(x, w, wt, n, k)

    pos = torch.zeros(cfg.seq, 3, device=DEV, dtype=torch.int64)
    i = torch.arange(cfg.n_img, device=DEV)
    pos[nt:, 1], pos[nt:, 2] = i // gw, i % gw
    rope = _rope(pos, cfg.axes, cfg.theta)
    patches = s["latent"].double().view(C, gh, p, gw, p).permute(1, 3, 2, 4, 0).reshape(cfg.n_img, C * p * p)
    h = torch.cat([mm(s["txt"], glob.txt_in, d, cfg.text_dim), mm(patches, glob.img_in, d, cfg.patch_dim, "q8_0")])
    half = cfg.t_emb_dim // 2
    ang = s["sigma"] * 1000.0 * torch.exp(-math.log(10000.0) * torch.arange(half, device=DEV).double() / half)
    vec = mm(torch.cat([ang.cos(), ang.sin()])[None], glob.time_in0, d, cfg.t_emb_dim)
    vec = _silu(mm(_silu(vec), glob.time_in1, d, d))

    def mod(w, n):
        return mm(vec, w, n * d, d).view(n, d)

    for w in doubles:
        parts = [(h[:nt], mod(w.txt_mod, 6), w.txt_qkv, w.txt_proj, w.txt_mlp0, w.txt_mlp2, w.txt_q_norm, w.txt_k_norm),
                 (h[nt:], mod(w.img_mod, 6), w.img_qkv, w.img_proj, w.img_mlp0, w.img_mlp2, w.img_q_norm, w.img_k_norm)]
        qs, ks, vs = [], [], []
        for (x, mo, wqkv, _, _, _, qn, kn), sl in zip(parts, (slice(0, nt), slice(nt, None))):
            qkv = mm(_layernorm(x, mo[0], mo[1]), wqkv, 3 * d, d)
            r = (rope[0][sl], rope[1][sl])
            qs.append(_heads(qkv[:, :d], qn, H, eps, r))
            ks.append(_heads(qkv[:, d:2 * d], kn, H, eps, r))
            vs.append(_heads(qkv[:, 2 * d:], None, H, eps))
        o = _attention(torch.cat(qs, 1), torch.cat(ks, 1), torch.cat(vs, 1))
        new = []
        for (x, mo, _, wp, w0, w2, _, _), sl in zip(parts, (slice(0, nt), slice(nt, None))):
            x = x + mo[2] * mm(o[sl], wp, d, d)
            new.append(x + mo[5] * mm(_gelu(mm(_layernorm(x, mo[3], mo[4]), w0, m, d)), w2, d, m))
        h = torch.cat(new)
    for w in singles:
        mo = mod(w.mod, 3)
        y = mm(_layernorm(h, mo[0], mo[1]), w.linear1, 3 * d + m, d)
        o = _attention(_heads(y[:, :d], w.q_norm, H, eps, rope), _heads(y[:, d:2 * d], w.k_norm, H, eps, rope),
                       _heads(y[:, 2 * d:3 * d], None, H, eps))
        h = h + mo[2] * mm(torch.cat([o, _gelu(y[:, 3 * d:])], 1), w.linear2, d, d + m)
    fm = mod(glob.final_mod, 2)
    vel = mm(_layernorm(h[nt:], fm[0], fm[1]), glob.final_linear, cfg.patch_dim, d)
    return vel.view(gh, gw, p, p, C).permute(4, 0, 2, 1, 3).reshape(C, cfg.latent_h, cfg.latent_w)


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "attention":
        return _attention(s["q"], s["k"], s["v"])
    if kind == "zimage":
        return _exact_zimage(s)
    if kind == "flux":
        return _exact_flux(s)
    N, K = case["out"], case["in"]
    if kind == "swiglu":
        return _silu(_mm(s["x"], s["w"], "q8_0", N, K)) * _mm(s["x"], s["w2"], "q8_0", N, K)
    y = _mm(s["x"], s["w"], case["w"], N, K)
    if kind == "lora":
        y += (s["x"].double() @ s["a"].double().t()) @ s["b"].double().t()
    return y
