"""The work this package is measured by: calls of its public entry points at the sizes its users run.

Every case is one pass of a user's program: an attention call with its tangent (a consistency-distillation step), one
without (sampling), one with its backward pass (training), the text cross-attention in the same three uses, the RMSNorm +
rotary step around them, a whole DiT block in its three modes, and a whole network sampling one image.

Sizes come from the 2B (16 heads) and 14B (40 heads) DiT with head dim 128: latent frames of 30 x 52 tokens (480p) and
44 x 80 tokens (720p), 1 to 24 of them, text of 512 tokens of 1024 channels; `draw` covers the ranges in between, ragged
sizes among them.
"""
import importlib
import math
import random

import torch

import __graft_entry__

D = 128                      # head dim of every DiT configuration
TEXT = 512                   # text tokens a network call is given
TEXT_DIM = 1024              # their channels after the network's own projection
LORA = 256                   # adaLN-LoRA rank
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
MAX_FLOPS = 1.75e14          # of the largest listed case; drawn ones stay below

_pkg = None


def package():
    global _pkg
    if _pkg is None:
        _pkg = __graft_entry__.load_package()
    return _pkg


def listed():
    return [
        # one distillation step's self-attention with all tangents: the largest call there is (720p, 24 latent frames)
        {"name": "jvp_720p", "kind": "attention_jvp", "B": 1, "H": 16, "L": 84480, "dtype": "bf16"},
        # the same for one 480p image (one latent frame)
        {"name": "jvp_image", "kind": "attention_jvp", "B": 1, "H": 16, "L": 1560, "dtype": "bf16"},
        # sampling: self-attention of a 480p video, and the smallest call, two images of 16 x 16 tokens less one (ragged), fp16
        {"name": "forward_480p", "kind": "attention", "B": 1, "H": 16, "L": 37440, "dtype": "bf16"},
        {"name": "forward_small", "kind": "attention", "B": 2, "H": 16, "L": 255, "dtype": "fp16"},
        # training: self-attention forward and backward, seven latent frames at 720p
        {"name": "train_720p_short", "kind": "attention_train", "B": 1, "H": 16, "L": 24640, "dtype": "bf16"},
        # text cross-attention of a distillation step: padded text, only the queries move
        {"name": "cross_jvp", "kind": "cross_jvp", "B": 2, "H": 16, "L": 37440, "text": 512, "dtype": "bf16"},
        # text cross-attention in training
        {"name": "cross_train", "kind": "cross_train", "B": 1, "H": 16, "L": 37440, "text": 512, "dtype": "bf16"},
        # RMSNorm + rotary embedding of the queries in training, 14B width
        {"name": "norm_rope_train", "kind": "norm_rope_train", "B": 1, "H": 40, "T": 16, "Hh": 30, "W": 52, "dtype": "bf16"},
        # one transformer block: sampling at 480p, with a tangent at 720p (a short clip), training step at 480p (a short clip)
        {"name": "block_forward", "kind": "block", "B": 1, "H": 16, "T": 24, "Hh": 30, "W": 52},
        {"name": "block_jvp", "kind": "block_jvp", "B": 1, "H": 16, "T": 5, "Hh": 44, "W": 80},
        {"name": "block_train", "kind": "block_train", "B": 1, "H": 16, "T": 7, "Hh": 30, "W": 52},
        # one sampling step of the whole 2B network on one 720p image
        {"name": "network_image", "kind": "network", "B": 1, "H": 16, "T": 1, "Hh": 44, "W": 80, "blocks": 28},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["attention_jvp", "attention", "attention_train", "cross_jvp", "cross_train", "norm_rope_jvp",
                       "norm_rope_train", "block", "block_jvp", "block_train", "network"])
    while True:
        c = {"kind": kind, "B": rng.choice([1, 1, 2]), "H": rng.choice([16, 16, 40])}
        if kind in ("attention_jvp", "attention", "attention_train"):
            c["L"] = _log_int(rng, 255, 84480)
            c["dtype"] = rng.choice(["bf16", "bf16", "bf16", "fp16"])
        elif kind in ("cross_jvp", "cross_train"):
            c["L"] = _log_int(rng, 1560, 84480)
            c["text"] = rng.choice([512, rng.randint(64, 511)])
            c["dtype"] = rng.choice(["bf16", "bf16", "bf16", "fp16"])
        else:     # a grid of tokens: frames x height x width
            c["T"] = rng.choice([1, rng.randint(1, 24)])
            c["Hh"], c["W"] = rng.choice([(30, 52), (44, 80), (32, 32), (rng.randint(12, 44), rng.randint(12, 80))])
            if kind.startswith("norm_rope"):
                c["dtype"] = rng.choice(["bf16", "bf16", "bf16", "fp16"])
            if kind == "network":
                c["H"], c["blocks"] = 16, rng.choice([28, rng.randint(2, 27)])
                c["T"] = rng.randint(1, 3)
        # (a backward pass runs at about 0.7 of the forward's rate)
        if _flops(c) * (1.4 if kind.endswith("_train") else 1.0) <= MAX_FLOPS and c["B"] * c.get("L", 0) <= 84480:
            return c


# ------------------------------------------------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, shape, dtype, std=1.0):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std).to(dtype)


def _unit_rms(g, shape, dtype):
    """Queries and keys as attention meets them: normalised per head."""
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    return (x * torch.rsqrt(x.pow(2).mean(dim=-1, keepdim=True) + 1e-6)).to(dtype)


def _angles(pkg, T, Hh, W):
    pe = pkg.VideoRopePosition3DEmb(head_dim=D, len_h=Hh, len_w=W, len_t=T, enable_fps_modulation=False).to("cuda")
    return pe.generate_embeddings((1, T, Hh, W, D))


def _fill(module, g, gates):
    """Weights of a trained module: every matrix normal with std 1 / sqrt(fan in), norm weights near one, the modulation's
    last layers of size `gates` (a freshly initialised block has them at zero)."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if p.dim() == 2:
                last = "adaln_modulation" in name and name.endswith(".2.weight")
                p.copy_(torch.randn(p.shape, generator=g, device="cuda", dtype=torch.float32) * (gates if last else p.shape[1] ** -0.5))
            elif "norm" in name:
                p.copy_(1.0 + 0.1 * torch.randn(p.shape, generator=g, device="cuda"))
            else:
                p.zero_()


def prepare(case, seed):
    pkg, g, kind = package(), _generator(seed), case["kind"]
    B, H = case["B"], case["H"]
    s = {"kind": kind, "pkg": pkg}
    if kind == "attention_jvp":                          # heads first, as the distillation call takes them
        dt, shape = DTYPES[case["dtype"]], (B, H, case["L"], D)
        s["in"] = [_unit_rms(g, shape, dt), _unit_rms(g, shape, dt), _normal(g, shape, dt)] + [_normal(g, shape, dt, 0.1) for _ in range(3)]
    elif kind in ("attention", "attention_train"):       # [B, S, H, D], as the blocks call it
        dt, shape = DTYPES[case["dtype"]], (B, case["L"], H, D)
        s["in"] = [_unit_rms(g, shape, dt), _unit_rms(g, shape, dt), _normal(g, shape, dt)]
        s["dtype"] = dt
        if kind == "attention_train":
            s["dout"] = _normal(g, shape, dt)
    elif kind == "cross_jvp":
        dt, q_shape, k_shape = DTYPES[case["dtype"]], (B, H, case["L"], D), (B, H, case["text"], D)
        s["in"] = [_unit_rms(g, q_shape, dt), _unit_rms(g, k_shape, dt), _normal(g, k_shape, dt), _normal(g, q_shape, dt, 0.1)]
        s["lens"] = torch.tensor(_key_lens(case), dtype=torch.int32, device="cuda")
    elif kind == "cross_train":
        dt, q_shape, k_shape = DTYPES[case["dtype"]], (B, case["L"], H, D), (B, case["text"], H, D)
        s["in"] = [_unit_rms(g, q_shape, dt), _unit_rms(g, k_shape, dt), _normal(g, k_shape, dt)]
        s["dtype"], s["dout"] = dt, _normal(g, q_shape, dt)
    elif kind in ("norm_rope_jvp", "norm_rope_train"):
        dt = DTYPES[case["dtype"]]
        shape = (B, case["T"] * case["Hh"] * case["W"], H, D)
        s["x"], s["other"] = _normal(g, shape, dt), _normal(g, shape, dt, 0.1)     # and the tangent, or the gradient
        s["weight"] = 1.0 + 0.1 * torch.randn(D, generator=g, device="cuda")
        s["angles"] = _angles(pkg, case["T"], case["Hh"], case["W"])
    elif kind in ("block", "block_jvp", "block_train"):
        K, grid = H * D, (B, case["T"], case["Hh"], case["W"])
        with torch.device("cuda"):
            m = pkg.Block(K, TEXT_DIM, H, mlp_ratio=4.0, use_adaln_lora=True, adaln_lora_dim=LORA)
        _fill(m, g, 1.0 / 16.0)
        m = m.to(dtype=torch.bfloat16)
        s["block"] = m.train() if kind == "block_train" else m.eval()
        s["x"], s["emb"] = _normal(g, (*grid, K), torch.bfloat16), _normal(g, (B, case["T"], K), torch.bfloat16)
        s["lora"], s["text"] = _normal(g, (B, case["T"], 3 * K), torch.bfloat16, 0.3), _normal(g, (B, TEXT, TEXT_DIM), torch.bfloat16)
        s["angles"] = _angles(pkg, case["T"], case["Hh"], case["W"])
        if kind == "block_jvp":
            s["tx"], s["temb"] = _normal(g, (*grid, K), torch.bfloat16, 0.1), _normal(g, (B, case["T"], K), torch.bfloat16, 0.1)
            s["tlora"] = _normal(g, (B, case["T"], 3 * K), torch.bfloat16, 0.03)
        if kind == "block_train":
            s["dout"] = _normal(g, (*grid, K), torch.bfloat16)
            s["x"].requires_grad_(True)
    elif kind == "network":                              # text to image / short clip, x [B, 16, T, H, W] latents
        frame = (2 * case["Hh"], 2 * case["W"])
        with torch.device("cuda"):
            torch.set_default_dtype(torch.bfloat16)
            try:
                net = pkg.MiniTrainDIT(max_img_h=240, max_img_w=240, max_frames=128, in_channels=16, out_channels=16, patch_spatial=2,
                                       patch_temporal=1, model_channels=H * D, num_blocks=case["blocks"], num_heads=H,
                                       concat_padding_mask=True, use_adaln_lora=True, adaln_lora_dim=LORA, crossattn_emb_channels=TEXT_DIM)
            finally:
                torch.set_default_dtype(torch.float32)
        _fill(net, g, 1.0 / 64.0)
        s["net"] = net.to(dtype=torch.bfloat16).eval()
        s["x"] = _normal(g, (B, 16, case["T"], *frame), torch.bfloat16)
        s["time"] = torch.full((B, 1), 0.6, device="cuda", dtype=torch.bfloat16)
        s["text"] = _normal(g, (B, TEXT, TEXT_DIM), torch.bfloat16)
        s["mask"] = torch.zeros(B, 1, *frame, device="cuda", dtype=torch.bfloat16)
        s["fps"] = torch.full((B,), 16.0, device="cuda")
    else:
        raise ValueError(kind)
    return s


def _key_lens(case):
    """Valid text lengths of the batch rows: from an eighth of the padded length to all of it, fixed by the case."""
    n = case["text"]
    return [random.Random(n * 131 + case["L"] + i).randint(max(1, n // 8), n) for i in range(case["B"])]


# ----------------------------------------------------------------------------------------------------------- one pass
def run(s):
    pkg, kind = s["pkg"], s["kind"]
    if kind == "attention_jvp":
        return pkg.attention_jvp(*s["in"])
    if kind == "attention":
        with torch.no_grad():
            return pkg.attention_forward(*s["in"], dtype=s["dtype"])
    if kind in ("attention_train", "cross_train"):
        q, k, v = (x.detach().requires_grad_(True) for x in s["in"])
        o = pkg.attention_forward(q, k, v, dtype=s["dtype"])
        return (o.detach(), *torch.autograd.grad(o, (q, k, v), s["dout"]))
    if kind == "cross_jvp":
        q, k, v, tq = s["in"]
        return pkg.attention_with_lse(q, k, v, tq, key_lens=s["lens"])
    if kind == "norm_rope_jvp":
        return pkg.norm_rope(s["x"], s["weight"], s["angles"], s["other"], out_layout="bhsd")
    if kind == "norm_rope_train":
        y, _ = pkg.norm_rope(s["x"], s["weight"], s["angles"], out_layout="bhsd")
        return (y, *pkg.norm_rope_bwd(s["x"], s["weight"], s["angles"], s["other"]))
    if kind == "block":
        with torch.no_grad():
            return s["block"](s["x"], s["emb"], s["text"], s["angles"], s["lora"])
    if kind == "block_jvp":
        return s["block"].forward_jvp(s["x"], s["tx"], s["emb"], s["temb"], s["text"], s["angles"], s["lora"], s["tlora"])
    if kind == "block_train":
        m, x = s["block"], s["x"]
        m.zero_grad(set_to_none=True)
        x.grad = None
        y = m(x, s["emb"], s["text"], s["angles"], s["lora"])
        y.backward(s["dout"])
        return {"y": y.detach(), "dx": x.grad, **{name: p.grad for name, p in m.named_parameters()}}
    with torch.no_grad():
        return s["net"](s["x"], s["time"], s["text"], fps=s["fps"], padding_mask=s["mask"])


# --------------------------------------------------------------------------------------------------------------- floor
def _gemms(rows, text_rows, K):
    """Products of one block's linear layers (forward, values only)."""
    return 2.0 * rows * K * K * (4 + 2 + 8) + 2.0 * text_rows * TEXT_DIM * K * 2


def _flops(c):
    kind, B, H = c["kind"], c["B"], c["H"]
    if kind.startswith("norm_rope"):
        return 0.0
    if kind in ("attention_jvp", "attention", "attention_train"):      # matrix products: 6, 2, 2 + 5
        return {"attention_jvp": 6, "attention": 2, "attention_train": 7}[kind] * 2.0 * B * H * c["L"] ** 2 * D
    if kind == "cross_jvp":                                            # 4 products over the valid keys
        return 4 * 2.0 * H * c["L"] * sum(_key_lens(c)) * D
    if kind == "cross_train":
        return 7 * 2.0 * B * H * c["L"] * c["text"] * D
    L = c["T"] * c["Hh"] * c["W"]
    gemms, one = _gemms(B * L, B * TEXT, H * D), 2.0 * B * H * L * D
    if kind == "block_jvp":
        return 2 * gemms + one * (6 * L + 4 * TEXT)
    if kind == "block_train":
        return 3 * gemms + 7 * one * (L + TEXT)
    return c.get("blocks", 1) * (gemms + 2 * one * (L + TEXT))


def _bytes(c):
    kind, B, H = c["kind"], c["B"], c["H"]
    if "L" in c:
        q, k = 2 * B * H * c["L"] * D, 2 * B * H * c.get("text", c["L"]) * D
        lse = 4 * B * H * c["L"]
        return {"attention_jvp": 4 * q + 4 * k, "attention": 2 * q + 2 * k, "attention_train": 4 * q + 4 * k,
                "cross_jvp": 4 * q + 2 * k + lse, "cross_train": 4 * q + 4 * k}[kind]
    L, K = c["T"] * c["Hh"] * c["W"], H * D
    x = 2 * B * L * K
    if kind.startswith("norm_rope"):            # x, tangent -> y, tangent | x, dy -> y, dx
        return 4 * x + 4 * L * D
    weights = 2 * (K * K * (4 + 2 + 8) + 2 * TEXT_DIM * K + 3 * LORA * 4 * K)
    if kind == "network":
        return c["blocks"] * weights + 2 * B * 2 * 16 * 4 * L
    return {"block": 2, "block_jvp": 4, "block_train": 4}[kind] * x + weights * (2 if kind == "block_train" else 1)


def work(case):
    return {"bytes": float(_bytes(case)), "flops": float(_flops(case))}


def tolerance(case):
    """Errors of another correct implementation at the same precision: about four times what a pass differs from one in 32
    bits on the same 16-bit inputs, relative-L2 / largest.  Measured: attention, RMSNorm + rotary and their gradients
    2.2e-3 - 2.9e-3 / 0.02 in bf16, 2.1e-4 - 3.6e-4 / 2.7e-3 in fp16 (8 times finer); a block 4.2e-3, its tangent 5.4e-3 / 0.05;
    a block's weight gradients 6e-3 - 1.2e-2 / 0.2; a network of 28 blocks 1.4e-2 / 0.06."""
    kind = case["kind"]
    if kind == "block_train":
        return {"rel": 3e-2, "max": 0.8}
    if kind == "network":
        return {"rel": 3e-2, "max": 0.25}
    if kind in ("block", "block_jvp"):
        return {"rel": 2e-2, "max": 0.2}
    return {"rel": 1.5e-3, "max": 0.0125} if case["dtype"] == "fp16" else {"rel": 1e-2, "max": 0.1}


# ---------------------------------------------------------------------------------------------------------- in 64 bits
ROWS = 4096                  # query rows worked on at once
EXACT_FLOPS = 4e13           # beyond that a pass in 64 bits takes too long


def _attend(q, k, v, tq=None, tk=None, tv=None, lens=None):
    """softmax(q k^T / sqrt(d)) v of [B, H, L, d] tensors in 64 bits, its tangent (None without tq) and the log-sum-exp."""
    scale = q.shape[-1] ** -0.5
    o, lse = torch.empty_like(q), torch.empty(q.shape[:-1], device=q.device, dtype=q.dtype)
    to = None if tq is None else torch.empty_like(q)
    for b in range(q.shape[0]):
        n = k.shape[2] if lens is None else int(lens[b])
        for h in range(q.shape[1]):
            kk, vv = k[b, h, :n], v[b, h, :n]
            for r in range(0, q.shape[2], ROWS):
                i = (b, h, slice(r, r + ROWS))
                p = (q[i] @ kk.T).mul_(scale)
                lse[i] = torch.logsumexp(p, dim=-1)
                p.sub_(lse[i][:, None]).exp_()
                o[i] = p @ vv
                if tq is not None:
                    s = tq[i] @ kk.T
                    if tk is not None:
                        s.addmm_(q[i], tk[b, h, :n].T)
                    s.mul_(scale).mul_(p)
                    to[i] = s @ vv - s.sum(dim=-1, keepdim=True) * o[i]
                    if tv is not None:
                        to[i] += p @ tv[b, h, :n]
    return o, to, lse


def _attend_grads(q, k, v, o, lse, dout):
    scale = q.shape[-1] ** -0.5
    dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    delta = (o * dout).sum(dim=-1, keepdim=True)
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            for r in range(0, q.shape[2], ROWS):
                i = (b, h, slice(r, r + ROWS))
                p = (q[i] @ k[b, h].T).mul_(scale).sub_(lse[i][:, None]).exp_()
                dv[b, h] += p.T @ dout[i]
                p.mul_((dout[i] @ v[b, h].T).sub_(delta[i])).mul_(scale)
                dq[i] = p @ k[b, h]
                dk[b, h] += p.T @ q[i]
    return dq, dk, dv


class _Attend(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v):
        o, _, lse = _attend(q, k, v)
        ctx.save_for_backward(q, k, v, o, lse)
        return o

    @staticmethod
    def backward(ctx, dout):
        return _attend_grads(*ctx.saved_tensors, dout)


def _norm_rope(x, weight, angles):
    """x [B, S, H, D]; angles [S, D] or None."""
    n = x * torch.rsqrt(x.pow(2).mean(dim=-1, keepdim=True) + 1e-6) * weight
    if angles is None:
        return n
    a = angles[:, None, :]
    return n * torch.cos(a) + torch.cat([-n[..., D // 2:], n[..., : D // 2]], dim=-1) * torch.sin(a)


def _both(f, primals, tangents):
    """f(*primals) as a tuple, and its tangents: Nones where `tangents` is None."""
    if tangents is None:
        y = f(*primals)
        return y, (None,) * len(y)
    return torch.func.jvp(f, primals, tuple(torch.zeros_like(p) if t is None else t for p, t in zip(primals, tangents)))


def _block(w, heads, x, emb, lora, text, angles, tx=None, temb=None, tlora=None):
    """A transformer block in 64 bits: x [B, T, H, W, K] -> its output and the output's tangent (None without tx)."""
    F = torch.nn.functional
    K, moves = x.shape[-1], tx is not None
    attend = _Attend.apply if torch.is_grad_enabled() else lambda q, k, v: _attend(q, k, v)[0]
    for name in ("self_attn", "cross_attn", "mlp"):
        mod = "adaln_modulation_%s." % name

        def modulated(x, emb, lora):
            m = F.linear(F.linear(F.silu(emb), w[mod + "1.weight"]), w[mod + "2.weight"]) + lora
            shift, scale, gate = (c[:, :, None, None, :] for c in m.chunk(3, dim=-1))
            return F.layer_norm(x, (K,), eps=1e-6) * (1 + scale) + shift, gate

        (n, gate), (tn, tgate) = _both(modulated, (x, emb, lora), (tx, temb, tlora) if moves else None)
        if name == "mlp":
            (r,), (tr,) = _both(lambda n: (F.linear(F.gelu(F.linear(n, w["mlp.layer1.weight"])), w["mlp.layer2.weight"]),),
                                (n,), (tn,) if moves else None)
        else:
            own, g = name == "self_attn", lambda part: w["%s.%s.weight" % (name, part)]
            split = lambda t: t.reshape(t.shape[0], -1, heads, D)
            query = lambda n: (_norm_rope(split(F.linear(n, g("q_proj"))), g("q_norm"), angles if own else None).transpose(1, 2),)
            keys = lambda c: (_norm_rope(split(F.linear(c, g("k_proj"))), g("k_norm"), angles if own else None).transpose(1, 2),
                              split(F.linear(c, g("v_proj"))).transpose(1, 2))
            (q,), (tq,) = _both(query, (n,), (tn,) if moves else None)
            (k, v), (tk, tv) = _both(keys, (n if own else text,), (tn,) if moves and own else None)
            merge = lambda o: F.linear(o.transpose(1, 2).flatten(-2), g("output_proj")).reshape(x.shape)
            if moves:
                o, to, _ = _attend(q, k, v, tq, tk, tv)
                r, tr = merge(o), merge(to)
            else:
                r, tr = merge(attend(q, k, v)), None
        (x,), (tx,) = _both(lambda x, r, gate: (x + gate * r,), (x, r, gate), (tx, tr, tgate) if moves else None)
    return x, tx


def _network(s, case):
    F = torch.nn.functional
    net, f = s["net"], lambda t: t.double()
    w = {n: f(p) for n, p in net.named_parameters()}
    B, T, Hh, W, K = case["B"], case["T"], case["Hh"], case["W"], case["H"] * D
    pos = net.pos_embedder
    rates = [10000.0 ** -f(r) for r in (pos.dim_temporal_range, pos.dim_spatial_range, pos.dim_spatial_range)]
    steps = [torch.arange(n, device="cuda", dtype=torch.float64) for n in (T, Hh, W)]
    steps[0] = steps[0] / f(s["fps"][0]) * pos.base_fps
    e = [torch.outer(p, r) for p, r in zip(steps, rates)]
    half = torch.cat([e[0][:, None, None].expand(T, Hh, W, -1), e[1][None, :, None].expand(T, Hh, W, -1),
                      e[2][None, None].expand(T, Hh, W, -1)], dim=-1).reshape(T * Hh * W, -1)
    angles = torch.cat([half, half], dim=-1)
    x = torch.cat([f(s["x"]), f(s["mask"])[:, :, None].expand(B, 1, T, 2 * Hh, 2 * W)], dim=1)
    x = x.reshape(B, -1, T, Hh, 2, W, 2).permute(0, 2, 3, 5, 1, 4, 6).flatten(-3)
    x = F.linear(x, w["x_embedder.proj.1.weight"])
    turn = f(s["time"])[..., None] * torch.exp(-math.log(10000.0) * torch.arange(K // 2, device="cuda", dtype=torch.float64) / (K // 2))
    wave = torch.cat([torch.cos(turn), torch.sin(turn)], dim=-1)
    lora = F.linear(F.silu(F.linear(wave, w["t_embedder.1.linear_1.weight"])), w["t_embedder.1.linear_2.weight"])
    emb = wave * torch.rsqrt(wave.pow(2).mean(dim=-1, keepdim=True) + 1e-6) * w["t_embedding_norm.weight"]
    for i in range(case["blocks"]):
        own = "blocks.%d." % i
        x, _ = _block({n[len(own):]: p for n, p in w.items() if n.startswith(own)}, case["H"], x, emb, lora, f(s["text"]), angles)
    m = F.linear(F.linear(F.silu(emb), w["final_layer.adaln_modulation.1.weight"]), w["final_layer.adaln_modulation.2.weight"])
    shift, scale = (c[:, :, None, None, :] for c in (m + lora[..., : 2 * K]).chunk(2, dim=-1))
    y = F.linear(F.layer_norm(x, (K,), eps=1e-6) * (1 + scale) + shift, w["final_layer.linear.weight"])
    y = y.reshape(B, T, Hh, W, 2, 2, 16)
    return y.permute(0, 6, 1, 2, 4, 3, 5).reshape(B, 16, T, 2 * Hh, 2 * W)


def exact(case, seed):
    """What `run` returns, in 64-bit torch arithmetic on the same inputs; None for the largest cases."""
    if _flops(case) > EXACT_FLOPS:
        return None
    s, kind = prepare(case, seed), case["kind"]
    f = lambda t: t.detach().double()
    if kind in ("attention_jvp", "cross_jvp"):
        o, to, lse = _attend(*(f(t) for t in s["in"][:4]), *(f(t) for t in s["in"][4:]), lens=s.get("lens"))
        return (o, to) if kind == "attention_jvp" else (o, to, lse)
    if kind in ("attention", "attention_train", "cross_train"):
        q, k, v = (f(t).transpose(1, 2).contiguous() for t in s["in"])
        o, _, lse = _attend(q, k, v)
        if kind == "attention":
            return o.transpose(1, 2).contiguous()
        grads = _attend_grads(q, k, v, o, lse, f(s["dout"]).transpose(1, 2).contiguous())
        return tuple(t.transpose(1, 2).contiguous() for t in (o, *grads))
    if kind.startswith("norm_rope"):
        x, weight, angles, other = f(s["x"]), f(s["weight"]), f(s["angles"]).reshape(-1, D), f(s["other"])
        if kind == "norm_rope_jvp":
            return torch.func.jvp(lambda x: _norm_rope(x, weight, angles), (x,), (other,))
        x.requires_grad_(True)
        weight.requires_grad_(True)
        y = _norm_rope(x, weight, angles)
        return (y.detach(), *torch.autograd.grad(y, (x, weight), other))
    if kind == "network":
        with torch.no_grad():
            return _network(s, case)
    train = kind == "block_train"
    w = {n: f(p).requires_grad_(train) for n, p in s["block"].named_parameters()}
    x, angles = f(s["x"]).requires_grad_(train), f(s["angles"]).reshape(-1, D)
    args = (w, case["H"], x, f(s["emb"]), f(s["lora"]), f(s["text"]), angles)
    if not train:
        with torch.no_grad():
            if kind == "block":
                return _block(*args)[0]
            return _block(*args, f(s["tx"]), f(s["temb"]), f(s["tlora"]))
    y, _ = _block(*args)
    y.backward(f(s["dout"]))
    return {"y": y.detach(), "dx": x.grad, **{n: p.grad for n, p in w.items()}}
