"""The DiT transformer ``Block`` (self-attention, cross-attention and MLP, each behind a LayerNorm with adaLN
modulation and a gated residual) on the HIP attention path, with a forward that also carries a tangent.

Reference: ``Block`` (cosmos_predict2/_src/predict2/networks/minimal_v4_dit.py:993-1242) and ``GPT2FeedForward``
(:222-249) -- same constructor arguments, sub-module and parameter names (``self_attn.*``, ``cross_attn.*``,
``mlp.layer1/2.weight``, ``adaln_modulation_{self_attn,cross_attn,mlp}.{1,2}.weight``: a reference state dict of the
block loads as is), ``init_weights``, ``forward(x_B_T_H_W_D, emb_B_T_D, crossattn_emb, rope_emb_L_1_1_D,
adaln_lora_B_T_3D, extra_per_block_pos_emb)``.

``forward_jvp`` pushes a tangent of ``(x, emb, adaln_lora)`` through the block: what a consistency-distillation step
needs when it differentiates the network along (x_t, t).  The reference ships the attention JVP kernel but no caller
that does this, so the rules are written out here: LayerNorm + modulation, GELU and the gated residuals each in one
fused HIP pass (fp32 arithmetic on 16-bit tensors), the tiny modulation MLP by torch forward AD, linear layers on
primal and tangent stacked in one GEMM (the fused passes write both into one buffer, so nothing is copied to stack
them), attention through ``Attention.forward_jvp``.
"""
from __future__ import annotations

import math
from typing import Optional, Tuple

import torch
import torch.nn.functional as F
from torch import nn

from . import ops
from .dit_attention import Attention, I2VCrossAttention
from .linear import bare, linear_one


def _per_row(m, like):
    """The modulation vectors m, one per group of consecutive rows, repeated to the shape of ``like``."""
    D = like.shape[-1]
    groups = m.reshape(-1, 1, D)
    return groups.expand(-1, like.numel() // D // groups.shape[0], D).reshape(like.shape)


def _per_group(t, m):
    """The sum of t's rows over each group of the modulation vector m, in m's shape and type."""
    D = t.shape[-1]
    return t.reshape(m.numel() // D, -1, D).sum(1).reshape(m.shape).to(m.dtype)


def _ln_modulate_bwd_differentiable(x, scale, dy, dskip, eps):
    """``ops.ln_modulate_bwd`` in differentiable tensor-library ops (fp32)."""
    mean = lambda t: t.mean(-1, keepdim=True)
    xc = x.float() - mean(x.float())
    r = (mean(xc * xc) + eps).rsqrt()
    n, dyf = xc * r, dy.float()
    dn = dyf * (1 + _per_row(scale.float(), dyf))
    dx = r * (dn - mean(dn) - n * mean(dn * n))
    if dskip is not None:
        dx = dx + dskip.float()
    return dx.to(x.dtype), _per_group(dyf, scale), _per_group(dyf * n, scale)


class _LnModulateFn(torch.autograd.Function):
    """``LayerNorm(x) * (1 + scale) + shift`` as the fused pass, differentiable (x ``[B, T, H, W, D]``, shift / scale
    ``[B, T, 1, 1, D]``).  Returns x as well, for the residual connection around what follows: both gradients of x then meet in
    the fused backward pass."""

    @staticmethod
    def forward(ctx, x, shift, scale, eps):
        D = x.shape[-1]
        y, _ = ops.ln_modulate(x, shift.reshape(-1, D), scale.reshape(-1, D), eps=eps)
        ctx.save_for_backward(x, scale)
        ctx.eps = eps
        ctx.set_materialize_grads(False)
        return y, x

    @staticmethod
    def backward(ctx, dy, dskip):
        x, scale = ctx.saved_tensors
        if dy is None:
            return dskip, None, None, None
        if torch.is_grad_enabled():      # create_graph: the gradients are differentiated again
            dx, dshift, dscale = _ln_modulate_bwd_differentiable(x, scale, dy, dskip, ctx.eps)
        else:
            dx, dshift, dscale = ops.ln_modulate_bwd(x, scale, dy, dskip, eps=ctx.eps)
        return dx, dshift.reshape(scale.shape), dscale.reshape(scale.shape), None


class _GatedResidualFn(torch.autograd.Function):
    """``x + gate * res`` as the fused pass, differentiable (gate ``[B, T, 1, 1, D]``)."""

    @staticmethod
    def forward(ctx, x, res, gate):
        out, _ = ops.gated_residual(x, res, gate.reshape(-1, x.shape[-1]))
        ctx.save_for_backward(res, gate)
        return out

    @staticmethod
    def backward(ctx, dy):
        res, gate = ctx.saved_tensors
        if torch.is_grad_enabled():      # create_graph, as above
            dres, dgate = dy * _per_row(gate, dy), _per_group(dy.float() * res.float(), gate)
        else:
            dres, dgate = ops.gated_residual_bwd(res, gate, dy)
        return dy, dres, dgate.reshape(gate.shape)


class _GeluFn(torch.autograd.Function):
    """Exact GELU as the fused pass, differentiable."""

    @staticmethod
    def forward(ctx, h):
        ctx.save_for_backward(h)
        return ops.gelu(h)[0]

    @staticmethod
    def backward(ctx, dy):
        (h,) = ctx.saved_tensors
        return torch.ops.aten.gelu_backward(dy, h, approximate="none")


class _ModulationFn(torch.autograd.Function):
    """The modulation vectors as ``ops.modulation`` makes them (values), differentiable in emb, lora and the six weights.  The
    backward pass forms the two small activations again; the gradients of emb and lora are summed over the three MLPs in fp32."""

    @staticmethod
    def forward(ctx, emb, lora, *w):
        ctx.save_for_backward(emb, *w)
        ctx.lora_shape = lora.shape
        return ops.modulation(emb, lora, w[:3], w[3:])[0]

    @staticmethod
    def backward(ctx, dout):
        emb, *w = ctx.saved_tensors
        need = ctx.needs_input_grad
        e = emb.reshape(-1, emb.shape[-1])
        a, rows = F.silu(e), e.shape[0]
        cat = lambda m: m.transpose(0, 1).reshape(rows, -1)          # [3, rows, D] -> [rows, 3 D]
        dw1, dw2, da = [None] * 3, [None] * 3, 0
        for i in range(3):
            dm = cat(dout[i])
            if need[5 + i]:
                dw2[i] = dm.t() @ (a @ w[i].t())
            if need[0] or need[2 + i]:
                dh = dm @ w[3 + i]
                if need[2 + i]:
                    dw1[i] = dh.t() @ a
                if need[0]:
                    da = da + (dh @ w[i]).float()
        demb = dlora = None
        if need[0]:
            ef = e.float()
            sig = torch.sigmoid(ef)
            demb = (da * (sig * (1 + ef * (1 - sig)))).to(emb.dtype).reshape(emb.shape)
        if need[1]:
            dlora = cat(dout.float().sum(0)).to(dout.dtype).reshape(ctx.lora_shape)
        return (demb, dlora, *dw1, *dw2)


# A call of up to this many rows (one per batch row and frame; with tangents as many again) forms the modulation vectors in two
# launches of its own kernels.  Those read the weights again for every 16 rows, the library's products once, so that many rows are
# the library's.  Measured, us, own kernels / modules, values only: in a replayed graph 5120 channels 64 rows 45 / 73, 128 rows
# 75 / 80, 192 rows 107 / 86; 2048 channels 64 rows 21 / 52, 256 rows 57 / 66, 512 rows 101 / 77.  With tangents, 64 rows: 76 / 291
# and 36 / 203.  Launched one by one the modules take 200, with tangents 910, at any of these sizes.  The line lies where the own
# kernels take at most two thirds of the modules' time on the GPU at both widths; at 5120 channels they stop winning at some 140 rows.
_FUSED_MODULATION_ROWS = 64


class GPT2FeedForward(nn.Module):
    def __init__(self, d_model: int, d_ff: int):
        super().__init__()
        self.activation = nn.GELU()
        self.layer1 = nn.Linear(d_model, d_ff, bias=False)
        self.layer2 = nn.Linear(d_ff, d_model, bias=False)
        self._layer_id = None
        self._dim = d_model
        self._hidden_dim = d_ff
        self.init_weights()

    def init_weights(self) -> None:
        """minimal_v4_dit.py:234-242: truncated normal, std 1/sqrt(fan_in), the second layer scaled down with depth."""
        std = 1.0 / math.sqrt(self._dim)
        torch.nn.init.trunc_normal_(self.layer1.weight, std=std, a=-3 * std, b=3 * std)
        std = 1.0 / math.sqrt(self._hidden_dim)
        if self._layer_id is not None:
            std = std / math.sqrt(2 * (self._layer_id + 1))
        torch.nn.init.trunc_normal_(self.layer2.weight, std=std, a=-3 * std, b=3 * std)

    def forward(self, x: torch.Tensor):
        h = linear_one(self.layer1, x)
        if h.is_cuda and h.numel() % 8 == 0 and h.dtype in (torch.bfloat16, torch.float16):
            if torch.is_grad_enabled() and h.requires_grad:
                return linear_one(self.layer2, _GeluFn.apply(h))
            return linear_one(self.layer2, ops.gelu(h, inplace=True)[0])      # inference: one fused pass, in place
        return self.layer2(self.activation(h))

    @torch.no_grad()
    def forward_jvp(self, x: torch.Tensor, tx: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
        b = x.shape[0]
        both = ops.as_stacked(x, tx)
        h = linear_one(self.layer1, both if both is not None else torch.cat([x, tx], dim=0))
        ops.gelu(h[:b], h[b:], inplace=True)       # a = gelu(h), ta = th gelu'(h), in place on the stacked buffer
        y = linear_one(self.layer2, h)
        return y[:b], y[b:]


class Block(nn.Module):
    def __init__(
        self,
        x_dim: int,
        context_dim: int,
        num_heads: int,
        mlp_ratio: float = 4.0,
        use_adaln_lora: bool = False,
        adaln_lora_dim: int = 256,
        backend: str = "hip",
        image_context_dim: Optional[int] = None,
        use_wan_fp32_strategy: bool = False,
    ):
        super().__init__()
        self.x_dim = x_dim
        fp32 = dict(use_wan_fp32_strategy=use_wan_fp32_strategy)
        self.layer_norm_self_attn = nn.LayerNorm(x_dim, elementwise_affine=False, eps=1e-6)
        self.self_attn = Attention(x_dim, None, num_heads, x_dim // num_heads, qkv_format="bshd", backend=backend, **fp32)
        self.layer_norm_cross_attn = nn.LayerNorm(x_dim, elementwise_affine=False, eps=1e-6)
        if image_context_dim is None:
            self.cross_attn = Attention(x_dim, context_dim, num_heads, x_dim // num_heads, qkv_format="bshd", backend=backend, **fp32)
        else:   # crossattn_emb is then the pair (text context, image context)
            self.cross_attn = I2VCrossAttention(x_dim, context_dim, num_heads, x_dim // num_heads,
                                                img_latent_dim=image_context_dim, qkv_format="bshd", backend=backend, **fp32)
        self.layer_norm_mlp = nn.LayerNorm(x_dim, elementwise_affine=False, eps=1e-6)
        self.mlp = GPT2FeedForward(x_dim, int(x_dim * mlp_ratio))

        self.use_adaln_lora = use_adaln_lora

        def modulation():
            if use_adaln_lora:
                return nn.Sequential(nn.SiLU(), nn.Linear(x_dim, adaln_lora_dim, bias=False),
                                     nn.Linear(adaln_lora_dim, 3 * x_dim, bias=False))
            return nn.Sequential(nn.SiLU(), nn.Linear(x_dim, 3 * x_dim, bias=False))

        self.adaln_modulation_self_attn = modulation()
        self.adaln_modulation_cross_attn = modulation()
        self.adaln_modulation_mlp = modulation()
        self.cp_size = None
        self.use_wan_fp32_strategy = use_wan_fp32_strategy

    def set_context_parallel_group(self, process_group, ranks, stream):
        self.cp_size = None if ranks is None else len(ranks)
        self.self_attn.set_context_parallel_group(process_group=process_group, ranks=ranks, stream=stream)

    def reset_parameters(self) -> None:
        """minimal_v4_dit.py:1095-1111: the last modulation layer starts at zero (the block starts as the identity)."""
        mods = (self.adaln_modulation_self_attn, self.adaln_modulation_cross_attn, self.adaln_modulation_mlp)
        if self.use_adaln_lora:
            std = 1.0 / math.sqrt(self.x_dim)
            for m in mods:
                torch.nn.init.trunc_normal_(m[1].weight, std=std, a=-3 * std, b=3 * std)
                torch.nn.init.zeros_(m[2].weight)
        else:
            for m in mods:
                torch.nn.init.zeros_(m[1].weight)

    def init_weights(self) -> None:
        self.reset_parameters()
        self.self_attn.init_weights()
        self.cross_attn.init_weights()
        self.mlp.init_weights()

    # ------------------------------------------------------------------ pieces
    def _modulation(self, mod: nn.Sequential, emb_B_T_D, adaln_lora_B_T_3D, like):
        """(shift, scale, gate), each ``[B, T, 1, 1, D]`` in the type of x (minimal_v4_dit.py:1131-1162).  With
        ``use_wan_fp32_strategy`` the modulation MLP runs in fp32 (an fp32 autocast region, as in the reference) on the
        fp32 time embedding and is rounded once, to the type of x."""
        with self._fp32_region(emb_B_T_D):
            m = mod(emb_B_T_D)
            if self.use_adaln_lora:
                m = m + adaln_lora_B_T_3D
        return tuple(c[:, :, None, None, :].type_as(like) for c in m.chunk(3, dim=-1))

    def _modulation_jvp(self, mod: nn.Sequential, emb, temb, lora, tlora, like):
        """Modulation and its tangent; the tensors are ``[B, T, 3 D]``, tiny next to x: forward AD does it."""
        f = (lambda e, l: mod(e) + l) if self.use_adaln_lora else (lambda e, l: mod(e))
        if lora is None:
            lora = emb.new_zeros(())
        temb = torch.zeros_like(emb) if temb is None else temb
        tlora = torch.zeros_like(lora) if tlora is None else tlora
        with self._fp32_region(emb):
            m, tm = torch.func.jvp(f, (emb, lora), (temb, tlora))
        cut = lambda z: tuple(c[:, :, None, None, :].type_as(like) for c in z.chunk(3, dim=-1))
        return cut(m), cut(tm)

    def _fused_modulations(self, emb, lora, like, temb=None, tlora=None, tangent=False):
        """All three sub-layers' modulation vectors in two launches: ``[3, 3, rows, D]`` (sub-layer; shift, scale, gate), through its
        autograd rule where grad mode is on, and its tangent; or None where the modules compute something else than the plain MLPs
        of one 16-bit type, or for many rows."""
        if not self.use_adaln_lora or self.use_wan_fp32_strategy or lora is None or torch.is_autocast_enabled("cuda"):
            return None
        mods = (self.adaln_modulation_self_attn, self.adaln_modulation_cross_attn, self.adaln_modulation_mlp)
        w1, w2 = [], []
        for m in mods:
            if type(m) is not nn.Sequential or len(m) != 3 or not bare(m) or not all(bare(c) for c in m):
                return None
            if type(m[0]) is not nn.SiLU or any(type(c) is not nn.Linear or c.bias is not None or type(c.weight) is not nn.Parameter for c in m[1:]):
                return None
            w1.append(m[1].weight)
            w2.append(m[2].weight)
        K, D = emb.shape[-1], like.shape[-1]
        rows = emb.numel() // K
        given = [t for t in (emb, lora, temb, tlora) if t is not None]
        if rows > _FUSED_MODULATION_ROWS or K % 32 or D % 16 or w1[0].shape[0] % 32 or like.dtype not in (torch.bfloat16, torch.float16):
            return None
        if any(t.dtype != like.dtype or t.device != like.device or not t.is_cuda for t in (*given, *w1, *w2)):
            return None
        if any(t.shape[:-1] != emb.shape[:-1] for t in given) or lora.shape[-1] != 3 * D or (tlora is not None and tlora.shape != lora.shape):
            return None
        if any(w.shape != (w1[0].shape[0], K) for w in w1) or any(w.shape != (3 * D, w1[0].shape[0]) for w in w2):
            return None
        if not all(ops._is_dense16(w) for w in (*w1, *w2)):     # (views of a flat buffer: the library's layers read them where they are)
            return None
        if torch.is_grad_enabled() and not tangent:
            return _ModulationFn.apply(emb, lora, *w1, *w2), None
        return ops.modulation(emb, lora, w1, w2, temb, tlora, tangent)

    def _modulations(self, emb, lora, like):
        """(shift, scale, gate) of one sub-layer after the other; modules are called when their turn comes."""
        fused = self._fused_modulations(emb, lora, like)
        vectors = None if fused is None else fused[0].flatten(0, 1).unbind(0)
        for i, m in enumerate((self.adaln_modulation_self_attn, self.adaln_modulation_cross_attn, self.adaln_modulation_mlp)):
            yield self._modulation(m, emb, lora, like) if fused is None else vectors[3 * i:3 * i + 3]

    def _fp32_region(self, t: torch.Tensor):
        return torch.autocast(t.device.type, enabled=self.use_wan_fp32_strategy, dtype=torch.float32)

    @staticmethod
    def _modulate_jvp(norm_layer, x, tx, mod, tmod):
        """LayerNorm + modulation of x and its tangent (one fused pass), written into the two halves of one buffer so
        that the projections that follow map both in one GEMM without a copy."""
        (shift, scale, _), (tshift, tscale, _) = mod, tmod
        y, ty = ops.stacked_pair(x.shape, x.dtype, x.device)
        flat = lambda m: m.reshape(-1, m.shape[-1])
        ops.ln_modulate(x, flat(shift), flat(scale), tx, flat(tshift), flat(tscale), eps=norm_layer.eps, out=y, tout=ty)
        return y, ty

    @staticmethod
    def _residual_modulate_jvp(norm_layer, x, tx, res, tres, gates, mod, tmod):
        """The gated residual of the sub-layer before (``gates``: its modulation and tangent) and :meth:`_modulate_jvp` of it."""
        (shift, scale, _), (tshift, tscale, _) = mod, tmod
        y, ty = ops.stacked_pair(x.shape, x.dtype, x.device)
        flat = lambda m: m.reshape(-1, m.shape[-1])
        return ops.gated_residual_ln_modulate(x, res, flat(gates[0][2]), flat(shift), flat(scale), tx, tres, flat(gates[1][2]), flat(tshift),
                                              flat(tscale), eps=norm_layer.eps, y=y, ty=ty)

    @staticmethod
    def _gated_residual_jvp(x, tx, res, tres, mod, tmod):
        flat = lambda m: m.reshape(-1, m.shape[-1])
        return ops.gated_residual(x, res, flat(mod[2]), tx, tres, flat(tmod[2]))

    # ------------------------------------------------------------------ the reference's surface
    def forward(
        self,
        x_B_T_H_W_D: torch.Tensor,
        emb_B_T_D: torch.Tensor,
        crossattn_emb: torch.Tensor,
        rope_emb_L_1_1_D: Optional[torch.Tensor] = None,
        adaln_lora_B_T_3D: Optional[torch.Tensor] = None,
        extra_per_block_pos_emb: Optional[torch.Tensor] = None,
    ) -> torch.Tensor:
        x = x_B_T_H_W_D
        if extra_per_block_pos_emb is not None:
            x = x + extra_per_block_pos_emb
        if not torch.is_grad_enabled() and x.is_cuda:
            return self._forward_fused(x, emb_B_T_D, crossattn_emb, rope_emb_L_1_1_D, adaln_lora_B_T_3D)
        return self._forward_autograd(x, emb_B_T_D, crossattn_emb, rope_emb_L_1_1_D, adaln_lora_B_T_3D)

    def _forward_autograd(self, x, emb, crossattn_emb, rope, lora):
        """The differentiable path: the same kernels as the inference path (so both give the same bits, as long as the attention
        call does not cut its keys into ranges, which the inference path's cross-attention never does), each behind an autograd
        rule: attention, RMSNorm + RoPE, LayerNorm + modulation and the gated residuals through their HIP backward kernels."""
        B, T, H, W, D = x.shape
        for name, norm, sub, (shift, scale, gate) in zip(("self_attn", "cross_attn", "mlp"),
                                                         (self.layer_norm_self_attn, self.layer_norm_cross_attn, self.layer_norm_mlp),
                                                         (self.self_attn, self.cross_attn, self.mlp), self._modulations(emb, lora, x)):
            n, x = _LnModulateFn.apply(x, shift, scale, norm.eps)
            if name == "mlp":
                r = sub(n)
            else:
                r = sub(n.reshape(B, T * H * W, D), None if name == "self_attn" else crossattn_emb, rope_emb=rope)
            x = _GatedResidualFn.apply(x, r.reshape(x.shape), gate)
        return x

    def _forward_fused(self, x, emb, crossattn_emb, rope, lora):
        """Inference (no autograd): the same arithmetic with LayerNorm + modulation, the gated residuals and GELU each as
        one fused HIP pass instead of a chain of tensor-library ops."""
        B, T, H, W, D = x.shape
        flat2 = lambda m: m.reshape(-1, D)
        for name, norm, sub, (shift, scale, gate) in zip(("self_attn", "cross_attn", "mlp"),
                                                         (self.layer_norm_self_attn, self.layer_norm_cross_attn, self.layer_norm_mlp),
                                                         (self.self_attn, self.cross_attn, self.mlp), self._modulations(emb, lora, x)):
            if name == "self_attn":
                n, _ = ops.ln_modulate(x, flat2(shift), flat2(scale), eps=norm.eps)
            else:
                x, _, n, _ = ops.gated_residual_ln_modulate(x, r, r_gate, flat2(shift), flat2(scale), eps=norm.eps)
            if name == "mlp":
                r = sub(n)
            else:
                r = sub(n.reshape(B, T * H * W, D), None if name == "self_attn" else crossattn_emb, rope_emb=rope)
            r, r_gate = r.reshape(x.shape), flat2(gate)
        return ops.gated_residual(x, r, r_gate)[0]

    # ------------------------------------------------------------------ forward mode
    @torch.no_grad()
    def forward_jvp(
        self,
        x_B_T_H_W_D: torch.Tensor,
        tx_B_T_H_W_D: torch.Tensor,
        emb_B_T_D: torch.Tensor,
        temb_B_T_D: Optional[torch.Tensor],
        crossattn_emb: torch.Tensor,
        rope_emb_L_1_1_D: Optional[torch.Tensor] = None,
        adaln_lora_B_T_3D: Optional[torch.Tensor] = None,
        tadaln_lora_B_T_3D: Optional[torch.Tensor] = None,
        extra_per_block_pos_emb: Optional[torch.Tensor] = None,
    ) -> Tuple[torch.Tensor, torch.Tensor]:
        """``(out, tout)``: the block's output and its derivative along ``(tx, temb, tadaln_lora)``; the text context
        and the positional terms do not move."""
        x, tx = x_B_T_H_W_D, tx_B_T_H_W_D
        assert tx.shape == x.shape
        if extra_per_block_pos_emb is not None:
            x = x + extra_per_block_pos_emb
        B, T, H, W, D = x.shape
        flat = lambda z: z.reshape(B, T * H * W, D)
        vid = lambda z: z.reshape(B, T, H, W, D)
        fused = self._fused_modulations(emb_B_T_D, adaln_lora_B_T_3D, x, temb_B_T_D, tadaln_lora_B_T_3D, tangent=True)

        def modulation(i, layers):
            if fused is not None:
                return fused[0][i].unbind(0), fused[1][i].unbind(0)
            return self._modulation_jvp(layers, emb_B_T_D, temb_B_T_D, adaln_lora_B_T_3D, tadaln_lora_B_T_3D, x)

        mod, tmod = modulation(0, self.adaln_modulation_self_attn)
        n, tn = self._modulate_jvp(self.layer_norm_self_attn, x, tx, mod, tmod)
        r, tr = self.self_attn.forward_jvp(flat(n), flat(tn), rope_emb=rope_emb_L_1_1_D)

        gates, (mod, tmod) = (mod, tmod), modulation(1, self.adaln_modulation_cross_attn)
        x, tx, n, tn = self._residual_modulate_jvp(self.layer_norm_cross_attn, x, tx, vid(r), vid(tr), gates, mod, tmod)
        r, tr = self.cross_attn.forward_jvp(flat(n), flat(tn), crossattn_emb, None, rope_emb=rope_emb_L_1_1_D)

        gates, (mod, tmod) = (mod, tmod), modulation(2, self.adaln_modulation_mlp)
        x, tx, n, tn = self._residual_modulate_jvp(self.layer_norm_mlp, x, tx, vid(r), vid(tr), gates, mod, tmod)
        r, tr = self.mlp.forward_jvp(n, tn)
        x, tx = self._gated_residual_jvp(x, tx, r, tr, mod, tmod)
        return x, tx
