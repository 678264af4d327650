"""Linear layers without bias (``nn.Linear``: the projections and the MLP of a block, cosmos_predict2/_src/predict2/networks/minimal_v4_dit.py:226-227,
:349-358) on the package's own matrix products where those are faster, several layers of one input in a launch; ``nn.Linear`` itself elsewhere.

The parameters stay where they are.  Whatever gives calling the module a meaning of its own (hooks, another class, a parametrization, autocast, function
transforms, forward-mode AD, compilation, tensor subclasses, modes that watch operators) goes through the module.
"""
from __future__ import annotations

from typing import Optional, Sequence

import torch
import torch.nn.functional as F
from torch import nn
from torch.autograd import forward_ad
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from . import ops


# Fewer rows than these are the library's in every layer (cosmos_attn_gemm_preferred): the layer's own product, and the first of its backward pass.  Asked first, as the
# checks and the descriptor cost a layer some 10 us on the host, which a call of few rows waits for.
FEWEST_ROWS = 1024
FEWEST_ROWS_BACKWARD = 256


def bare(m: nn.Module) -> bool:
    """Is calling m the same as computing its forward?"""
    return not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks or "forward" in m.__dict__
                or nn.modules.module._has_any_global_hook())


def _memory_says_all(*tensors: torch.Tensor) -> bool:
    """Is nothing lost by reading the tensors' memory: no tangent (dual levels), no level of a function transform or of batched gradients (their tensors have
    no storage of their own, ``is_grads_batched``'s older ones with no other mark), no subclass?"""
    return forward_ad._current_level < 0 and all(
        type(t) in (torch.Tensor, nn.Parameter) and torch._C._has_storage(t) and not torch._C._functorch.is_functorch_wrapped_tensor(t) for t in tensors)


def _watched() -> bool:
    """Does a mode see the operators that are called (a FLOP counter, selective checkpointing, a user's own)?  Products launched by address pass it by.  (A default
    device is a mode as well, of factory functions.)"""
    if torch._C._len_torch_dispatch_stack():
        return True
    return bool(torch._C._len_torch_function_stack()) and any(type(m) is not DeviceContext for m in _get_current_function_mode_stack())


def _weights(layers: Sequence[nn.Module], x: torch.Tensor) -> Optional[list]:
    """The layers' weights, if their products with x may be formed by ``ops.gemm``."""
    if not x.is_cuda or x.dtype not in (torch.bfloat16, torch.float16) or type(x) is not torch.Tensor or x.numel() == 0:
        return None
    if torch.is_autocast_enabled("cuda") or torch.compiler.is_compiling() or torch.jit.is_tracing() or _watched():
        return None
    if not _memory_says_all(x) or not ops._is_dense16(x):
        return None
    ws = []
    for m in layers:
        if type(m) is not nn.Linear or m.bias is not None or not bare(m):
            return None
        w = m.weight
        if type(w) is not nn.Parameter or not _memory_says_all(w) or w.dtype != x.dtype or w.device != x.device or w.shape != layers[0].weight.shape or not ops._is_dense16(w):
            return None
        ws.append(w)
    if ws[0].shape[1] != x.shape[-1]:
        return None
    return ws


class _LinearFn(torch.autograd.Function):
    """``x w_i^T`` for up to three weights of one shape: the outputs in one launch, their part of x's gradient summed in one, the weights' gradients in one."""

    @staticmethod
    def forward(ctx, made, x, *w):
        # as nn.Linear: x for the weights' gradients, the weights for x's; what no gradient asks for may be freed or written over
        ctx.save_for_backward(x if any(ctx.needs_input_grad[2:]) else None, *(w if ctx.needs_input_grad[1] else ()))
        ctx.x_shape = x.shape
        ctx.set_materialize_grads(False)
        return tuple(made if made is not None else [F.linear(x, v) for v in w])

    @staticmethod
    def backward(ctx, *dy):
        x, *w = ctx.saved_tensors
        given = [i for i, g in enumerate(dy) if g is not None]
        g2 = {i: dy[i].reshape(-1, dy[i].shape[-1]) for i in given}
        dx, dw = None, [None] * len(dy)
        # (create_graph: the gradients are differentiated again)
        own = not torch.is_grad_enabled() and not _watched() and _memory_says_all(*w, *(t for t in (x, *(dy[i] for i in given)) if t is not None))
        if own:          # (hooks on saved tensors may bring them back in another layout)
            g2, w = {i: ops._dense16(g) for i, g in g2.items()}, [ops._dense16(v) for v in w]
        if ctx.needs_input_grad[1] and given:
            gs, ws = [g2[i] for i in given], [w[i] for i in given]
            dx = ops.gemm("xw", gs, ws, total=True, if_preferred=True) if own else None
            if dx is None:
                for g, v in zip(gs, ws):
                    dx = g @ v if dx is None else dx + g @ v
            dx = dx.reshape(ctx.x_shape)
        wanted = [i for i in given if ctx.needs_input_grad[2 + i]]
        if wanted:
            x2 = x.reshape(-1, x.shape[-1])
            if own:
                x2 = ops._dense16(x2)
            made = ops.gemm("xtx", [g2[i] for i in wanted], [x2] * len(wanted), if_preferred=True) if own else None
            for k, i in enumerate(wanted):
                dw[i] = made[k] if made is not None else g2[i].t() @ x2
        return (None, dx, *dw)


def linear(layers: Sequence[nn.Module], x: torch.Tensor) -> list:
    """``[m(x) for m in layers]``: up to three layers without bias."""
    rows = x.shape[:-1].numel()
    recording = torch.is_grad_enabled()
    if rows < (FEWEST_ROWS_BACKWARD if recording else FEWEST_ROWS):
        return [m(x) for m in layers]
    ws = _weights(layers, x)
    if ws is None:
        return [m(x) for m in layers]
    made = None
    if rows >= FEWEST_ROWS:
        made = ops.gemm("xwt", [x.detach().view(rows, -1)] * len(ws), ws, if_preferred=True, lead=x.shape[:-1])
    if recording and (x.requires_grad or any(w.requires_grad for w in ws)):
        return list(_LinearFn.apply(made, x, *ws))
    return made if made is not None else [m(x) for m in layers]
