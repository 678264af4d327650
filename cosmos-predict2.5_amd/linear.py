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


# Fewer rows than these are the library's in every layer (cosmos_attn_gemm_preferred): the layer's own product, and the first of its backward pass.  Asked first: the
# sizes cost a layer 2 us on the host, all of the checks 7.
FEWEST_ROWS = 1024
FEWEST_ROWS_BACKWARD = 256
# One or two layers whose own product is the library's for want of rows have an autograd rule of their own only from this many operations on, where the GPU takes as long as the
# host: 10 to 30 us a layer more than nn.Linear's.  Forward and backward, us, module / own: an MLP 1024 wide, 520 rows 280 / 310, 2048 wide 900 rows (3e10) 280 / 307; one layer of 5120 x 5120,
# 768 rows (4e10) 145 / 171, 1000 rows (5.2e10) 199 / 180; three layers together from the fewest rows on (2048 x 2048, 256 rows 349 / 324).
LEAST_RECORDED = 4e10


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


def _plain_input(x: torch.Tensor) -> bool:
    return type(x) is torch.Tensor and x.is_cuda and x.dtype in (torch.bfloat16, torch.float16) and x.numel() > 0 and not torch.compiler.is_compiling() and not torch.jit.is_tracing()


def _own(rows: int, cols: int, depth: int, count: int, recording: bool):
    """Are the layers' products, and is any of their backward pass, the package's own?"""
    forward = rows >= FEWEST_ROWS and ops.gemm_preferred("xwt", rows, cols, depth, depth, depth, count)
    if rows < FEWEST_ROWS and count < 3 and 2 * rows * cols * depth < LEAST_RECORDED:
        return False, False
    backward = recording and (ops.gemm_preferred("xw", rows, depth, cols, cols, depth, count, True) or ops.gemm_preferred("xtx", cols, depth, rows, cols, depth, count))
    return forward, backward


def _weights(layers: Sequence[nn.Module], x: torch.Tensor, cols: int, depth: int) -> Optional[list]:
    """The layers' weights, if their products with x may be formed by ``ops.gemm``."""
    if torch.is_autocast_enabled("cuda") or _watched() or not _memory_says_all(x) or not ops._is_dense16(x):
        return None
    ws = []
    for m in layers:
        if type(m) is not nn.Linear or m.bias is not None or not bare(m):
            return None
        w = m.weight
        if type(w) is not nn.Parameter or not _memory_says_all(w) or w.dtype != x.dtype or w.device != x.device or w.shape != (cols, depth) or not ops._is_dense16(w):
            return None
        ws.append(w)
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
        wanted = [i for i in given if ctx.needs_input_grad[2 + i]]
        dx, dw = None, [None] * len(dy)
        if not given:
            return (None, dx, *dw)
        of_x = ctx.needs_input_grad[1]
        depth, cols = ctx.x_shape[-1], dy[given[0]].shape[-1]
        g2 = {i: dy[i].reshape(-1, cols) for i in given}
        x2 = x.reshape(-1, depth) if wanted else None
        # (grad mode: the gradients are differentiated again.  Hooks on saved tensors may bring them back as something else, or in another layout)
        saved = ([x2] if wanted else []) + (w if of_x else [])
        like = g2[given[0]]
        as_saved = (not wanted or x.shape == ctx.x_shape) and all(t.dtype == like.dtype and t.device == like.device for t in saved) and (not of_x or all(v.shape == (cols, depth) for v in w))
        own = as_saved and not torch.is_grad_enabled() and not _watched() and _memory_says_all(*saved, *(dy[i] for i in given))
        rows = like.shape[0]
        if own:
            g2 = {i: ops._dense16(g) for i, g in g2.items()}
        if of_x:
            gs, ws = [g2[i] for i in given], [w[i] for i in given]
            if own and ops.gemm_preferred("xw", rows, depth, cols, cols, depth, len(gs), True):
                dx = ops.launch_gemm("xw", rows, depth, cols, cols, depth, gs, [ops._dense16(v) for v in ws], total=True, lead=ctx.x_shape[:-1])
            else:
                for g, v in zip(gs, ws):
                    dx = g @ v if dx is None else dx + g @ v
                dx = dx.reshape(ctx.x_shape)
        if wanted:
            if own and ops.gemm_preferred("xtx", cols, depth, rows, cols, depth, len(wanted)):
                x2 = ops._dense16(x2)
                for i, made in zip(wanted, ops.launch_gemm("xtx", cols, depth, rows, cols, depth, [g2[i] for i in wanted], [x2] * len(wanted))):
                    dw[i] = made
            else:
                for i in wanted:
                    dw[i] = g2[i].t() @ x2
        return (None, dx, *dw)


def linear(layers: Sequence[nn.Module], x: torch.Tensor) -> list:
    """``[m(x) for m in layers]``: up to three layers without bias."""
    rows, recording, first = x.shape[:-1].numel(), torch.is_grad_enabled(), layers[0]
    if rows < (FEWEST_ROWS_BACKWARD if recording else FEWEST_ROWS) or type(first) is not nn.Linear or first.in_features != x.shape[-1] or not _plain_input(x):
        return [m(x) for m in layers]
    cols, depth = first.out_features, first.in_features
    forward, backward = _own(rows, cols, depth, len(layers), recording)
    ws = _weights(layers, x, cols, depth) if forward or backward else None
    if ws is None:
        return [m(x) for m in layers]
    made = ops.launch_gemm("xwt", rows, cols, depth, depth, depth, [x] * len(ws), ws, lead=x.shape[:-1]) if forward else None
    if recording and (x.requires_grad or any(w.requires_grad for w in ws)):
        return list(_LinearFn.apply(made, x, *ws))
    return made if made is not None else [m(x) for m in layers]


def linear_one(layer: nn.Module, x: torch.Tensor) -> torch.Tensor:
    """``layer(x)``"""
    if x.shape[:-1].numel() < (FEWEST_ROWS_BACKWARD if torch.is_grad_enabled() else FEWEST_ROWS):
        return layer(x)
    return linear([layer], x)[0]
