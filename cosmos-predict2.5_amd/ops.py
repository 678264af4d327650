"""Host side of the HIP attention forward + JVP: argument checks, workspace, launch.

``fwd_jvp`` is the one function that talks to the C ABI.  It takes heads-first views
``[B, H, L, d]`` (any batch/head/row strides, innermost stride 1), launches on torch's current
stream, never synchronises, and allocates outputs with ``torch.empty`` like the reference wrapper
(cosmos_predict2/_src/predict2/utils/flash_attention_jvp_triton.py:451-455).
"""
from __future__ import annotations

import ctypes
import functools
import struct
from typing import Optional, Tuple

import torch

from . import _lib

_DTYPES = {torch.bfloat16: _lib.DTYPE_BF16, torch.float16: _lib.DTYPE_FP16}
SUPPORTED_HEAD_DIMS = (16, 32, 64, 128, 256)   # (attention at 256 runs slower kernels of its own)
FORWARD_HEAD_DIMS = SUPPORTED_HEAD_DIMS
REFERENCE_HEAD_DIMS = (16, 32, 64, 128, 256)  # what the reference accepts (…jvp_triton.py:444-445)


def _kernel_ready(x: torch.Tensor) -> bool:
    """True if the view can be handed to the kernel as is: d stride 1, 16-byte rows and base."""
    *outer, last = x.stride()
    if last != 1 or x.data_ptr() % 16:
        return False
    for s in outer:
        if s % 8:
            return False
    return True


def _prep_pair(x: torch.Tensor, tx: Optional[torch.Tensor]):
    """Primal and tangent must end up with identical strides (the kernel reads both through one set)."""
    if tx is None:
        return (x if _kernel_ready(x) else x.contiguous()), None
    if _kernel_ready(x) and _kernel_ready(tx) and x.stride() == tx.stride():
        return x, tx
    return x.contiguous(), tx.contiguous()


_Int64x3 = ctypes.c_int64 * 3


def _strides3(x: torch.Tensor):
    return _Int64x3(*x.stride()[:3])


def _on_device(device: torch.device, launch):
    """``launch(stream)`` with ``device`` current, ``stream`` its current stream's handle.  The usual case, that it is current
    already, goes without torch's device guard and stream object: they cost 5 us a call."""
    if torch.cuda.current_device() == device.index:
        return launch(torch._C._cuda_getCurrentRawStream(device.index))
    with torch.cuda.device(device):
        return launch(torch.cuda.current_stream(device).cuda_stream)


def _alloc_outputs(B, H, Lq, d_v, q, have_tangent, out_layout, need_lse):
    if out_layout == "bhld":
        o = torch.empty((B, H, Lq, d_v), device=q.device, dtype=q.dtype)
        to = torch.empty_like(o) if have_tangent else None
    elif out_layout == "blhd" and have_tangent:
        # o and to as the two halves of one buffer: a following linear layer maps both in one GEMM without a copy
        both = torch.empty((2, B, Lq, H, d_v), device=q.device, dtype=q.dtype)
        o, to = both[0].transpose(1, 2), both[1].transpose(1, 2)
    elif out_layout == "blhd":
        o, to = torch.empty((B, Lq, H, d_v), device=q.device, dtype=q.dtype).transpose(1, 2), None
    else:
        raise ValueError(f"out_layout={out_layout!r}")
    lse = torch.empty((B, H, Lq), device=q.device, dtype=torch.float32) if need_lse else None
    return o, to, lse


def fwd_jvp(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    tq: Optional[torch.Tensor] = None,
    tk: Optional[torch.Tensor] = None,
    tv: Optional[torch.Tensor] = None,
    causal: bool = False,
    sm_scale: Optional[float] = None,
    key_lens: Optional[torch.Tensor] = None,
    out_layout: str = "bhld",
    need_lse: bool = True,
) -> Tuple[torch.Tensor, Optional[torch.Tensor], Optional[torch.Tensor]]:
    """(o, to, lse) for q,k,v (+ tangents) given as ``[B, H, L, d]`` views on one GPU.

    Tangents: none (forward only, ``to`` is None), ``tq`` only, or any mix (missing ones are
    treated as zeros).  ``out_layout``: "bhld" -> o is contiguous ``[B,H,Lq,dv]``; "blhd" -> the
    memory is contiguous ``[B,Lq,H,dv]`` and a ``[B,H,Lq,dv]`` view of it is returned.
    ``key_lens``: optional int32 ``[B]`` device tensor, keys >= key_lens[b] are masked.
    """
    assert q.dim() == 4 and k.dim() == 4 and v.dim() == 4, "q, k, v must be [B, H, L, d]"
    assert q.shape[:-2] == k.shape[:-2] and k.shape[:-2] == v.shape[:-2]
    assert k.shape[-2] == v.shape[-2] and q.shape[-1] == k.shape[-1]
    B, H, Lq, d_qk = q.shape
    Lkv, d_v = v.shape[-2], v.shape[-1]
    assert d_qk in REFERENCE_HEAD_DIMS and d_v in REFERENCE_HEAD_DIMS
    if d_qk not in FORWARD_HEAD_DIMS or d_v not in FORWARD_HEAD_DIMS:
        raise NotImplementedError(f"head dims ({d_qk}, {d_v}): the HIP kernels are built for {FORWARD_HEAD_DIMS}")
    assert (Lq == Lkv) or (not causal), "Causal cross-attention is currently not supported."
    if not q.is_cuda:
        raise RuntimeError("cosmos attention (HIP) needs tensors on a GPU; there is no CPU path")
    if q.dtype not in _DTYPES:
        raise NotImplementedError(f"dtype={q.dtype} is not supported (bf16 / fp16)")
    assert k.dtype == q.dtype and v.dtype == q.dtype
    assert k.device == q.device and v.device == q.device
    for t_, x_ in ((tq, q), (tk, k), (tv, v)):
        if t_ is not None:
            assert t_.shape == x_.shape and t_.dtype == x_.dtype and t_.device == x_.device

    have_tangent = any(t_ is not None for t_ in (tq, tk, tv))
    if have_tangent and tq is None:
        tq = torch.zeros_like(q)
    if tk is not None or tv is not None:  # kernels are built for: none / q only / all three
        tk = torch.zeros_like(k) if tk is None else tk
        tv = torch.zeros_like(v) if tv is None else tv
    q, tq = _prep_pair(q, tq)
    k, tk = _prep_pair(k, tk)
    v, tv = _prep_pair(v, tv)

    if sm_scale is None:
        sm_scale = d_qk ** (-0.5)

    o, to, lse = _alloc_outputs(B, H, Lq, d_v, q, have_tangent, out_layout, need_lse)

    if key_lens is not None:
        assert not causal, "key_lens with causal is not supported"
        key_lens = key_lens.to(device=q.device, dtype=torch.int32).contiguous()
        assert key_lens.shape == (B,)

    desc = _lib.AttnDesc()
    desc.abi_version = _lib.ABI_VERSION
    desc.dtype = _DTYPES[q.dtype]
    desc.B, desc.H, desc.Lq, desc.Lkv, desc.d_qk, desc.d_v = B, H, Lq, Lkv, d_qk, d_v
    desc.causal = 1 if causal else 0
    desc.sm_scale = float(sm_scale)
    desc.q, desc.k, desc.v = q.data_ptr(), k.data_ptr(), v.data_ptr()
    desc.tq = tq.data_ptr() if tq is not None else None
    desc.tk = tk.data_ptr() if tk is not None else None
    desc.tv = tv.data_ptr() if tv is not None else None
    desc.q_stride, desc.k_stride, desc.v_stride = _strides3(q), _strides3(k), _strides3(v)
    desc.o, desc.to = o.data_ptr(), (to.data_ptr() if to is not None else None)
    desc.o_stride = _strides3(o)
    desc.lse = lse.data_ptr() if lse is not None else None
    desc.key_lens = key_lens.data_ptr() if key_lens is not None else None

    lib = _lib.load_library()
    ws_bytes = lib.cosmos_attn_workspace_bytes(ctypes.byref(desc))
    if ws_bytes == 0:
        # invalid descriptor: let the launch entry produce the precise status
        _lib.raise_for_status(lib.cosmos_attn_fwd_jvp(ctypes.byref(desc), None, 0, None) or _lib.ST_BAD_ARG)
    workspace = torch.empty(ws_bytes, device=q.device, dtype=torch.uint8)
    _lib.raise_for_status(_on_device(q.device, lambda stream: lib.cosmos_attn_fwd_jvp(ctypes.byref(desc), workspace.data_ptr(), ws_bytes, stream)))
    # workspace / converted inputs are freed to torch's caching allocator here; it is stream-ordered on
    # the launch stream, so reuse by later work on this stream is safe.
    return o, to, lse


# struct cosmos_attn_desc in one go: the fields one by one take 2.5 us, a tenth of a small call
_ATTN_DESC = struct.Struct("@9if6Q9q2Q3q2Q")
assert _ATTN_DESC.size == ctypes.sizeof(_lib.AttnDesc)
_ONE_DESCRIPTOR_ROWS = 6144      # (of a longer call nobody sees the host's share)


def forward_short(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, causal: bool, sm_scale: Optional[float]) -> Optional[torch.Tensor]:
    """Forward-only attention of ``[B, S, H, 128]`` tensors, up to some thousand queries, with the least work on the host: one packed descriptor, given to the call
    that reads k and v where they are, and where the library does not do that, to the one that re-tiles them.  None where the call is another one, whatever is
    wrong or special about it.  A pass of few queries, us, here / through ``fwd_jvp``: in place 12 / 27, re-tiled 17 / 27."""
    if q.dim() != 4 or k.dim() != 4 or not q.is_cuda:
        return None
    B, S, H, D = q.shape
    Lkv = k.shape[1]
    if D != 128 or S > _ONE_DESCRIPTOR_ROWS or k.shape != (B, Lkv, H, D) or v.shape != (B, Lkv, H, D):
        return None
    code, device = _DTYPES.get(q.dtype), q.device
    if code is None or k.dtype != q.dtype or v.dtype != q.dtype or k.device != device or v.device != device or (causal and S != Lkv) or min(B, S, H, Lkv) < 1:
        return None
    qb, ql, qh, q1 = q.stride()
    kb, kl, kh, k1 = k.stride()
    vb, vl, vh, v1 = v.stride()
    pq, pk, pv = q.data_ptr(), k.data_ptr(), v.data_ptr()
    if q1 != 1 or k1 != 1 or v1 != 1 or (pq | pk | pv) & 15 or (qb | ql | qh | kb | kl | kh | vb | vl | vh) & 7:
        return None
    o = torch.empty((B, S, H, D), device=device, dtype=q.dtype)
    desc = _ATTN_DESC.pack(_lib.ABI_VERSION, code, B, H, S, Lkv, D, D, 1 if causal else 0, D ** -0.5 if sm_scale is None else sm_scale,
                           pq, pk, pv, 0, 0, 0, qb, qh, ql, kb, kh, kl, vb, vh, vl, o.data_ptr(), 0, S * H * D, D, H * D, 0, 0)
    lib = _lib.load_library()
    status = _on_device(device, lambda stream: lib.cosmos_attn_fwd_in_place(desc, stream))
    if status == _lib.ST_WORKSPACE:
        same = _lib.AttnDesc.from_buffer_copy(desc)
        ws_bytes = lib.cosmos_attn_workspace_bytes(same)
        workspace = torch.empty(ws_bytes, device=device, dtype=torch.uint8)
        status = _on_device(device, lambda stream: lib.cosmos_attn_fwd_jvp(same, workspace.data_ptr(), ws_bytes, stream))
    _lib.raise_for_status(status)
    return o


class PackedKV:
    """The re-tiled image of one (k, v) pair (no tangents), made by :func:`pack_kv` and consumed by :func:`run_packed`:
    for keys and values that stay the same over many calls (the text context of the DiT's cross-attention)."""

    __slots__ = ("image", "B", "H", "Lkv", "d_qk", "d_v", "dtype", "device")

    def __init__(self, image, B, H, Lkv, d_qk, d_v, dtype, device):
        self.image, self.B, self.H, self.Lkv, self.d_qk, self.d_v, self.dtype, self.device = image, B, H, Lkv, d_qk, d_v, dtype, device


def _packed_desc(B, H, Lq, Lkv, d_qk, d_v, dtype, sm_scale):
    desc = _lib.AttnDesc()
    desc.abi_version = _lib.ABI_VERSION
    desc.dtype = _DTYPES[dtype]
    desc.B, desc.H, desc.Lq, desc.Lkv, desc.d_qk, desc.d_v = B, H, Lq, Lkv, d_qk, d_v
    desc.causal = 0
    desc.sm_scale = float(sm_scale)
    desc.tk = desc.tv = None
    return desc


def pack_kv(k: torch.Tensor, v: torch.Tensor) -> PackedKV:
    """Re-tile k, v (``[B, H, Lkv, d]`` views) once (``cosmos_attn_pack_kv``)."""
    assert k.dim() == 4 and v.dim() == 4 and k.shape[:-1] == v.shape[:-1]
    B, H, Lkv, d_qk = k.shape
    d_v = v.shape[-1]
    assert d_qk in REFERENCE_HEAD_DIMS and d_v in REFERENCE_HEAD_DIMS
    if d_qk not in FORWARD_HEAD_DIMS or d_v not in FORWARD_HEAD_DIMS:
        raise NotImplementedError(f"head dims ({d_qk}, {d_v}): the HIP kernels are built for {FORWARD_HEAD_DIMS}")
    if not k.is_cuda:
        raise RuntimeError("cosmos attention (HIP) needs tensors on a GPU; there is no CPU path")
    if k.dtype not in _DTYPES:
        raise NotImplementedError(f"dtype={k.dtype} is not supported (bf16 / fp16)")
    assert v.dtype == k.dtype and v.device == k.device
    k, _ = _prep_pair(k, None)
    v, _ = _prep_pair(v, None)
    desc = _packed_desc(B, H, 1, Lkv, d_qk, d_v, k.dtype, 1.0)
    desc.k, desc.v = k.data_ptr(), v.data_ptr()
    desc.k_stride, desc.v_stride = _strides3(k), _strides3(v)
    # pack_kv does not touch q / o: any valid addresses and strides pass the descriptor checks
    desc.q, desc.o, desc.tq, desc.to, desc.lse, desc.key_lens = k.data_ptr(), k.data_ptr(), None, None, None, None
    desc.q_stride, desc.o_stride = _strides3(k), _strides3(k)
    lib = _lib.load_library()
    nbytes = lib.cosmos_attn_packed_bytes(ctypes.byref(desc))
    if nbytes == 0:
        _lib.raise_for_status(lib.cosmos_attn_pack_kv(ctypes.byref(desc), None, 0, None) or _lib.ST_BAD_ARG)
    image = torch.empty(nbytes, device=k.device, dtype=torch.uint8)
    _lib.raise_for_status(_on_device(k.device, lambda stream: lib.cosmos_attn_pack_kv(ctypes.byref(desc), image.data_ptr(), nbytes, stream)))
    return PackedKV(image, B, H, Lkv, d_qk, d_v, k.dtype, k.device)


def run_packed(
    q: torch.Tensor,
    packed: PackedKV,
    tq: Optional[torch.Tensor] = None,
    sm_scale: Optional[float] = None,
    key_lens: Optional[torch.Tensor] = None,
    out_layout: str = "bhld",
    need_lse: bool = True,
) -> Tuple[torch.Tensor, Optional[torch.Tensor], Optional[torch.Tensor]]:
    """:func:`fwd_jvp` (forward only, or tangent on q) against a packed (k, v): ``cosmos_attn_run``.  Same results, bit for bit,
    as the one-call form whenever that one does not cut key ranges (it never does with ``key_lens``)."""
    assert q.dim() == 4
    B, H, Lq, d_qk = q.shape
    assert (B, H, d_qk) == (packed.B, packed.H, packed.d_qk) and q.dtype == packed.dtype and q.device == packed.device
    if tq is not None:
        assert tq.shape == q.shape and tq.dtype == q.dtype and tq.device == q.device
    q, tq = _prep_pair(q, tq)
    d_v = packed.d_v
    if sm_scale is None:
        sm_scale = d_qk ** (-0.5)
    o, to, lse = _alloc_outputs(B, H, Lq, d_v, q, tq is not None, out_layout, need_lse)
    if key_lens is not None:
        key_lens = key_lens.to(device=q.device, dtype=torch.int32).contiguous()
        assert key_lens.shape == (B,)
    desc = _packed_desc(B, H, Lq, packed.Lkv, d_qk, d_v, q.dtype, sm_scale)
    desc.q, desc.tq = q.data_ptr(), (tq.data_ptr() if tq is not None else None)
    desc.k = desc.v = packed.image.data_ptr()          # only tested for NULL by cosmos_attn_run
    desc.q_stride = _strides3(q)
    desc.k_stride = desc.v_stride = (ctypes.c_int64 * 3)(packed.H * packed.Lkv * 8, packed.Lkv * 8, 8)
    desc.o, desc.to = o.data_ptr(), (to.data_ptr() if to is not None else None)
    desc.o_stride = _strides3(o)
    desc.lse = lse.data_ptr() if lse is not None else None
    desc.key_lens = key_lens.data_ptr() if key_lens is not None else None
    lib = _lib.load_library()
    _lib.raise_for_status(_on_device(q.device, lambda stream: lib.cosmos_attn_run(
        ctypes.byref(desc), packed.image.data_ptr(), packed.image.numel(), stream)))
    return o, to, lse


def bwd(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    o: torch.Tensor,
    lse: torch.Tensor,
    dout: torch.Tensor,
    causal: bool = False,
    sm_scale: Optional[float] = None,
    max_ds_mib: Optional[int] = None,
) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """(dq, dk, dv) for the cotangent ``dout`` of o; all tensors ``[B, H, L, d]`` views on one GPU, ``lse`` the
    forward's ``[B, H, Lq]`` fp32.  Mirrors the reference's ``_attention.backward``
    (cosmos_predict2/_src/predict2/utils/flash_attention_jvp_triton.py:505-561): equal head dims only (:507-509),
    outputs allocated like ``torch.empty_like`` of q, k, v (:513).

    ``max_ds_mib``: workspace the call may spend on keeping the 16-bit dS tiles between its two passes (the descriptor's
    field of that name; negative = never).  Default: 32 GiB, but no more than 40 % of the device memory free right now.
    """
    assert q.shape[-1] == k.shape[-1] and k.shape[-1] == v.shape[-1], "Backward not supported with different headdim."
    B, H, Lq, d = q.shape
    Lkv = k.shape[-2]
    assert k.shape == (B, H, Lkv, d) and v.shape == (B, H, Lkv, d)
    assert o.shape == q.shape and dout.shape == q.shape and lse.shape == (B, H, Lq)
    assert d in REFERENCE_HEAD_DIMS
    if d not in FORWARD_HEAD_DIMS:
        raise NotImplementedError(f"head dim {d}: the HIP kernels are built for {FORWARD_HEAD_DIMS}")
    assert (Lq == Lkv) or (not causal), "Causal cross-attention is currently not supported."
    if not q.is_cuda:
        raise RuntimeError("cosmos attention (HIP) needs tensors on a GPU; there is no CPU path")
    if q.dtype not in _DTYPES:
        raise NotImplementedError(f"dtype={q.dtype} is not supported (bf16 / fp16)")
    for x in (k, v, o, dout):
        assert x.dtype == q.dtype and x.device == q.device
    ready = lambda x: x if _kernel_ready(x) else x.contiguous()
    q, k, v, o, dout = (ready(x) for x in (q, k, v, o, dout))
    lse = lse.to(torch.float32).contiguous()
    if sm_scale is None:
        sm_scale = d ** (-0.5)
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    if not all(_kernel_ready(x) for x in (dq, dk, dv)):   # empty_like of an exotic view: fall back to plain layouts
        dq, dk, dv = (torch.empty(x.shape, device=x.device, dtype=x.dtype) for x in (q, k, v))

    desc = _lib.AttnBwdDesc()
    desc.abi_version = _lib.ABI_VERSION
    desc.dtype = _DTYPES[q.dtype]
    desc.B, desc.H, desc.Lq, desc.Lkv, desc.d = B, H, Lq, Lkv, d
    desc.causal = 1 if causal else 0
    desc.sm_scale = float(sm_scale)
    if max_ds_mib is None:
        free_bytes, _ = torch.cuda.mem_get_info(q.device)
        max_ds_mib = max(1, min(32 * 1024, int(0.4 * free_bytes) >> 20))
    desc.max_ds_mib = int(max_ds_mib)
    desc.q, desc.k, desc.v, desc.o, desc.dout = (x.data_ptr() for x in (q, k, v, o, dout))
    desc.lse = lse.data_ptr()
    desc.dq, desc.dk, desc.dv = dq.data_ptr(), dk.data_ptr(), dv.data_ptr()
    desc.q_stride, desc.k_stride, desc.v_stride = _strides3(q), _strides3(k), _strides3(v)
    desc.o_stride, desc.dout_stride = _strides3(o), _strides3(dout)
    desc.dq_stride, desc.dk_stride, desc.dv_stride = _strides3(dq), _strides3(dk), _strides3(dv)

    lib = _lib.load_library()
    ws_bytes = lib.cosmos_attn_bwd_workspace_bytes(ctypes.byref(desc))
    if ws_bytes == 0:
        _lib.raise_for_status(lib.cosmos_attn_bwd(ctypes.byref(desc), None, 0, None) or _lib.ST_BAD_ARG)
    workspace = torch.empty(ws_bytes, device=q.device, dtype=torch.uint8)
    _lib.raise_for_status(_on_device(q.device, lambda stream: lib.cosmos_attn_bwd(ctypes.byref(desc), workspace.data_ptr(), ws_bytes, stream)))
    return dq, dk, dv


def _norm_weight(weight: Optional[torch.Tensor], x: torch.Tensor) -> Optional[torch.Tensor]:
    """RMSNorm's weight as the kernels take it: of the element type as it is, anything else as fp32."""
    if weight is None:
        return None
    if weight.dtype == x.dtype and weight.device == x.device and weight.is_contiguous() and weight.data_ptr() % 16 == 0:
        return weight
    return weight.to(device=x.device, dtype=torch.float32).contiguous()


def _norm_rope_dtype(x: torch.Tensor, weight: Optional[torch.Tensor]) -> int:
    return _DTYPES[x.dtype] | (_lib.NORM_ROPE_WEIGHT_16 if weight is not None and weight.dtype == x.dtype else 0)


def norm_rope(
    x: torch.Tensor,
    weight: Optional[torch.Tensor] = None,
    rope_emb: Optional[torch.Tensor] = None,
    tx: Optional[torch.Tensor] = None,
    eps: float = 1e-6,
    out_layout: str = "bshd",
) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """Per-head RMSNorm followed by the rotary embedding, and the tangent of both for ``tx``: what the DiT does to q and
    k between the projections and the attention call (cosmos_predict2/_src/predict2/networks/minimal_v4_dit.py:405-415).

    ``x`` (and ``tx``): ``[B, S, H, D]`` 16-bit; ``weight``: RMSNorm's ``[D]`` parameter (None = ones);
    ``rope_emb``: the angles ``[S, 1, 1, D]`` / ``[S, D]`` of minimal_v4_dit.py:648-658 (None = no rotation, as for
    cross-attention keys).  Returns ``(y, ty)`` with the shape of ``x``; ``out_layout="bhsd"`` makes the memory
    heads-first (a ``[B, S, H, D]`` view of it is returned), ready for the attention kernels without a transpose.
    """
    assert x.dim() == 4, "x must be [B, S, H, D]"
    B, S, H, D = x.shape
    assert D in REFERENCE_HEAD_DIMS
    if D not in SUPPORTED_HEAD_DIMS:
        raise NotImplementedError(f"head dim {D}: the HIP kernels are built for {SUPPORTED_HEAD_DIMS}")
    if x.dtype not in _DTYPES:
        raise NotImplementedError(f"dtype={x.dtype} is not supported (bf16 / fp16)")
    if tx is not None:
        assert tx.shape == x.shape and tx.dtype == x.dtype and tx.device == x.device
    assert weight is None or weight.shape == (D,)
    assert rope_emb is None or rope_emb.numel() == S * D, "rope_emb must hold one angle per (position, channel)"
    if not x.is_cuda:
        raise RuntimeError("cosmos attention (HIP) needs tensors on a GPU; there is no CPU path")
    x, tx = _prep_pair(x, tx)
    weight = _norm_weight(weight, x)
    if rope_emb is not None:
        rope_emb = rope_emb.to(device=x.device, dtype=torch.float32).reshape(S, D).contiguous()
    if out_layout == "bshd":
        y = torch.empty((B, S, H, D), device=x.device, dtype=x.dtype)
    elif out_layout == "bhsd":
        y = torch.empty((B, H, S, D), device=x.device, dtype=x.dtype).transpose(1, 2)
    else:
        raise ValueError(f"out_layout={out_layout!r}")
    ty = torch.empty_like(y) if tx is not None else None

    desc = _lib.NormRopeDesc()
    desc.abi_version = _lib.ABI_VERSION
    desc.dtype = _norm_rope_dtype(x, weight)
    desc.B, desc.S, desc.H, desc.D = B, S, H, D
    desc.eps = float(eps)
    desc.reserved = 0
    desc.x, desc.tx = x.data_ptr(), (tx.data_ptr() if tx is not None else None)
    desc.weight = weight.data_ptr() if weight is not None else None
    desc.angles = rope_emb.data_ptr() if rope_emb is not None else None
    desc.y, desc.ty = y.data_ptr(), (ty.data_ptr() if ty is not None else None)
    desc.x_stride, desc.y_stride = _strides3(x), _strides3(y)
    _launch("cosmos_norm_rope", desc, x.device)
    return y, ty


def norm_rope_bwd(
    x: torch.Tensor,
    weight: Optional[torch.Tensor],
    rope_emb: Optional[torch.Tensor],
    dy: torch.Tensor,
    eps: float = 1e-6,
    need_dweight: bool = True,
) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """Reverse mode of :func:`norm_rope`: ``(dx, dweight)`` from the gradient ``dy`` of its output.  ``x``, ``dy``:
    ``[B, S, H, D]`` views (any batch / sequence / head strides that are multiples of 8 elements); ``dx`` is contiguous
    ``[B, S, H, D]``; ``dweight`` is fp32 ``[D]`` (None if not wanted).  This is what autograd derives for the RMSNorm and
    rotary ops of cosmos_predict2/_src/predict2/networks/minimal_v4_dit.py:405-415."""
    assert x.dim() == 4 and dy.shape == x.shape and dy.dtype == x.dtype and dy.device == x.device
    B, S, H, D = x.shape
    assert D in REFERENCE_HEAD_DIMS
    if D not in SUPPORTED_HEAD_DIMS:
        raise NotImplementedError(f"head dim {D}: the HIP kernels are built for {SUPPORTED_HEAD_DIMS}")
    if x.dtype not in _DTYPES:
        raise NotImplementedError(f"dtype={x.dtype} is not supported (bf16 / fp16)")
    assert weight is None or weight.shape == (D,)
    assert rope_emb is None or rope_emb.numel() == S * D, "rope_emb must hold one angle per (position, channel)"
    if not x.is_cuda:
        raise RuntimeError("cosmos attention (HIP) needs tensors on a GPU; there is no CPU path")
    x = x if _kernel_ready(x) else x.contiguous()
    dy = dy if _kernel_ready(dy) else dy.contiguous()
    weight = _norm_weight(weight, x)
    if rope_emb is not None:
        rope_emb = rope_emb.to(device=x.device, dtype=torch.float32).reshape(S, D).contiguous()
    dx = torch.empty((B, S, H, D), device=x.device, dtype=x.dtype)
    dweight = torch.empty((D,), device=x.device, dtype=torch.float32) if need_dweight else None

    desc = _lib.NormRopeBwdDesc()
    desc.abi_version = _lib.ABI_VERSION
    desc.dtype = _norm_rope_dtype(x, weight)
    desc.B, desc.S, desc.H, desc.D = B, S, H, D
    desc.eps = float(eps)
    desc.reserved = 0
    desc.x, desc.dy, desc.dx = x.data_ptr(), dy.data_ptr(), dx.data_ptr()
    desc.weight = weight.data_ptr() if weight is not None else None
    desc.angles = rope_emb.data_ptr() if rope_emb is not None else None
    desc.dweight = dweight.data_ptr() if dweight is not None else None
    desc.x_stride, desc.dy_stride, desc.dx_stride = _strides3(x), _strides3(dy), _strides3(dx)
    _launch_with_workspace("cosmos_norm_rope_bwd", desc, x.device)
    return dx, dweight


# ------------------------------------------------------------------ elementwise steps of the DiT block (+ tangents)
def stacked_pair(shape, dtype, device):
    """Two tensors of ``shape`` that are the halves of one ``[2, *shape]`` buffer (see :func:`as_stacked`)."""
    both = torch.empty((2, *shape), device=device, dtype=dtype)
    return both[0], both[1]


def as_stacked(x: torch.Tensor, tx: torch.Tensor) -> Optional[torch.Tensor]:
    """If ``x`` and ``tx`` are the two contiguous halves of one buffer, the ``[2 * x.shape[0], ...]`` view of it (no
    copy); otherwise None."""
    if (x.shape == tx.shape and x.dtype == tx.dtype and x.is_contiguous() and tx.is_contiguous() and x.dim() >= 1
            and x._base is not None and x._base is tx._base
            and tx.data_ptr() == x.data_ptr() + x.numel() * x.element_size()):
        both = x._base
        if both.is_contiguous() and both.data_ptr() == x.data_ptr() and both.numel() == 2 * x.numel():
            return both.view(2 * x.shape[0], *x.shape[1:])
    return None


def _is_dense16(t: torch.Tensor) -> bool:
    return t.is_contiguous() and t.data_ptr() % 16 == 0


def _dense16(t: torch.Tensor) -> torch.Tensor:
    """``t``, or a copy where it is not contiguous or does not start at 16 bytes (``.contiguous()`` returns a contiguous slice of a
    larger buffer as it is, wherever that starts)."""
    return t if _is_dense16(t) else t.clone(memory_format=torch.contiguous_format)


def _check_elementwise(x: torch.Tensor) -> None:
    if not x.is_cuda:
        raise RuntimeError("cosmos attention (HIP) needs tensors on a GPU; there is no CPU path")
    if x.dtype not in _DTYPES:
        raise NotImplementedError(f"dtype={x.dtype} is not supported (bf16 / fp16)")


def _check_outputs(x: torch.Tensor, *outs: Optional[torch.Tensor]) -> None:
    """Outputs that a caller may have preallocated: the kernels write ``x.numel()`` elements of ``x``'s type there."""
    for t in outs:
        assert t is None or (t.is_contiguous() and t.shape == x.shape and t.dtype == x.dtype and t.device == x.device)


def _launch(fn_name: str, desc, device) -> None:
    fn = getattr(_lib.load_library(), fn_name)
    _lib.raise_for_status(_on_device(device, lambda stream: fn(ctypes.byref(desc), stream)))


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def ln_modulate(x, shift, scale, tx=None, tshift=None, tscale=None, eps: float = 1e-6, out=None, tout=None):
    """``LayerNorm(x) * (1 + scale) + shift`` over the last dim (no affine parameters) and its tangent, one pass
    (cosmos_predict2/_src/predict2/networks/minimal_v4_dit.py:1166-1167).  ``x``: ``[..., D]``; ``shift`` / ``scale``:
    ``[G, D]`` with ``G`` dividing the number of rows (consecutive rows share a vector).  ``out`` / ``tout``: optional
    preallocated outputs (e.g. the two halves of one stacked buffer).  Returns ``(y, ty)``."""
    _check_elementwise(x)
    D = x.shape[-1]
    x = _dense16(x)
    rows = x.numel() // D
    shift, scale = _dense16(shift.to(x.dtype)).reshape(-1, D), _dense16(scale.to(x.dtype)).reshape(-1, D)
    assert shift.shape == scale.shape and rows % shift.shape[0] == 0
    if tx is not None:
        assert tx.shape == x.shape and tx.dtype == x.dtype
        tx = _dense16(tx)
        tshift = None if tshift is None else _dense16(tshift.to(x.dtype)).reshape(-1, D)
        tscale = None if tscale is None else _dense16(tscale.to(x.dtype)).reshape(-1, D)
        assert (tshift is None or tshift.shape == shift.shape) and (tscale is None or tscale.shape == shift.shape)
    y = torch.empty_like(x) if out is None else out
    ty = (torch.empty_like(x) if tout is None else tout) if tx is not None else None
    _check_outputs(x, y, ty)
    d = _lib.LnModulateDesc()
    d.abi_version, d.dtype = _lib.ABI_VERSION, _DTYPES[x.dtype]
    d.D, d.rows_per_group, d.eps, d.reserved, d.rows = D, rows // shift.shape[0], float(eps), 0, rows
    d.x, d.tx, d.shift, d.scale = _ptr(x), _ptr(tx), _ptr(shift), _ptr(scale)
    d.tshift, d.tscale = (_ptr(tshift), _ptr(tscale)) if tx is not None else (None, None)
    d.y, d.ty = _ptr(y), _ptr(ty)
    _launch("cosmos_ln_modulate", d, x.device)
    return y, ty


def gated_residual(x, res, gate, tx=None, tres=None, tgate=None, inplace: bool = False):
    """``x + gate * res`` and its tangent ``tx + tgate * res + gate * tres`` in one pass
    (cosmos_predict2/_src/predict2/networks/minimal_v4_dit.py:1199, :1231, :1241).  ``gate``: ``[G, D]`` as in
    :func:`ln_modulate`.  ``inplace`` overwrites ``x`` / ``tx``.  Returns ``(out, tout)``."""
    _check_elementwise(x)
    D = x.shape[-1]
    assert res.shape == x.shape and res.dtype == x.dtype
    xs, res = _dense16(x), _dense16(res)
    rows = xs.numel() // D
    gate = _dense16(gate.to(x.dtype)).reshape(-1, D)
    assert rows % gate.shape[0] == 0
    if tx is not None:
        assert tres is not None and tx.shape == x.shape and tres.shape == x.shape
        txs, tres = _dense16(tx), _dense16(tres)
        tgate = None if tgate is None else _dense16(tgate.to(x.dtype)).reshape(-1, D)
    else:
        txs = None
    out = xs if (inplace and xs is x) else torch.empty_like(xs)
    tout = None if tx is None else (txs if (inplace and txs is tx) else torch.empty_like(txs))
    d = _lib.GatedResidualDesc()
    d.abi_version, d.dtype = _lib.ABI_VERSION, _DTYPES[x.dtype]
    d.D, d.rows_per_group, d.rows = D, rows // gate.shape[0], rows
    d.x, d.tx, d.res, d.tres = _ptr(xs), _ptr(txs), _ptr(res), (_ptr(tres) if tx is not None else None)
    d.gate, d.tgate = _ptr(gate), (_ptr(tgate) if tx is not None else None)
    d.out, d.tout = _ptr(out), _ptr(tout)
    _launch("cosmos_gated_residual", d, x.device)
    return out, tout


def gated_residual_ln_modulate(x, res, gate, shift, scale, tx=None, tres=None, tgate=None, tshift=None, tscale=None,
                               eps: float = 1e-6, y=None, ty=None):
    """:func:`gated_residual` and :func:`ln_modulate` of its result in one pass (two, where ``gate`` and ``shift`` have different
    ``G``, or ``D > 5120``): ``(out, tout, y, ty)``.  ``y`` / ``ty``: optional preallocated outputs."""
    _check_elementwise(x)
    D = x.shape[-1]
    if gate.numel() != shift.numel():
        out, tout = gated_residual(x, res, gate, tx, tres, tgate)
        return out, tout, *ln_modulate(out, shift, scale, tout, tshift, tscale, eps=eps, out=y, tout=ty)
    assert res.shape == x.shape and res.dtype == x.dtype
    x, res = _dense16(x), _dense16(res)
    rows = x.numel() // D
    vector = lambda m: None if m is None else _dense16(m.to(x.dtype)).reshape(-1, D)
    gate, shift, scale = vector(gate), vector(shift), vector(scale)
    assert gate.shape == shift.shape == scale.shape and rows % gate.shape[0] == 0
    if tx is not None:
        assert tres is not None and tx.shape == x.shape == tres.shape and tx.dtype == x.dtype == tres.dtype
        tx, tres, tgate, tshift, tscale = _dense16(tx), _dense16(tres), vector(tgate), vector(tshift), vector(tscale)
        assert all(t is None or t.shape == gate.shape for t in (tgate, tshift, tscale))
    else:
        tres = tgate = tshift = tscale = ty = None
    out, tout = torch.empty_like(x), None if tx is None else torch.empty_like(x)
    y = torch.empty_like(x) if y is None else y
    ty = torch.empty_like(x) if ty is None and tx is not None else ty
    _check_outputs(x, y, ty)
    d = _lib.GatedResidualLnModulateDesc()
    d.abi_version, d.dtype = _lib.ABI_VERSION, _DTYPES[x.dtype]
    d.D, d.rows_per_group, d.eps, d.reserved, d.rows = D, rows // gate.shape[0], float(eps), 0, rows
    d.x, d.tx, d.res, d.tres, d.gate, d.tgate = _ptr(x), _ptr(tx), _ptr(res), _ptr(tres), _ptr(gate), _ptr(tgate)
    d.shift, d.scale, d.tshift, d.tscale = _ptr(shift), _ptr(scale), _ptr(tshift), _ptr(tscale)
    d.out, d.tout, d.y, d.ty = _ptr(out), _ptr(tout), _ptr(y), _ptr(ty)
    _launch("cosmos_gated_residual_ln_modulate", d, x.device)
    return out, tout, y, ty


def _launch_with_workspace(fn_name: str, desc, device) -> None:
    lib = _lib.load_library()
    fn, n = getattr(lib, fn_name), getattr(lib, fn_name + "_workspace_bytes")(ctypes.byref(desc))
    workspace = torch.empty(n, device=device, dtype=torch.uint8) if n else None
    _lib.raise_for_status(_on_device(device, lambda stream: fn(ctypes.byref(desc), _ptr(workspace), n, stream)))


def ln_modulate_bwd(x, scale, dy, dskip=None, eps: float = 1e-6):
    """Reverse mode of :func:`ln_modulate` (what autograd derives for
    cosmos_predict2/_src/predict2/networks/minimal_v4_dit.py:1166-1167): ``(dx, dshift, dscale)`` for the gradient ``dy`` of its
    output; ``dskip``: a gradient that reaches ``x`` on another way, added to ``dx``.  ``dshift`` / ``dscale``: ``[G, D]``."""
    _check_elementwise(x)
    D = x.shape[-1]
    assert dy.shape == x.shape and dy.dtype == x.dtype and (dskip is None or (dskip.shape == x.shape and dskip.dtype == x.dtype))
    xs, dy, dskip = _dense16(x), _dense16(dy), (None if dskip is None else _dense16(dskip))
    scale = _dense16(scale.to(x.dtype)).reshape(-1, D)
    rows = xs.numel() // D
    assert rows % scale.shape[0] == 0
    dx, dshift, dscale = torch.empty_like(xs), torch.empty_like(scale), torch.empty_like(scale)
    d = _lib.LnModulateBwdDesc()
    d.abi_version, d.dtype = _lib.ABI_VERSION, _DTYPES[x.dtype]
    d.D, d.rows_per_group, d.eps, d.reserved, d.rows = D, rows // scale.shape[0], float(eps), 0, rows
    d.x, d.scale, d.dy, d.dskip = _ptr(xs), _ptr(scale), _ptr(dy), _ptr(dskip)
    d.dx, d.dshift, d.dscale = _ptr(dx), _ptr(dshift), _ptr(dscale)
    _launch_with_workspace("cosmos_ln_modulate_bwd", d, x.device)
    return dx, dshift, dscale


def gated_residual_bwd(res, gate, dy):
    """Reverse mode of :func:`gated_residual` for ``res`` and ``gate``: ``(dres, dgate)``, ``dgate`` ``[G, D]``; the gradient of
    ``x`` is ``dy`` itself."""
    _check_elementwise(res)
    D = res.shape[-1]
    assert dy.shape == res.shape and dy.dtype == res.dtype
    res, dy, gate = _dense16(res), _dense16(dy), _dense16(gate.to(res.dtype)).reshape(-1, D)
    rows = res.numel() // D
    assert rows % gate.shape[0] == 0
    dres, dgate = torch.empty_like(res), torch.empty_like(gate)
    d = _lib.GatedResidualBwdDesc()
    d.abi_version, d.dtype = _lib.ABI_VERSION, _DTYPES[res.dtype]
    d.D, d.rows_per_group, d.rows = D, rows // gate.shape[0], rows
    d.dy, d.res, d.gate, d.dres, d.dgate = _ptr(dy), _ptr(res), _ptr(gate), _ptr(dres), _ptr(dgate)
    _launch_with_workspace("cosmos_gated_residual_bwd", d, res.device)
    return dres, dgate


def modulation(emb, lora, w1, w2, temb=None, tlora=None, tangent: bool = False):
    """The modulation vectors of a block's three sub-layers (cosmos_predict2/_src/predict2/networks/minimal_v4_dit.py:1131-1162):
    ``w2[i] (w1[i] silu(emb)) + lora`` for i = 0, 1, 2, as ``[3, 3, rows, D]`` (sub-layer; shift, scale, gate), and with
    ``tangent`` its derivative along (``temb``, ``tlora``; None = it does not move), else None.  ``emb``: ``[..., K]``;
    ``lora``: ``[..., 3 D]`` of as many rows; ``w1``: three ``[hidden, K]``; ``w2``: three ``[3 D, hidden]``; one 16-bit type."""
    _check_elementwise(emb)
    K, D = emb.shape[-1], lora.shape[-1] // 3
    rows, hidden = emb.numel() // K, w1[0].shape[0]
    assert lora.shape[-1] == 3 * D and lora.numel() == rows * 3 * D
    assert all(w.shape == (hidden, K) for w in w1) and all(w.shape == (3 * D, hidden) for w in w2)
    assert (temb is None or temb.shape == emb.shape) and (tlora is None or tlora.shape == lora.shape)
    ins = [None if t is None else _dense16(t) for t in (emb, temb, lora, tlora, *w1, *w2)]
    assert all(t is None or (t.dtype == emb.dtype and t.device == emb.device) for t in ins)
    assert tangent or (temb is None and tlora is None)
    out = torch.empty((3, 3, rows, D), device=emb.device, dtype=emb.dtype)
    tout = torch.empty_like(out) if tangent else None
    d = _lib.ModulationDesc()
    d.abi_version, d.dtype = _lib.ABI_VERSION, _DTYPES[emb.dtype]
    d.rows, d.K, d.hidden, d.D = rows, K, hidden, D
    d.emb, d.temb, d.lora, d.tlora = (_ptr(t) for t in ins[:4])
    for i in range(3):
        d.w1[i], d.w2[i] = _ptr(ins[4 + i]), _ptr(ins[7 + i])
    d.out, d.tout = _ptr(out), _ptr(tout)
    _launch_with_workspace("cosmos_ln_modulation", d, emb.device)
    return out, tout


GEMM_ORDERS = {"xwt": _lib.GEMM_XWT, "xw": _lib.GEMM_XW, "xtx": _lib.GEMM_XTX}


# struct cosmos_attn_gemm_desc in one go, as _ATTN_DESC
_GEMM_DESC = struct.Struct("@10i3q9Q")
assert _GEMM_DESC.size == ctypes.sizeof(_lib.GemmDesc)


def _pack_gemm(order: str, dtype: int, rows: int, cols: int, depth: int, lda: int, ldb: int, a, b, c, total: bool, shape: int = 0) -> bytes:
    three = lambda p: (*p, 0, 0)[:3]
    return _GEMM_DESC.pack(_lib.ABI_VERSION, dtype, GEMM_ORDERS[order], _lib.GEMM_SUM if total else 0, len(a), shape, rows, cols, depth, 0,
                           lda, ldb, cols, *three(a), *three(b), *three(c))


@functools.lru_cache(maxsize=4096)
def gemm_preferred(order: str, rows: int, cols: int, depth: int, lda: int, ldb: int, count: int = 1, total: bool = False) -> bool:
    """Does the library take ``count`` such products, and faster than the vendor's library does?  Follows from the sizes alone."""
    if max(rows, cols, depth) >= 1 << 31:
        return False
    at = (16,) * count
    return bool(_lib.load_library().cosmos_attn_gemm_preferred(_pack_gemm(order, _lib.DTYPE_BF16, rows, cols, depth, lda, ldb, at, at, at, total)))


def launch_gemm(order: str, rows: int, cols: int, depth: int, lda: int, ldb: int, a, b, total: bool = False, shape: int = 0, lead=None):
    """:func:`gemm` of operands that are known to be right: of tensors of any dimensions only the address is taken."""
    like = a[0]
    outs = [torch.empty((*(lead or (rows,)), cols), device=like.device, dtype=like.dtype) for _ in range(1 if total else len(a))]
    at = lambda ts: [t.data_ptr() for t in ts]
    D = _pack_gemm(order, _DTYPES[like.dtype], rows, cols, depth, lda, ldb, at(a), at(b), at(outs), total, shape)
    run = _lib.load_library().cosmos_attn_gemm
    _lib.raise_for_status(_on_device(like.device, lambda stream: run(D, stream)))
    return outs[0] if total else outs


def gemm(order: str, a, b, total: bool = False, shape: int = 0, if_preferred: bool = False, lead=None):
    """Up to three matrix products of one shape in one launch, 16-bit matrices, fp32 sums.  ``order``: "xwt" ``a [rows, depth]`` by the transpose of
    ``b [cols, depth]``; "xw" ``a [rows, depth]`` by ``b [depth, cols]``; "xtx" the transpose of ``a [depth, rows]`` by ``b [depth, cols]``.  Returns the
    list of ``[rows, cols]`` products; with ``total`` their sum alone.  Lines are read where they are (any line stride that is a multiple of 8).
    ``if_preferred``: None instead where the library's products are faster or the kernel does not take the matrices.  ``lead``: dimensions that the
    outputs have in the place of their rows."""
    assert 1 <= len(a) == len(b) <= 3
    _check_elementwise(a[0])
    for group, like in ((a, a[0]), (b, b[0])):
        for t in group:
            if t.dim() != 2 or t.shape != like.shape or t.stride() != like.stride() or t.stride(1) != 1:
                if if_preferred:
                    return None
                raise ValueError("the matrices of a launch need one shape and one line stride, with elements of a line side by side")
            if t.dtype != a[0].dtype or t.device != a[0].device:
                if if_preferred:
                    return None
                raise ValueError("the matrices of a launch need one type and device")
    rows, depth = a[0].shape if order != "xtx" else a[0].shape[::-1]
    cols, same = b[0].shape[::-1] if order != "xwt" else b[0].shape
    if depth != same:
        raise ValueError("the matrices' contractions differ")
    lda, ldb = a[0].stride(0), b[0].stride(0)
    if if_preferred and (any(t.data_ptr() % 16 for t in (*a, *b)) or not gemm_preferred(order, rows, cols, depth, lda, ldb, len(a), total)):
        return None
    return launch_gemm(order, rows, cols, depth, lda, ldb, a, b, total, shape, lead)


def gelu(h, th=None, inplace: bool = False):
    """Exact (erf) GELU and its tangent ``th * gelu'(h)`` in one pass (``nn.GELU()`` of
    cosmos_predict2/_src/predict2/networks/minimal_v4_dit.py:225).  Returns ``(a, ta)``."""
    _check_elementwise(h)
    hs = _dense16(h)
    assert hs.numel() % 8 == 0, "the number of elements must be a multiple of 8"
    ths = None
    if th is not None:
        assert th.shape == h.shape and th.dtype == h.dtype
        ths = _dense16(th)
    a = hs if (inplace and hs is h) else torch.empty_like(hs)
    ta = None if th is None else (ths if (inplace and ths is th) else torch.empty_like(ths))
    d = _lib.GeluDesc()
    d.abi_version, d.dtype, d.n = _lib.ABI_VERSION, _DTYPES[h.dtype], hs.numel()
    d.h, d.th, d.a, d.ta = _ptr(hs), _ptr(ths), _ptr(a), _ptr(ta)
    _launch("cosmos_gelu", d, h.device)
    return a, ta
