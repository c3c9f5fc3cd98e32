"""PyTorch-ROCm wrappers over the C ABI of ``libdflash_hip.so``.

Tensors must live on a ROCm device; every call is enqueued on the current
torch stream of that device, allocates its outputs and workspace through
torch, and raises :class:`DflashError` with the library's message on any
nonzero status.  There is no CPU or dense fallback (reference policy,
``model/qwen35_moe_dflash/fused/ops.py:133-135``).
"""
from __future__ import annotations

import contextlib
import ctypes
from typing import NamedTuple, Optional

import torch
from torch.autograd import forward_ad

from . import _lib
from .packing import PackedW4, SharedExpert


class Routing(NamedTuple):
    """Device routing of ``T`` tokens over ``E`` experts (see ``include/dflash_hip.h``)."""

    ids: torch.Tensor        # int32 [T, k]
    weights: torch.Tensor    # fp32 [T, k]
    perm: torch.Tensor       # int32 [T*k]
    inv: torch.Tensor        # int32 [T*k]
    offsets: torch.Tensor    # int32 [E+1]


def _require_device(*tensors) -> torch.device:
    device = None
    for t in tensors:
        if t is None:
            continue
        if not isinstance(t, torch.Tensor) or t.device.type != "cuda":
            raise ValueError("mi355x-hip operations require tensors on a ROCm device")
        if device is None:
            device = t.device
        elif t.device != device:
            raise ValueError("all tensors must be on the same device")
    if device is None:
        raise ValueError("no tensor given")
    return device


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _stream(device: torch.device):
    return ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)


def _desc(w: PackedW4) -> _lib.W4Desc:
    return _lib.W4Desc(
        packed=w.packed.data_ptr(), scales=w.scales.data_ptr(), experts=w.experts, rows=w.rows, cols=w.cols,
        group_size=w.group_size,
        scale_dtype=_lib.DTYPE_F32 if w.scales.dtype == torch.float32 else _lib.DTYPE_BF16,
        layout=_lib.LAYOUT_TILED if w.layout == "tiled" else _lib.LAYOUT_PORTABLE)


def _workspace(nbytes: int, device: torch.device, workspace: Optional[torch.Tensor]) -> torch.Tensor:
    if workspace is not None:
        if workspace.dtype != torch.uint8 or workspace.numel() < nbytes or workspace.device != device:
            raise ValueError(f"workspace must be a uint8 tensor of at least {nbytes} bytes on {device}")
        return workspace
    return torch.empty(max(nbytes, 256), dtype=torch.uint8, device=device)


_SOURCE_SCALE_DTYPES = {torch.float32: _lib.DTYPE_F32, torch.float16: _lib.DTYPE_F16, torch.bfloat16: _lib.DTYPE_BF16}


def from_int8(values: torch.Tensor, scales: torch.Tensor, group_size: int, *, layout: str = "tiled") -> PackedW4:
    """Pack the original checkpoint's int8-carried int4 weights into a bank with fp32 scales.

    ``values`` int8 ``[N, K]`` or ``[E, N, K]`` in [-8, 7]; ``scales`` fp16/fp32/bf16
    ``[..., N, K/G]`` (a linear's ``[N, K/G, 1]`` is accepted, as the reference's
    reader stores it: ``target/original_quant.py:214-240``).  Raises ``ValueError``
    with the reader's messages for values outside [-8, 7] and for negative or
    non-finite scales (``:252-272``); synchronises the stream to check them, as a
    load-time step.
    """
    device = _require_device(values, scales)
    if values.dtype != torch.int8 or values.ndim not in (2, 3):
        raise ValueError("original quantized weights must be int8 [N, K] or [E, N, K]")
    if layout not in ("portable", "tiled"):
        raise ValueError("layout must be 'portable' or 'tiled'")
    *lead, n, k = values.shape
    if k % group_size:
        raise ValueError(f"K={k} is not a multiple of group_size={group_size}")
    sc = scales.reshape(*scales.shape[:-1]) if scales.ndim == values.ndim + 1 and scales.shape[-1] == 1 else scales
    if tuple(sc.shape) != (*lead, n, k // group_size) or sc.dtype not in _SOURCE_SCALE_DTYPES:
        raise ValueError(f"scales must be fp16/fp32/bf16 [{', '.join(map(str, (*lead, n, k // group_size)))}]")
    vals, sc = values.contiguous(), sc.contiguous()
    packed = torch.empty((*lead, n, k // 2), dtype=torch.uint8, device=device)
    out_scales = torch.empty((*lead, n, k // group_size), dtype=torch.float32, device=device)
    invalid = torch.empty(2, dtype=torch.int32, device=device)
    _lib.call("dflash_w4_from_int8", _ptr(vals), _ptr(sc), _SOURCE_SCALE_DTYPES[sc.dtype], lead[0] if lead else 1,
              n, k, group_size, _lib.LAYOUT_TILED if layout == "tiled" else _lib.LAYOUT_PORTABLE, _ptr(packed),
              _ptr(out_scales), _ptr(invalid), _stream(device))
    bad_values, bad_scales = (int(v) for v in invalid.cpu())
    if bad_values:
        raise ValueError("original quantized weight contains values outside signed I4 [-8,7]")
    if bad_scales:
        raise ValueError("original quantization scales must be finite and nonnegative")
    return PackedW4(packed, out_scales, group_size, layout)


def to_tiled(w: PackedW4) -> PackedW4:
    """Repack a portable bank into the tiled layout (new tensors, same shapes, on w's device)."""
    w.validate("weight")
    if w.layout != "portable":
        raise ValueError("to_tiled needs a portable bank")
    device = _require_device(w.packed)
    packed = torch.empty_like(w.packed)
    scales = torch.empty_like(w.scales)
    desc = _desc(w)
    _lib.call("dflash_w4_to_tiled", ctypes.byref(desc), _ptr(packed), _ptr(scales), _stream(device))
    return PackedW4(packed, scales, w.group_size, "tiled")


def _plain(x) -> bool:
    """Whether a call on ``x`` is first offered to the native form (``csrc/host.cpp``, where there is one), which takes it
    or returns None."""
    return type(x) is torch.Tensor and x.is_cuda


def qlinear(x: torch.Tensor, weight: PackedW4, *, workspace: Optional[torch.Tensor] = None,
            out_dtype: torch.dtype = torch.bfloat16) -> torch.Tensor:
    """W4A16 linear ``x[..., K] -> [..., N]`` (bf16 in, fp32 accumulation; bf16 out, or the
    unrounded fp32 sums with ``out_dtype=torch.float32``)."""
    if (workspace is None and _plain(x) and (out_dtype is torch.bfloat16 or out_dtype is torch.float32)
            and (host := _lib.host())):
        y = host.linear(x, weight, out_dtype is torch.float32)
        if y is not None:
            return y
    weight.validate("weight")
    if weight.packed.ndim != 2:
        raise ValueError("qlinear takes one packed matrix [N, K/2]")
    if out_dtype not in (torch.bfloat16, torch.float32):
        raise ValueError("qlinear writes bfloat16 or float32")
    device = _require_device(x, weight.packed)
    if x.dtype != torch.bfloat16 or x.shape[-1] != weight.cols:
        raise ValueError(f"x must be bfloat16 [..., {weight.cols}]")
    flat = x.reshape(-1, weight.cols).contiguous()
    m = flat.shape[0]
    out = torch.empty((m, weight.rows), dtype=out_dtype, device=device)
    lib = _lib.load()
    ws = _workspace(lib.dflash_qlinear_workspace_bytes(m, weight.cols, weight.group_size), device, workspace)
    desc = _desc(weight)
    entry = "dflash_qlinear_w4a16_f32" if out_dtype == torch.float32 else "dflash_qlinear_w4a16"
    _lib.call(entry, _ptr(flat), m, ctypes.byref(desc), _ptr(out), _ptr(ws), ws.numel(), _stream(device))
    return out.reshape(*x.shape[:-1], weight.rows)


class GdnMixer(NamedTuple):
    """Outputs of :func:`gdn_mixer` (see ``dflash_gdn_mixer`` in ``include/dflash_hip.h``)."""

    mid: torch.Tensor        # fp32 [T, H] residual after the mixer
    normed: torch.Tensor     # bf16 [T, H] its post-norm
    window: torch.Tensor     # bf16 [1, C, 3 + T]
    tail: torch.Tensor       # bf16 [1, C, 3], its last columns
    states: torch.Tensor     # fp32 [chunks, 1, Hv, 128, 128]
    keys: torch.Tensor       # fp32 [1, Hv, T, 128]
    u: torch.Tensor          # fp32 [1, Hv, T, 128]
    cum: torch.Tensor        # fp32 [1, Hv, T]
    core: torch.Tensor       # fp32 [1, Hv, T, 128]


def gdn_mixer(hidden: torch.Tensor, history: torch.Tensor, state: torch.Tensor, *, in_proj: PackedW4,
              out_proj: PackedW4, input_norm: torch.Tensor, post_norm: torch.Tensor, norm: torch.Tensor,
              a_log: torch.Tensor, dt_bias: torch.Tensor, conv: torch.Tensor, key_heads: int, eps: float) -> GdnMixer:
    """A GDN layer from its residual to the MoE input, in one call: norm, in_proj, conv, gated delta rule, gated
    norm, out_proj, residual add, post-norm.  Tensors as :func:`gdn_mixer_fits` accepts them."""
    device, t, h = hidden.device, hidden.shape[0], hidden.shape[1]
    hv = a_log.shape[0]
    f32 = dict(dtype=torch.float32, device=device)
    b16 = dict(dtype=torch.bfloat16, device=device)
    rows = (1, hv, t, 128)
    r = GdnMixer(torch.empty((t, h), **f32), torch.empty((t, h), **b16),
                 torch.empty((1, conv.shape[0], 3 + t), **b16), torch.empty((1, conv.shape[0], 3), **b16),
                 torch.empty(((t + 15) // 16, 1, hv, 128, 128), **f32), torch.empty(rows, **f32),
                 torch.empty(rows, **f32), torch.empty((1, hv, t), **f32), torch.empty(rows, **f32))
    desc = _lib.GdnDesc(_desc(in_proj), _desc(out_proj), input_norm.data_ptr(), post_norm.data_ptr(), norm.data_ptr(),
                        a_log.data_ptr(), dt_bias.data_ptr(), conv.data_ptr(), h, key_heads, hv, eps)
    ws = _workspace(_lib.load().dflash_gdn_workspace_bytes(t, h, key_heads, hv), device, None)
    _lib.call("dflash_gdn_mixer", ctypes.byref(desc), _ptr(hidden), t, _ptr(history), _ptr(state), _ptr(r.mid),
              _ptr(r.normed), _ptr(r.window), _ptr(r.tail), _ptr(r.states), _ptr(r.keys), _ptr(r.u), _ptr(r.cum), _ptr(r.core),
              _ptr(ws), ws.numel(), _stream(device))
    return r


def rms_norm(hidden: torch.Tensor, weight: torch.Tensor, eps: float) -> Optional[torch.Tensor]:
    """``layers.rms_normalise(hidden, weight, eps, 1.0)`` of a plain fp32 residual ``[T, H]`` in one launch; None for other
    forms (and where autograd follows it)."""
    return host.rms_norm(hidden, weight, eps) if _plain(hidden) and (host := _lib.host()) else None


def gdn_mixer_plain(hidden, history, state, *, in_proj, out_proj, input_norm, post_norm, norm, a_log, dt_bias, conv,
                    key_heads, eps) -> Optional[GdnMixer]:
    """:func:`gdn_mixer` of arguments :func:`gdn_mixer_fits` accepts, both in one native call; None for others."""
    if not (_plain(hidden) and (host := _lib.host())):
        return None
    r = host.gdn(hidden, history, state, in_proj, out_proj, input_norm, post_norm, norm, a_log, dt_bias, conv, key_heads,
                 eps)
    return None if r is None else GdnMixer(*r)


def attention_mixer_plain(hidden, keys, values, position, *, in_proj, out_proj, input_norm, post_norm, q_norm, k_norm,
                          inv_freq, heads, kv_heads, head_dim, eps) -> Optional[tuple]:
    """:func:`attention_mixer` of arguments :func:`attention_mixer_fits` accepts, both in one native call; None for
    others."""
    if not (_plain(hidden) and (host := _lib.host())):
        return None
    return host.attention(hidden, keys, values, position, in_proj, out_proj, input_norm, post_norm, q_norm, k_norm,
                          inv_freq, heads, kv_heads, head_dim, eps)


def _as(t, dtype: torch.dtype, shape: tuple, device: torch.device) -> bool:
    """Whether ``t`` is what a kernel reads as is: this dtype, shape and device, contiguous, 16-byte aligned."""
    return (isinstance(t, torch.Tensor) and t.dtype == dtype and t.shape == shape and t.device == device
            and t.is_contiguous() and t.data_ptr() % 16 == 0)


def _tracked(*tensors) -> bool:
    """Whether autograd follows any of them (a gradient is asked for, or it carries a forward-mode tangent): the kernels
    drop both, so such calls take the PyTorch form."""
    return ((torch.is_grad_enabled() and any(t.requires_grad for t in tensors))
            or any(forward_ad.unpack_dual(t).tangent is not None for t in tensors))


def _matrix(w, rows: int, cols: int, device: torch.device) -> bool:
    """Whether ``w`` is a valid packed matrix of this size on this device."""
    if not isinstance(w, PackedW4) or w.packed.ndim != 2 or (w.rows, w.cols) != (rows, cols):
        return False
    w.validate("weight")
    return w.packed.device == device


def _residual(hidden: torch.Tensor) -> bool:
    """Whether the mixer kernels take this residual: fp32 ``[T, H]`` as it lies, at least one token, H they can
    normalise."""
    return (_as(hidden, torch.float32, hidden.shape, hidden.device) and hidden.is_cuda and hidden.ndim == 2
            and 1 <= hidden.shape[0] <= 1 << 19 and hidden.shape[1] % 512 == 0 and 512 <= hidden.shape[1] <= 8192)


def gdn_mixer_fits(hidden: torch.Tensor, history: torch.Tensor, state: torch.Tensor, *, in_proj: PackedW4,
                   out_proj: PackedW4, input_norm: torch.Tensor, post_norm: torch.Tensor, norm: torch.Tensor,
                   a_log: torch.Tensor, dt_bias: torch.Tensor, conv: torch.Tensor, key_heads: int, eps: float) -> bool:
    """Whether :func:`gdn_mixer` takes these arguments: head dims 128, four taps, plain contiguous tensors of the
    dtypes the target keeps, at least one token, and nothing that autograd follows."""
    if not _residual(hidden):
        return False
    device = hidden.device
    h, hv, f32, b16 = hidden.shape[1], a_log.shape[0], torch.float32, torch.bfloat16
    width = 128 * (2 * key_heads + hv)
    return (hv <= 1024 and hv % key_heads == 0
            and _as(history, b16, (1, width, 3), device) and _as(state, f32, (1, hv, 128, 128), device)
            and _as(conv, b16, (width, 1, 4), device) and _as(norm, f32, (128,), device)
            and _as(input_norm, f32, (h,), device) and _as(post_norm, f32, (h,), device)
            and _as(a_log, f32, (hv,), device) and _as(dt_bias, f32, (hv,), device)
            and not _tracked(hidden, history, state, conv, norm, input_norm, post_norm, a_log, dt_bias)
            and _matrix(in_proj, width + 128 * hv + 2 * hv, h, device) and _matrix(out_proj, h, 128 * hv, device))


def gdn_commit(state: torch.Tensor, keys: torch.Tensor, u: torch.Tensor, cum: torch.Tensor, accepted: int,
               window: torch.Tensor, first: int) -> Optional[tuple]:
    """``(recurrent state, conv history)`` after the first ``accepted`` tokens of one chunk of :func:`gdn_mixer`
    (``layers.state_after`` and the window's columns ``[first, first + 3)``) in one launch; ``None`` when the tensors
    are not laid out as that call leaves them, or autograd follows them."""
    if _plain(state) and (host := _lib.host()):
        done = host.commit(state, keys, u, cum, accepted, window, first)
        if done is not None:
            return done
    hv, device = state.shape[1], state.device
    if (device.type != "cuda" or not 1 <= accepted <= 16 or hv > 1024 or not 0 <= first <= 1 << 24
            or not _as(state, torch.float32, (1, hv, 128, 128), device)
            or keys.shape[:2] != (1, hv) or keys.shape[2] < accepted or keys.shape[3] != 128 or u.shape != keys.shape
            or cum.shape != keys.shape[:3]
            or any(t.dtype != torch.float32 or t.device != device for t in (keys, u, cum))
            or keys.stride()[2:] != (128, 1) or u.stride() != keys.stride() or cum.stride(2) != 1
            or window.dtype != torch.bfloat16 or window.ndim != 3 or window.shape[0] != 1 or window.device != device
            or not window.is_contiguous() or first + 3 > window.shape[2] or _tracked(state, keys, u, cum, window)):
        return None
    out = torch.empty_like(state)
    history = torch.empty((1, window.shape[1], 3), dtype=window.dtype, device=device)
    _lib.call("dflash_gdn_commit", _ptr(state), _ptr(keys), _ptr(u), _ptr(cum), keys.stride(1), cum.stride(1), hv,
              accepted, _ptr(out), _ptr(window), window.shape[2], first, window.shape[1], _ptr(history),
              _stream(device))
    return out, history


def attention_mixer_fits(hidden: torch.Tensor, keys: torch.Tensor, values: torch.Tensor, position: int, *,
                         in_proj: PackedW4, out_proj: PackedW4, input_norm: torch.Tensor, post_norm: torch.Tensor,
                         q_norm: torch.Tensor, k_norm: torch.Tensor, inv_freq: torch.Tensor, heads: int,
                         kv_heads: int, head_dim: int, eps: float) -> bool:
    """Whether :func:`attention_mixer` takes these arguments: head dim 128 or 256, plain contiguous tensors of the
    dtypes the target keeps, room in the cache, and nothing that autograd follows."""
    if not _residual(hidden) or head_dim not in (128, 256) or keys.ndim != 4 or keys.shape[2] > 1 << 24:
        return False
    device, (t, h) = hidden.device, hidden.shape
    f32, b16, cache, half = torch.float32, torch.bfloat16, (1, kv_heads, keys.shape[2], head_dim), inv_freq.shape[0]
    return (t * heads <= 1 << 22 and heads <= 1024 and heads % kv_heads == 0 and position + t <= keys.shape[2]
            and half > 0 and half % (head_dim // 64) == 0 and 2 * half <= head_dim
            and _as(keys, b16, cache, device) and _as(values, b16, cache, device)
            and _as(inv_freq, f32, (half,), device)
            and _as(input_norm, f32, (h,), device) and _as(post_norm, f32, (h,), device)
            and _as(q_norm, f32, (head_dim,), device) and _as(k_norm, f32, (head_dim,), device)
            and not _tracked(hidden, keys, values, inv_freq, input_norm, post_norm, q_norm, k_norm)
            and _matrix(in_proj, 2 * (heads + kv_heads) * head_dim, h, device)
            and _matrix(out_proj, h, heads * head_dim, device))


def attention_mixer(hidden: torch.Tensor, keys: torch.Tensor, values: torch.Tensor, position: int, *,
                    in_proj: PackedW4, out_proj: PackedW4, input_norm: torch.Tensor, post_norm: torch.Tensor,
                    q_norm: torch.Tensor, k_norm: torch.Tensor, inv_freq: torch.Tensor, heads: int, kv_heads: int,
                    head_dim: int, eps: float) -> tuple[torch.Tensor, torch.Tensor]:
    """An attention layer from its residual to the MoE input, in one call: norm, in_proj, Q/K norms, rotary, cache
    append, attention, output gate, out_proj, residual add, post-norm.  Returns ``(mid, normed)`` (fp32, bf16
    ``[T, H]``).  Tensors as :func:`attention_mixer_fits` accepts them."""
    device, (t, h) = hidden.device, hidden.shape
    mid = torch.empty((t, h), dtype=torch.float32, device=device)
    normed = torch.empty((t, h), dtype=torch.bfloat16, device=device)
    desc = _lib.AttentionDesc(_desc(in_proj), _desc(out_proj), input_norm.data_ptr(), post_norm.data_ptr(),
                              q_norm.data_ptr(), k_norm.data_ptr(), inv_freq.data_ptr(), h, heads, kv_heads, head_dim,
                              2 * inv_freq.shape[0], eps)
    ws = _workspace(_lib.load().dflash_attention_workspace_bytes(t, h, heads, kv_heads, head_dim), device, None)
    _lib.call("dflash_attention_mixer", ctypes.byref(desc), _ptr(hidden), t, position, _ptr(keys), _ptr(values),
              keys.shape[2], _ptr(mid), _ptr(normed), _ptr(ws), ws.numel(), _stream(device))
    return mid, normed


def router_logits(hidden: torch.Tensor, router_weight: torch.Tensor) -> torch.Tensor:
    """fp32 ``[T, E]`` logits from bf16 ``hidden [..., H]`` and bf16 ``router_weight [E, H]``."""
    device = _require_device(hidden, router_weight)
    if hidden.dtype != torch.bfloat16 or router_weight.dtype != torch.bfloat16:
        raise ValueError("router needs bfloat16 hidden and router_weight")
    if router_weight.ndim != 2 or router_weight.shape[1] != hidden.shape[-1]:
        raise ValueError("router_weight must be [E, H]")
    flat = hidden.reshape(-1, hidden.shape[-1]).contiguous()
    w = router_weight.contiguous()
    logits = torch.empty((flat.shape[0], w.shape[0]), dtype=torch.float32, device=device)
    _lib.call("dflash_router_logits", _ptr(flat), flat.shape[0], flat.shape[1], _ptr(w), w.shape[0], _ptr(logits),
              _stream(device))
    return logits


def _routing_buffers(t: int, e: int, k: int, device) -> Routing:
    return Routing(
        ids=torch.empty((t, k), dtype=torch.int32, device=device),
        weights=torch.empty((t, k), dtype=torch.float32, device=device),
        perm=torch.empty((t * k,), dtype=torch.int32, device=device),
        inv=torch.empty((t * k,), dtype=torch.int32, device=device),
        offsets=torch.empty((e + 1,), dtype=torch.int32, device=device))


def route(logits: torch.Tensor, top_k: int, *, workspace: Optional[torch.Tensor] = None) -> Routing:
    """Top-k routing and stable expert permutation from fp32 logits ``[T, E]``."""
    device = _require_device(logits)
    if logits.dtype != torch.float32 or logits.ndim != 2:
        raise ValueError("router logits must be float32 [T, E]")
    if type(top_k) is not int:
        raise ValueError("top_k must be an int")
    logits = logits.contiguous()
    t, e = logits.shape
    r = _routing_buffers(t, e, top_k, device)
    lib = _lib.load()
    ws = _workspace(lib.dflash_moe_route_workspace_bytes(t, e, top_k), device, workspace)
    _lib.call("dflash_moe_route", _ptr(logits), t, e, top_k, _ptr(r.ids), _ptr(r.weights), _ptr(r.perm),
              _ptr(r.inv), _ptr(r.offsets), _ptr(ws), ws.numel(), _stream(device))
    return r


def _shared_args(shared: Optional[SharedExpert]):
    if shared is None:
        return None, None, None, None
    if not isinstance(shared, SharedExpert):
        raise ValueError("shared must be a SharedExpert")
    shared.gate_up.validate("shared.gate_up")
    shared.down.validate("shared.down")
    gw = shared.gate_weight
    if gw.dtype != torch.bfloat16:
        raise ValueError("shared.gate_weight must be bfloat16 [H]")
    gw = gw.reshape(-1).contiguous()
    return _desc(shared.gate_up), _desc(shared.down), gw, (shared.gate_up.packed, shared.down.packed)


def _moe_common(hidden, gate_up: PackedW4, down: PackedW4, shared):
    gate_up.validate("gate_up")
    down.validate("down")
    if gate_up.packed.ndim != 3 or down.packed.ndim != 3:
        raise ValueError("expert banks must be [E, N, K/2]")
    device = _require_device(hidden, gate_up.packed, down.packed)
    if hidden.dtype != torch.bfloat16:
        raise ValueError("hidden must be bfloat16")
    h = hidden.shape[-1]
    flat = hidden.reshape(-1, h).contiguous()
    sgu, sdn, sgate, keep = _shared_args(shared)
    if keep is not None:
        _require_device(hidden, *keep, sgate)
    return device, flat, sgu, sdn, sgate


def _check_routing(routing: Routing, t: int, e: int, device: torch.device) -> int:
    """Validate a caller-given routing against the layer (the kernels index with it); returns top_k."""
    if not isinstance(routing, Routing):
        raise ValueError("routing must be a Routing (ids, weights, perm, inv, offsets)")
    ids = routing.ids
    if not isinstance(ids, torch.Tensor) or ids.ndim != 2 or ids.shape[0] != t:
        raise ValueError(f"routing.ids must be int32 [{t}, k]")
    k = ids.shape[1]
    if not 0 < k <= e:
        raise ValueError(f"routing top_k must be in (0, {e}]")
    expected = {"ids": (torch.int32, (t, k)), "weights": (torch.float32, (t, k)), "perm": (torch.int32, (t * k,)),
                "inv": (torch.int32, (t * k,)), "offsets": (torch.int32, (e + 1,))}
    for name, (dtype, shape) in expected.items():
        v = getattr(routing, name)
        if (not isinstance(v, torch.Tensor) or v.dtype != dtype or tuple(v.shape) != shape
                or v.device != device or not v.is_contiguous()):
            raise ValueError(f"routing.{name} must be a contiguous {dtype} {list(shape)} tensor on {device}")
    return k


def moe_experts(hidden: torch.Tensor, routing: Routing, gate_up: PackedW4, down: PackedW4, *,
                shared: Optional[SharedExpert] = None, workspace: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Expert FFN + combine for a given routing (as ``route`` returns it); bf16 ``[T, H]``.

    The routing's arrays are checked for device, dtype, shape and contiguity;
    their values are trusted (a routing not made by ``route`` must satisfy its
    invariants: a permutation, offsets ascending from 0 to T*k).
    """
    device, flat, sgu, sdn, sgate = _moe_common(hidden, gate_up, down, shared)
    t, h = flat.shape
    k = _check_routing(routing, t, gate_up.experts, device)
    out = torch.empty_like(flat)
    lib = _lib.load()
    ws = _workspace(lib.dflash_moe_workspace_bytes(t, h, gate_up.rows // 2, gate_up.experts, k, gate_up.group_size,
                                                   int(shared is not None)), device, workspace)
    gu, dn = _desc(gate_up), _desc(down)
    _lib.call("dflash_moe_experts_w4a16", _ptr(flat), t, h, k, _ptr(routing.weights),
              _ptr(routing.perm), _ptr(routing.inv), _ptr(routing.offsets), ctypes.byref(gu), ctypes.byref(dn),
              None if sgu is None else ctypes.byref(sgu), None if sdn is None else ctypes.byref(sdn), _ptr(sgate),
              _ptr(out), _ptr(ws), ws.numel(), _stream(device))
    return out


def moe_w4a16(hidden: torch.Tensor, gate_up: PackedW4, down: PackedW4, *, top_k: int,
              router_weight: Optional[torch.Tensor] = None, router_logits: Optional[torch.Tensor] = None,
              shared: Optional[SharedExpert] = None, workspace: Optional[torch.Tensor] = None,
              return_routing: bool = False):
    """Whole routed-MoE layer (+ optional shared expert) on packed banks; bf16 ``[T, H]``.

    With ``return_routing=True`` also returns ``(Routing, logits)``; ``logits``
    are the fp32 router logits the routing was computed from.
    """
    if router_logits is None and not return_routing and _plain(hidden) and (host := _lib.host()):
        out = host.moe(hidden, gate_up, down, top_k, router_weight, shared, workspace, None)
        if out is not None:
            return out
    device, flat, sgu, sdn, sgate = _moe_common(hidden, gate_up, down, shared)
    if type(top_k) is not int:
        raise ValueError("top_k must be an int")
    t, h = flat.shape
    e = gate_up.experts
    if router_logits is not None:
        _require_device(router_logits)
        if router_logits.dtype != torch.float32 or tuple(router_logits.shape) != (t, e):
            raise ValueError(f"router_logits must be float32 [{t}, {e}]")
        logits_in = router_logits.contiguous()
        logits_out = logits_in
    else:
        if router_weight is None:
            raise ValueError("router_weight or router_logits is required")
        _require_device(router_weight)
        if router_weight.dtype != torch.bfloat16 or tuple(router_weight.shape) != (e, h):
            raise ValueError(f"router_weight must be bfloat16 [{e}, {h}]")
        logits_in = None
        logits_out = torch.empty((t, e), dtype=torch.float32, device=device)
    rw = None if router_weight is None else router_weight.contiguous()
    r = _routing_buffers(t, e, top_k, device)
    out = torch.empty_like(flat)
    lib = _lib.load()
    ws = _workspace(lib.dflash_moe_workspace_bytes(t, h, gate_up.rows // 2, e, top_k, gate_up.group_size,
                                                   int(shared is not None)), device, workspace)
    gu, dn = _desc(gate_up), _desc(down)
    _lib.call("dflash_moe_w4a16", _ptr(flat), t, h, _ptr(logits_in), _ptr(rw), top_k, ctypes.byref(gu),
              ctypes.byref(dn), None if sgu is None else ctypes.byref(sgu), None if sdn is None else ctypes.byref(sdn),
              _ptr(sgate), _ptr(out), _ptr(logits_out if logits_in is None else None), _ptr(r.ids), _ptr(r.weights),
              _ptr(r.perm), _ptr(r.inv), _ptr(r.offsets), _ptr(ws), ws.numel(), _stream(device))
    if return_routing:
        return out, r, logits_out
    return out


def moe_w4a16_add(residual: torch.Tensor, hidden: torch.Tensor, gate_up: PackedW4, down: PackedW4, *, top_k: int,
                  router_weight: torch.Tensor, shared: Optional[SharedExpert] = None,
                  workspace: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``residual + moe_w4a16(hidden, ...)`` in fp32 ``[T, H]`` without a launch for the add; ``residual`` is contiguous
    fp32 of hidden's shape."""
    if _plain(hidden) and (host := _lib.host()):
        out = host.moe(hidden, gate_up, down, top_k, router_weight, shared, workspace, residual)
        if out is not None:
            return out
    device, flat, sgu, sdn, sgate = _moe_common(hidden, gate_up, down, shared)
    if type(top_k) is not int:
        raise ValueError("top_k must be an int")
    t, h = flat.shape
    e = gate_up.experts
    if not _as(residual, torch.float32, (t, h), device):
        raise ValueError(f"residual must be a contiguous float32 [{t}, {h}] tensor on {device}")
    _require_device(router_weight)
    if router_weight.dtype != torch.bfloat16 or tuple(router_weight.shape) != (e, h):
        raise ValueError(f"router_weight must be bfloat16 [{e}, {h}]")
    if _tracked(residual):
        return residual + moe_w4a16(hidden, gate_up, down, top_k=top_k, router_weight=router_weight, shared=shared,
                                    workspace=workspace).float()
    rw = router_weight.contiguous()
    logits = torch.empty((t, e), dtype=torch.float32, device=device)
    r = _routing_buffers(t, e, top_k, device)
    out = torch.empty_like(residual)
    ws = _workspace(_lib.load().dflash_moe_workspace_bytes(t, h, gate_up.rows // 2, e, top_k, gate_up.group_size,
                                                           int(shared is not None)), device, workspace)
    gu, dn = _desc(gate_up), _desc(down)
    _lib.call("dflash_moe_w4a16_residual", _ptr(flat), t, h, _ptr(rw), top_k, ctypes.byref(gu), ctypes.byref(dn),
              None if sgu is None else ctypes.byref(sgu), None if sdn is None else ctypes.byref(sdn), _ptr(sgate),
              _ptr(residual), _ptr(out), _ptr(logits), _ptr(r.ids), _ptr(r.weights), _ptr(r.perm), _ptr(r.inv),
              _ptr(r.offsets), _ptr(ws), ws.numel(), _stream(device))
    return out


NOALLOC_SCRATCH_BYTES = 8 << 20


def moe_w4a16_noalloc(hidden: torch.Tensor, gate_up: PackedW4, down: PackedW4, *, top_k: int,
                      router_weight: Optional[torch.Tensor] = None, router_logits: Optional[torch.Tensor] = None,
                      shared: Optional[SharedExpert] = None, out: Optional[torch.Tensor] = None,
                      routing: Optional[Routing] = None, logits_out: Optional[torch.Tensor] = None):
    """``moe_w4a16`` through ``dflash_moe_w4a16_noalloc``: no workspace, the library's static scratch.

    The library allocates nothing; this wrapper allocates the outputs only when the caller
    does not pass them (``out`` bf16 ``[T, H]``, ``routing`` buffers, ``logits_out`` fp32
    ``[T, E]``).  Returns ``(out, routing, logits)``.  Layers needing more than
    ``NOALLOC_SCRATCH_BYTES`` of scratch raise :class:`DflashError`.
    """
    device, flat, sgu, sdn, sgate = _moe_common(hidden, gate_up, down, shared)
    if type(top_k) is not int:
        raise ValueError("top_k must be an int")
    t, h = flat.shape
    e = gate_up.experts
    if router_logits is not None:
        _require_device(router_logits)
        if router_logits.dtype != torch.float32 or tuple(router_logits.shape) != (t, e):
            raise ValueError(f"router_logits must be float32 [{t}, {e}]")
        router_logits = router_logits.contiguous()
        logits_out = router_logits
    else:
        if router_weight is None:
            raise ValueError("router_weight or router_logits is required")
        _require_device(router_weight)
        if router_weight.dtype != torch.bfloat16 or tuple(router_weight.shape) != (e, h):
            raise ValueError(f"router_weight must be bfloat16 [{e}, {h}]")
        router_weight = router_weight.contiguous()
        if logits_out is None:
            logits_out = torch.empty((t, e), dtype=torch.float32, device=device)
        elif (logits_out.dtype != torch.float32 or tuple(logits_out.shape) != (t, e) or logits_out.device != device
              or not logits_out.is_contiguous()):
            raise ValueError(f"logits_out must be a contiguous float32 [{t}, {e}] tensor on {device}")
    if routing is None:
        routing = _routing_buffers(t, e, top_k, device)
    elif _check_routing(routing, t, e, device) != top_k:
        raise ValueError("routing buffers must hold top_k slots per token")
    if out is None:
        out = torch.empty_like(flat)
    elif out.dtype != torch.bfloat16 or tuple(out.shape) != (t, h) or out.device != device or not out.is_contiguous():
        raise ValueError(f"out must be a contiguous bfloat16 [{t}, {h}] tensor on {device}")
    gu, dn = _desc(gate_up), _desc(down)
    r = routing
    _lib.call("dflash_moe_w4a16_noalloc", _ptr(flat), t, h, _ptr(router_logits), _ptr(router_weight), top_k,
              ctypes.byref(gu), ctypes.byref(dn), None if sgu is None else ctypes.byref(sgu),
              None if sdn is None else ctypes.byref(sdn), _ptr(sgate), _ptr(out),
              None if router_logits is not None else _ptr(logits_out), _ptr(r.ids), _ptr(r.weights), _ptr(r.perm),
              _ptr(r.inv), _ptr(r.offsets), _stream(device))
    return out, routing, logits_out


def qlinear_workspace_bytes(m: int, k: int, group_size: int = 128) -> int:
    return int(_lib.load().dflash_qlinear_workspace_bytes(m, k, group_size))


def moe_workspace_bytes(tokens: int, hidden: int, inter: int, experts: int, top_k: int, group_size: int,
                        has_shared: bool) -> int:
    return int(_lib.load().dflash_moe_workspace_bytes(tokens, hidden, inter, experts, top_k, group_size,
                                                      int(has_shared)))


_split_down = False  # the library's process-wide switch, as last set through set_split_down


def set_split_down(enable: bool) -> None:
    """Process-wide: run a verify block's down GEMM inside its gate/up launch where it fits
    (opt-in; off, the default, runs the separate down launch)."""
    global _split_down
    _lib.call("dflash_set_split_down", int(bool(enable)))
    _split_down = bool(enable)


@contextlib.contextmanager
def split_down(enable: bool):
    """Sets the split-K down switch for a block of calls and restores the previous setting."""
    prev = _split_down
    set_split_down(enable)
    try:
        yield
    finally:
        set_split_down(prev)


@contextlib.contextmanager
def tile_pieces(pieces: int):
    """Forces the prefill tile kernels' tail split (1, 2 or 4 pieces) for a block of calls,
    then restores the grid-chosen default."""
    _lib.call("dflash_set_tile_pieces", int(pieces))
    try:
        yield
    finally:
        _lib.call("dflash_set_tile_pieces", 0)


def moe_split_down(tokens: int, hidden: int, inter: int, experts: int, top_k: int, group_size: int,
                   has_shared: bool, scale_dtype: torch.dtype = torch.bfloat16, layout: str = "tiled") -> bool:
    """Whether a ``moe_w4a16`` call of this shape runs the split-K down on the current device."""
    return bool(_lib.load().dflash_moe_split_down(
        tokens, hidden, inter, experts, top_k, group_size, int(has_shared),
        _lib.DTYPE_F32 if scale_dtype == torch.float32 else _lib.DTYPE_BF16,
        _lib.LAYOUT_TILED if layout == "tiled" else _lib.LAYOUT_PORTABLE))


STAGE_GATE_UP = _lib.STAGE_GATE_UP
STAGE_DOWN = _lib.STAGE_DOWN
STAGE_EXPERTS = _lib.STAGE_EXPERTS


def set_measure_stage(stage: int) -> None:
    """Measurement mode: later MoE calls launch only ``stage``'s kernel (0 restores full calls).

    The kernel reuses what an earlier full call with the same arguments left
    in the same workspace; the layer output is not written.
    """
    _lib.call("dflash_set_measure_stage", int(stage))
