"""Device-tensor wrappers over the C ABI, plus the autograd binding.

Tensors are torch tensors on a ROCm device; torch only supplies device
memory and the current HIP stream.  All arithmetic runs in ``libmfattn.so``.
The autograd ``Function`` plays the role of the reference's ``jax.custom_vjp``
boundary: the forward saves ``(q, k, v, out, lse, plan)`` and the backward
calls the HIP backward once.
"""

from __future__ import annotations

import collections
import threading
import weakref

import torch

from . import _lib

_DTYPES = {torch.float32: _lib.DTYPE_F32, torch.bfloat16: _lib.DTYPE_BF16}


# The current stream's handle by device index.  torch.cuda.current_stream
# builds a Stream object for the same number (1.9 us against 0.1); it serves a
# torch without the private query (a build for the CPU has none).
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None) or (
    lambda index: torch.cuda.current_stream(index).cuda_stream)


def _stream(device: torch.device) -> int:
    return _raw_stream(device.index)


def _ptr(t: torch.Tensor | None) -> int | None:
    return None if t is None else t.data_ptr()


def require_device(*tensors: torch.Tensor) -> torch.device:
    """Every operand must already live on one ROCm device (no host fallback)."""
    device = tensors[0].device
    index = device.index
    for t in tensors:
        if not t.is_cuda:
            raise ValueError(
                "mfattn runs on the GPU only; got a tensor on " + str(t.device)
            )
        if t.get_device() != index:
            raise ValueError("all operands must be on the same device")
    return device


def dtype_code(t: torch.Tensor) -> int:
    try:
        return _DTYPES[t.dtype]
    except KeyError:
        raise ValueError(f"Unsupported dtype {t.dtype}; mfattn serves float32 and bfloat16") from None


def same_dtype(what: str, *tensors: torch.Tensor) -> int:
    """The one dtype code every tensor shares; a mix raises before any launch.

    The kernels index every operand with the element size of that one dtype,
    so a float32 query over a bfloat16 cache would read past the cache.
    """
    first = tensors[0].dtype
    for t in tensors[1:]:
        if t.dtype != first:
            raise ValueError(f"{what} must share one dtype (got {first} and {t.dtype})")
    return dtype_code(tensors[0])


def _require_shape(t: torch.Tensor, shape: tuple[int, ...], what: str) -> None:
    if t.shape != shape:  # torch.Size compares as a tuple
        raise ValueError(f"{what} must be {list(shape)}, got {list(t.shape)}")


def require_contiguous(what: str, *tensors: torch.Tensor) -> None:
    """The kernels address every operand as a dense row-major array from its
    ``data_ptr()``: a slice or transposed view would be read (or written) as
    if it were dense, so it is refused before any launch.  Callers that hold
    views pass ``.contiguous()`` copies (the drop-in functions do)."""
    for t in tensors:
        if t is not None and not t.is_contiguous():
            raise ValueError(f"{what} must be contiguous (got a strided view of shape "
                             f"{list(t.shape)}); pass .contiguous()")


def _require_lse(lse: torch.Tensor, b: int, hq: int, t: int) -> None:
    if lse.dtype != torch.float32:
        raise ValueError("lse must be float32")
    _require_shape(lse, (b, hq, t), "lse")
    require_contiguous("lse", lse)


def _require_workspace(ws: torch.Tensor, b: int, t: int, hq: int) -> None:
    need = _lib.LIB.mf_attn_bwd_workspace_bytes(b, t, hq)
    if ws.dtype != torch.uint8 or ws.numel() < need:
        raise ValueError(f"the backward workspace must be a uint8 tensor of at least {need} bytes")
    require_contiguous("the backward workspace", ws)


def as_mask(mask: torch.Tensor, mode: int) -> tuple[torch.Tensor, int]:
    """Mask in a dtype the C ABI reads (int32 or uint8), values preserved.

    Other dtypes are reduced to their activity first: ``> 0`` for the packed
    causal mode (``attention.py:97``), ``!= 0`` for the bidirectional modes
    (``bidirectional.py:22,25``).
    """
    dtype = mask.dtype
    if dtype is torch.int32:
        return mask.contiguous(), _lib.MASK_I32
    if dtype is torch.bool or dtype is torch.uint8:
        return mask.contiguous().view(torch.uint8), _lib.MASK_U8
    active = mask > 0 if mode == _lib.MODE_PACKED_CAUSAL else mask != 0
    return active.to(torch.uint8).contiguous(), _lib.MASK_U8


class Plan:
    """Device block map (canonical ids, tile map, work lists) of one call."""

    def __init__(self, buf: torch.Tensor, batch: int, q_len: int, kv_len: int, mode: int):
        self.buf, self.batch, self.q_len, self.kv_len, self.mode = buf, batch, q_len, kv_len, mode

    @property
    def nbytes(self) -> int:
        return self.buf.numel()  # uint8

    def section(self, index: int, dtype: torch.dtype, shape: tuple[int, ...]) -> torch.Tensor:
        offs = _lib.plan_layout(self.batch, self.q_len, self.kv_len)
        count = 1
        for s in shape:
            count *= s
        width = torch.empty((), dtype=dtype).element_size()
        raw = self.buf[offs[index] : offs[index] + count * width]
        return raw.view(dtype).view(shape)

    def tile_map(self) -> torch.Tensor:
        nq, nk = -(-self.q_len // _lib.TILE), -(-self.kv_len // _lib.TILE)
        return self.section(2, torch.uint8, (self.batch, nq, nk))


_BLOCK_MAP_CALLS = [0]  # block-map launches made through this module (plan reuse is tested on it)


def block_map(segment_ids: torch.Tensor | None, mask: torch.Tensor, mode: int,
              q_len: int, kv_len: int, batch: int | None = None) -> Plan:
    """Build the plan of ``(segment_ids, mask, mode)``.

    ``mask`` must be ``[B, S]`` and ``segment_ids`` ``[B, T]`` exactly: the
    kernel reads B * S mask entries and B * T ids, and the attention kernels
    index the plan with the query's batch, so ``batch`` (default
    ``mask.shape[0]``) is checked against both.
    """
    batch = mask.shape[0] if batch is None else batch
    _require_shape(mask, (batch, kv_len), "mask")
    if segment_ids is not None:
        _require_shape(segment_ids, (batch, q_len), "segment_ids")
    device = require_device(mask) if segment_ids is None else require_device(mask, segment_ids)
    m, mcode = as_mask(mask, mode)
    seg = segment_ids
    if seg is not None:
        if seg.dtype is not torch.int32:
            seg = seg.to(torch.int32)
        seg = seg.contiguous()
    nbytes = _lib.LIB.mf_plan_bytes(batch, q_len, kv_len)
    if nbytes == 0:
        raise ValueError("Sizes must be positive")
    buf = torch.empty(nbytes, dtype=torch.uint8, device=device)
    _lib.check(_lib.LIB.mf_block_map(_ptr(seg), m.data_ptr(), mcode, mode, batch, q_len, kv_len,
                                     buf.data_ptr(), nbytes, _raw_stream(device.index)))
    _BLOCK_MAP_CALLS[0] += 1
    return Plan(buf, batch, q_len, kv_len, mode)


def block_map_from_placements(placements: torch.Tensor, mode: int, batch: int,
                              length: int) -> tuple[Plan, torch.Tensor, torch.Tensor]:
    """Plan, segment ids and positions from packer placements ``[N, 3]`` (row, start, len)."""
    device = require_device(placements)
    pl = placements.to(torch.int32).contiguous()
    if pl.dim() != 2 or pl.shape[1] != 3:
        raise ValueError("placements must be [count, 3] (row, start, length)")
    nbytes = _lib.LIB.mf_plan_bytes(batch, length, length)
    if nbytes == 0:
        raise ValueError("Sizes must be positive")
    buf = torch.empty(nbytes, dtype=torch.uint8, device=device)
    seg = torch.empty((batch, length), dtype=torch.int32, device=device)
    pos = torch.empty_like(seg)
    _lib.check(_lib.LIB.mf_block_map_placements(_ptr(pl), pl.shape[0], mode, batch, length,
                                                _ptr(buf), nbytes, _ptr(seg), _ptr(pos),
                                                _stream(device)))
    return Plan(buf, batch, length, length, mode), seg, pos


def check_attention_operands(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                             plan: Plan | None = None, mode: int | None = None) -> int:
    """Shapes, dtypes and plan of one attention call; returns the dtype code.

    ``q [B, T, Hq, D]``, ``k`` and ``v`` ``[B, S, Hkv, D]`` with one dtype; a
    plan must have been built for the same batch, lengths and mode.
    """
    code = same_dtype("query, key and value", q, k, v)
    qs, ks = q.shape, k.shape
    if len(qs) != 4 or len(ks) != 4 or ks != v.shape or qs[0] != ks[0] or qs[3] != ks[3]:
        raise ValueError("Packed attention query/KV shapes are incompatible")
    require_contiguous("query, key and value", q, k, v)
    if plan is not None:
        if plan.batch != qs[0] or plan.q_len != qs[1] or plan.kv_len != ks[1]:
            raise ValueError(
                f"plan was built for batch {plan.batch}, lengths {plan.q_len}/{plan.kv_len}; "
                f"the call has {qs[0]}, {qs[1]}/{ks[1]}")
        if mode is not None and plan.mode != mode:
            raise ValueError(f"plan was built for mask mode {plan.mode}, the call uses {mode}")
    return code


def attn_fwd(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, plan: Plan, mode: int,
             scale: float) -> tuple[torch.Tensor, torch.Tensor]:
    code = check_attention_operands(q, k, v, plan, mode)
    device = require_device(q, k, v)
    b, t, hq, d = q.shape
    _, s, hkv, _ = k.shape
    out = torch.empty_like(q)
    lse = torch.empty((b, hq, t), dtype=torch.float32, device=device)
    _lib.check(_lib.LIB.mf_attn_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), code, b, t, s, hq,
                                    hkv, d, mode, float(scale), plan.buf.data_ptr(), plan.nbytes,
                                    out.data_ptr(), lse.data_ptr(), _raw_stream(device.index)))
    return out, lse


def attn_fwd_rope_q(q_raw: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                    q_gain: torch.Tensor, positions: torch.Tensor | None, plan: Plan, mode: int,
                    scale: float, *, eps: float, rope_theta: float
                    ) -> tuple[torch.Tensor, torch.Tensor]:
    """``attn_fwd`` of the query after RMS norm and RoPE, both applied in the kernel's query
    loads (``mf_attn_fwd_rope_q``): equal bit for bit to ``attn_fwd(qk_norm_rope(q_raw)[0],
    k, v, ...)`` with ``k`` already normalised and rotated.  bf16; no autograd.

    ``q_gain`` ``[D]`` in the tensor dtype, ``positions`` ``[B, T]`` int32 or ``None``.
    """
    code = check_attention_operands(q_raw, k, v, plan, mode)
    device = require_device(q_raw, k, v, q_gain)
    if q_raw.dtype != torch.bfloat16:
        raise ValueError("the fused query prologue serves bfloat16 tensors")
    b, t, hq, d = q_raw.shape
    s, hkv = k.shape[1], k.shape[2]
    if q_gain.shape != (d,) or q_gain.dtype != q_raw.dtype:
        raise ValueError("q_gain must be a [D] tensor of the query's dtype")
    if positions is not None and (positions.shape != (b, t) or positions.dtype != torch.int32):
        raise ValueError("positions must be a [B, T] int32 tensor")
    require_contiguous("positions", positions)
    q_gain = q_gain.contiguous()
    table_bytes = _lib.LIB.mf_rope_table_bytes(b, t)
    table = torch.empty(table_bytes // 4, dtype=torch.int32, device=device)
    out = torch.empty_like(q_raw)
    lse = torch.empty((b, hq, t), dtype=torch.float32, device=device)
    _lib.check(_lib.LIB.mf_attn_fwd_rope_q(
        _ptr(q_raw), _ptr(k), _ptr(v), _ptr(q_gain), _ptr(positions), code, b, t,
        s, hq, hkv, d, mode, float(scale), float(eps), float(rope_theta), _ptr(plan.buf),
        plan.nbytes, _ptr(table), table_bytes, _ptr(out), _ptr(lse), _stream(device)))
    return out, lse


def attn_bwd(q, k, v, out, dout, lse, plan: Plan, mode: int, scale: float):
    check_attention_operands(q, k, v, plan, mode)
    code = same_dtype("query, key, value, output and its gradient", q, k, v, out, dout)
    qs = q.shape
    if out.shape != qs or dout.shape != qs:
        raise ValueError("the output and its gradient must have the query's shape")
    require_contiguous("the output and its gradient", out, dout)
    b, t, hq, d = qs
    _, s, hkv, _ = k.shape
    _require_lse(lse, b, hq, t)
    device = require_device(q, k, v, out, dout, lse)
    dq = torch.empty_like(q)
    dk = torch.empty_like(k)
    dv = torch.empty_like(v)
    ws_bytes = _lib.LIB.mf_attn_bwd_workspace_bytes(b, t, hq)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=device)
    _lib.check(_lib.LIB.mf_attn_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                                    dout.data_ptr(), lse.data_ptr(), code, b, t, s, hq, hkv, d,
                                    mode, float(scale), plan.buf.data_ptr(), plan.nbytes,
                                    dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), ws.data_ptr(),
                                    ws_bytes, _raw_stream(device.index)))
    return dq, dk, dv


def bwd_workspace(q: torch.Tensor) -> torch.Tensor:
    b, t, hq, _ = q.shape
    return torch.empty(_lib.LIB.mf_attn_bwd_workspace_bytes(b, t, hq), dtype=torch.uint8,
                       device=q.device)


def attn_bwd_delta(out, dout, lse, ws) -> None:
    """Phase 1 of the backward: -rowsum(dO * O) and lse * log2(e) into ``ws``."""
    same_dtype("output and its gradient", out, dout)
    if dout.shape != out.shape or out.dim() != 4:
        raise ValueError("the output and its gradient must be [B, T, Hq, D] of one shape")
    require_contiguous("the output and its gradient", out, dout)
    b, t, hq, d = out.shape
    _require_lse(lse, b, hq, t)
    _require_workspace(ws, b, t, hq)
    _lib.check(_lib.LIB.mf_attn_bwd_delta(_ptr(out), _ptr(dout), _ptr(lse), dtype_code(out), b, t,
                                          hq, d, _ptr(ws), ws.numel(), _stream(out.device)))


def attn_bwd_dq(q, k, v, dout, lse, plan: Plan, mode: int, scale: float, ws, dq) -> None:
    """Phase 2 of the backward: dq (reads the delta phase's ``ws``)."""
    check_attention_operands(q, k, v, plan, mode)
    same_dtype("query, output gradient and dq", q, dout, dq)
    if dout.shape != q.shape or dq.shape != q.shape:
        raise ValueError("the output gradient and dq must have the query's shape")
    require_contiguous("the output gradient and dq", dout, dq)
    b, t, hq, d = q.shape
    s, hkv = k.shape[1], k.shape[2]
    _require_lse(lse, b, hq, t)
    _require_workspace(ws, b, t, hq)
    _lib.check(_lib.LIB.mf_attn_bwd_dq(_ptr(q), _ptr(k), _ptr(v), _ptr(dout), _ptr(lse),
                                       dtype_code(q), b, t, s, hq, hkv, d, mode, float(scale),
                                       _ptr(plan.buf), plan.nbytes, _ptr(dq), _ptr(ws), ws.numel(),
                                       _stream(q.device)))


def attn_bwd_dkdv(q, k, v, dout, lse, plan: Plan, mode: int, scale: float, ws, dk, dv) -> None:
    """Phase 3 of the backward: dk and dv (reads the delta phase's ``ws``)."""
    check_attention_operands(q, k, v, plan, mode)
    same_dtype("query, output gradient, dk and dv", q, dout, dk, dv)
    if dout.shape != q.shape or dk.shape != k.shape or dv.shape != k.shape:
        raise ValueError("the output gradient must have the query's shape, dk and dv the key's")
    require_contiguous("the output gradient, dk and dv", dout, dk, dv)
    b, t, hq, d = q.shape
    s, hkv = k.shape[1], k.shape[2]
    _require_lse(lse, b, hq, t)
    _require_workspace(ws, b, t, hq)
    _lib.check(_lib.LIB.mf_attn_bwd_dkdv(_ptr(q), _ptr(k), _ptr(v), _ptr(dout), _ptr(lse),
                                         dtype_code(q), b, t, s, hq, hkv, d, mode, float(scale),
                                         _ptr(plan.buf), plan.nbytes, _ptr(dk), _ptr(dv), _ptr(ws),
                                         ws.numel(), _stream(q.device)))


def _check_decode_shapes(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor) -> None:
    qs, ks = q.shape, k_cache.shape
    if (len(qs) != 4 or qs[1] != 1 or len(ks) != 4 or ks != v_cache.shape or ks[0] != qs[0]
            or ks[3] != qs[3]):
        raise ValueError("Cached attention query/KV shapes are incompatible")


def _check_lengths(lengths: torch.Tensor, batch: int, what: str) -> None:
    if lengths.dtype is not torch.int32 or lengths.shape != (batch,) \
            or not lengths.is_contiguous():
        raise ValueError(f"{what} must be a contiguous int32 [{batch}] tensor")


def decode_append(q: torch.Tensor, k_new: torch.Tensor, v_new: torch.Tensor,
                  k_cache: torch.Tensor, v_cache: torch.Tensor, positions: torch.Tensor,
                  scale: float) -> torch.Tensor:
    """Write each row's new key/value into its cache slot (in place), then decode."""
    code = same_dtype("query, new key/value and the KV caches", q, k_new, v_new, k_cache, v_cache)
    _check_decode_shapes(q, k_cache, v_cache)
    b, _, hq, d = q.shape
    _, cap, hkv, _ = k_cache.shape
    for t in (k_new, v_new):
        _require_shape(t, (b, 1, hkv, d), "the new key/value rows")
    _check_lengths(positions, b, "positions")
    for t in (k_cache, v_cache):
        if not t.is_contiguous():
            raise ValueError("the KV caches must be contiguous to be updated in place")
    device = require_device(q, k_new, v_new, k_cache, v_cache, positions)
    q, k_new, v_new = q.contiguous(), k_new.contiguous(), v_new.contiguous()
    out = torch.empty_like(q)
    ws_bytes = _lib.LIB.mf_decode_workspace_bytes(b, cap, hq, d)
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=device)
    _lib.check(_lib.LIB.mf_decode_append(_ptr(q), _ptr(k_new), _ptr(v_new), _ptr(positions), code,
                                         b, cap, hq, hkv, d, float(scale), _ptr(k_cache),
                                         _ptr(v_cache), _ptr(out), _ptr(ws), ws_bytes,
                                         _stream(device)))
    return out


def decode(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
           lengths: torch.Tensor, scale: float) -> torch.Tensor:
    code = same_dtype("query and the KV caches", q, k_cache, v_cache)
    _check_decode_shapes(q, k_cache, v_cache)
    b, _, hq, d = q.shape
    _, cap, hkv, _ = k_cache.shape
    _check_lengths(lengths, b, "lengths")
    device = require_device(q, k_cache, v_cache, lengths)
    q, k_cache, v_cache = q.contiguous(), k_cache.contiguous(), v_cache.contiguous()
    out = torch.empty_like(q)
    ws_bytes = _lib.LIB.mf_decode_workspace_bytes(b, cap, hq, d)
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=device)
    _lib.check(_lib.LIB.mf_decode(_ptr(q), _ptr(k_cache), _ptr(v_cache), _ptr(lengths), code, b,
                                  cap, hq, hkv, d, float(scale), _ptr(out), _ptr(ws), ws_bytes,
                                  _stream(device)))
    return out


class PlanCache:
    """Plans keyed on the identity and in-place version of the id and mask tensors.

    A plan depends only on ``(segment_ids, mask, mode, lengths)``.  The
    encoder passes one ``(segment_ids, mask)`` pair to every attention layer
    (``models/lfm2_5/encoder.py:64-110``) and rematerialisation runs each
    forward twice, so the block map runs once per distinct pair.  An entry
    holds weak references to the tensors it was built from: it is used only
    while both are the very objects passed and their version counters (bumped
    by every in-place torch write) are unchanged, so a freed, replaced or
    modified tensor misses.  Writes that bypass torch (a raw pointer handed to
    other code) are not seen: such callers pass ``plan=`` explicitly or clear
    the cache.

    Two cases never touch the cache:

    * graph capture: a captured step must record its own block map, because
      a replay runs with whatever ids the static input buffers then hold
      (copied in with ``copy_`` between replays), and a plan built under
      capture holds nothing until the graph is replayed, so it is neither
      looked up nor stored while the current stream is capturing;
    * another stream: the key includes the current stream, so a plan is only
      reused on the stream that built it, where stream order already makes
      its contents visible to every later call.
    """

    def __init__(self, capacity: int = 8):
        self.capacity = capacity
        self.enabled = True
        self._entries: collections.OrderedDict = collections.OrderedDict()
        self._lock = threading.Lock()

    @staticmethod
    def _state(t: torch.Tensor | None):
        return (None, None) if t is None else (weakref.ref(t), t._version)

    def get(self, segment_ids: torch.Tensor | None, mask: torch.Tensor, mode: int, q_len: int,
            kv_len: int, batch: int) -> Plan:
        if not self.enabled or (mask.device.type == "cuda"
                                and torch.cuda.is_current_stream_capturing()):
            return block_map(segment_ids, mask, mode, q_len, kv_len, batch)
        stream = _stream(mask.device) if mask.device.type == "cuda" else None
        key = (id(segment_ids), id(mask), mode, q_len, kv_len, batch, mask.device, stream)
        with self._lock:
            entry = self._entries.get(key)
            if entry is not None:
                (seg_ref, seg_ver), (mask_ref, mask_ver), plan = entry
                seg_ok = segment_ids is None if seg_ref is None else (
                    seg_ref() is segment_ids and segment_ids._version == seg_ver)
                if seg_ok and mask_ref() is mask and mask._version == mask_ver:
                    self._entries.move_to_end(key)
                    return plan
        plan = block_map(segment_ids, mask, mode, q_len, kv_len, batch)
        with self._lock:
            self._entries[key] = (self._state(segment_ids), self._state(mask), plan)
            while len(self._entries) > self.capacity:
                self._entries.popitem(last=False)
        return plan

    def clear(self) -> None:
        with self._lock:
            self._entries.clear()


PLANS = PlanCache()


class PackedAttention(torch.autograd.Function):
    """Masked attention with a HIP forward and a HIP backward.

    ``forward(q, k, v, mask, segment_ids, mode, scale, plan)``: integer inputs
    get no gradient (the reference's float0 cotangents).  ``plan`` is a
    :class:`Plan` built for the same ids, mask and mode, or ``None`` to take
    one from :data:`PLANS`.
    """

    @staticmethod
    def forward(ctx, q, k, v, mask, segment_ids, mode, scale, plan=None):
        q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
        check_attention_operands(q, k, v)
        if plan is None:
            plan = PLANS.get(segment_ids, mask, mode, q.shape[1], k.shape[1], q.shape[0])
        out, lse = attn_fwd(q, k, v, plan, mode, scale)
        ctx.save_for_backward(q, k, v, out, lse)
        ctx.plan, ctx.mode, ctx.scale = plan, mode, scale
        return out

    @staticmethod
    def backward(ctx, dout):
        q, k, v, out, lse = ctx.saved_tensors
        dq, dk, dv = attn_bwd(q, k, v, out, dout.contiguous(), lse, ctx.plan, ctx.mode, ctx.scale)
        return dq, dk, dv, None, None, None, None, None


def packed_attention(q, k, v, mask, segment_ids, mode: int, scale: float,
                     plan: Plan | None = None) -> torch.Tensor:
    return PackedAttention.apply(q, k, v, mask, segment_ids, mode, scale, plan)
