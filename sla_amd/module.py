"""``SparseLinearAttention`` with the constructor, parameters and forward of the reference
module (``sparse_linear_attention/core.py:24-105``), running on the HIP kernels."""
from __future__ import annotations

import functools

import torch
import torch.autograd.forward_ad as forward_ad
import torch.nn as nn

from . import _lib
from .block_map import get_block_map, topk_count
from .linear import linear_complement_bwd, linear_complement_fwd, linear_state_fwd
from .sparse_attn import sparse_attn_bwd, sparse_attn_fwd

FEATURE_MAPS = ("elu", "relu", "softmax")


def module_bwd(q, k, v, o_s, d_out, lse, sparse_map, lut, topk, BLKQ, BLKK, qk_scale, weight, bias, fmap, states=None,
               grads=None, side_stream=None):
    """Backward of the whole operator in one library call (``sla_module_bwd``): the kernels of
    :func:`sparse_attn_bwd` and of :func:`linear_bwd` accumulating into the same gradients, bit for bit, the short kernels
    in the launches of longer ones (``side_stream`` is accepted and not used).  Returns ``(dq, dk, dv, d_weight, d_bias)``.
    For callers that hold the forward's parts in tensors of their own; the operators below keep them in one allocation and
    take :func:`_module_bwd_saved`.

    q, k, v (and ``grads=(dq, dk, dv)`` when given) may be row-contiguous views sharing their strides, ``d_out`` a
    row-contiguous view of its own; ``o_s`` and ``lse`` are contiguous.  ``states`` as in :func:`linear_bwd`."""
    _lib.require_gpu(q, k, v, o_s, d_out, lse, sparse_map, lut, weight, bias)
    B, H, L, D = q.shape
    dev = q.device
    dt = _lib.dtype_code(q.dtype)
    dq, dk, dv = (torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)) if grads is None else grads
    assert o_s.is_contiguous() and lse.is_contiguous() and sparse_map.is_contiguous() and lut.is_contiguous()
    ws_s = _lib.workspace(_lib.WS_SPARSE_BWD, dt, B, H, L, D, BLKQ, BLKK, topk, dev)
    ws_l = _lib.workspace(_lib.WS_LINEAR_BWD, dt, B, H, L, D, 64, 64, 0, dev)
    flags = 0
    if states is not None:
        ws_l[:states.numel()].copy_(states)
        flags |= _lib.BWD_STATES_READY
    dw = torch.empty((D, D), dtype=torch.float32, device=dev)
    db = torch.empty((D,), dtype=torch.float32, device=dev)
    if all(t.is_contiguous() for t in (q, k, v, d_out, dq, dk, dv)):
        s_qkv = s_do = None
    else:
        assert _lib.row_strided(q, k, v, dq, dk, dv) and _lib.row_strided(d_out), "tensors must be row-contiguous views"
        s_qkv, s_do = _lib.strides_arg(q), _lib.strides_arg(d_out)
    side = 0 if side_stream is None else side_stream.cuda_stream
    rc = _lib.load().sla_module_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), s_qkv, o_s.data_ptr(), d_out.data_ptr(), s_do,
                                    lse.data_ptr(), sparse_map.data_ptr(), lut.data_ptr(), lut.element_size(),
                                    weight.data_ptr(), bias.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                                    dw.data_ptr(), db.data_ptr(), dt, _lib.FMAP[fmap], B, H, L, D, BLKQ, BLKK, topk,
                                    float(qk_scale), flags, ws_s.data_ptr(), ws_s.numel(), ws_l.data_ptr(), ws_l.numel(),
                                    _lib.stream_ptr(dev), side)
    _lib.check(rc)
    return dq, dk, dv, dw, db


@functools.lru_cache(maxsize=1024)
def _plan(in_dt, dt, B, H, L, D, BLKQ, BLKK, T, keep):
    """Sizes of one forward: ``(workspace bytes, bytes to keep, offsets)``.  What a backward needs of the forward lies in one
    allocation (states, look-up table, log-sum-exp, and with ``keep`` map, attention output, the 16-bit copies of
    fp32 inputs); without a backward the same parts are scratch behind the workspace."""
    M, N = -(-L // BLKQ), -(-L // BLKK)
    elems = B * H * L * D
    parts = {"states": _lib.workspace_bytes(_lib.WS_LINEAR_STATES, dt, B, H, L, D, 64, 64, 0),
             "lut": B * H * M * T * 4, "lse": B * H * L * 4}
    if keep:
        parts["map"] = B * H * M * N
        parts["o_s"] = elems * 2
    if in_dt == _lib.SLA_F32:
        parts["cast"] = 3 * elems * 2
    ws = -(-_lib.workspace_bytes(_lib.WS_MODULE_FWD, in_dt if in_dt >= 0 else dt, B, H, L, D, BLKQ, BLKK, T) // 256) * 256
    off, at = {}, 0 if keep else ws
    for name, n in parts.items():
        off[name] = at
        at += -(-n // 256) * 256
    return ws, at, off


def _module_fwd(q, k, v, weight, bias, topk_ratio, BLKQ, BLKK, fmap, dtype, keep, mask=None):
    """The whole forward as one library call (``sla_module_fwd``).  q, k, v: ``dtype`` (contiguous, or row-contiguous views
    sharing their strides) or contiguous fp32; ``mask``: a ``(sparse_map, lut)`` built elsewhere.  Returns
    ``(out, kept allocation or None, real topk)``; out is in ``dtype``, or of fp32 inputs the same values in fp32."""
    B, H, L, D = q.shape
    dev = q.device
    dt, in_dt = _lib.dtype_code(dtype), _lib.dtype_code(q.dtype)
    T = topk_count(-(-L // BLKK), topk_ratio)
    if mask is not None:
        in_dt = _lib.SLA_MASK_GIVEN
    ws_bytes, total, off = _plan(in_dt, dt, B, H, L, D, BLKQ, BLKK, T, keep)
    ws = torch.empty(ws_bytes if keep else total, dtype=torch.uint8, device=dev)
    saved = torch.empty(total, dtype=torch.uint8, device=dev) if keep else None
    base = (saved if keep else ws).data_ptr()
    if mask is not None:
        sparse_map, lut = mask
        (saved if keep else ws)[off["lut"]:off["lut"] + lut.numel() * 4].view(torch.int32).copy_(lut.view(-1))
        if keep:
            saved[off["map"]:off["map"] + sparse_map.numel()].view(torch.int8).copy_(sparse_map.view(-1))
    if q.is_contiguous() and k.is_contiguous() and v.is_contiguous():
        s_in = s_out = None
        out = torch.empty((B, H, L, D), dtype=torch.float32 if in_dt == _lib.SLA_F32 else dtype, device=dev)
    else:
        assert _lib.row_strided(q, k, v), "q, k, v must be contiguous or share row-contiguous strides"
        out = _lib.empty_like_rows(q)
        s_in, s_out = _lib.strides_arg(q), _lib.strides_arg(out)
    rc = _lib.load().sla_module_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), s_in, _lib.SLA_F32_BOTH if in_dt == _lib.SLA_F32 else in_dt,
        base + off["cast"] if in_dt == _lib.SLA_F32 else None,
        weight.data_ptr(), bias.data_ptr(), out.data_ptr(), s_out, base + off["o_s"] if keep else None, base + off["lse"],
        base + off["map"] if keep else None, base + off["lut"], 4, base + off["states"], dt, _lib.FMAP[fmap], B, H, L, D, BLKQ,
        BLKK, T, D ** -0.5, ws.data_ptr(), ws_bytes, _lib.stream_ptr(dev), None)
    _lib.check(rc)
    return out, saved, T


def _module_bwd_saved(saved, off, q_ptr, k_ptr, v_ptr, s_qkv, d_out, s_do, weight, bias, grads, shape, dtype, T, BLKQ, BLKK, fmap):
    """Backward from what :func:`_module_fwd` kept; writes ``grads`` (three pointers, laid out like q, k, v) and returns
    ``(d_weight, d_bias)``."""
    B, H, L, D = shape
    dev = saved.device
    dt = _lib.dtype_code(dtype)
    n_s = _lib.workspace_bytes(_lib.WS_SPARSE_BWD, dt, B, H, L, D, BLKQ, BLKK, T)
    n_l = _lib.workspace_bytes(_lib.WS_LINEAR_BWD_STATES_APART, dt, B, H, L, D, 64, 64, 0)
    n_s = -(-n_s // 256) * 256
    ws = torch.empty(n_s + n_l, dtype=torch.uint8, device=dev)
    dw = torch.empty((D, D), dtype=torch.float32, device=dev)
    db = torch.empty((D,), dtype=torch.float32, device=dev)
    base, w0 = saved.data_ptr(), ws.data_ptr()
    rc = _lib.load().sla_module_bwd_states(
        q_ptr, k_ptr, v_ptr, s_qkv, base + off["o_s"], d_out.data_ptr(), s_do, base + off["lse"], base + off["map"],
        base + off["lut"], 4, weight.data_ptr(), bias.data_ptr(), base + off["states"], *grads, dw.data_ptr(),
        db.data_ptr(), dt, _lib.FMAP[fmap], B, H, L, D, BLKQ, BLKK, T, D ** -0.5, w0, n_s, w0 + n_s, n_l,
        _lib.stream_ptr(dev), None)
    _lib.check(rc)
    return dw, db


def _through_autograd(*tensors):
    """Whether a call goes through its autograd function: where a gradient may be asked for, inside a forward-mode level
    (the function has no jvp and refuses dual tensors; the library call alone would drop their tangents), and under a trace
    (which records the function; of the library call alone it would record the allocations)."""
    return (torch.is_grad_enabled() and any(t.requires_grad for t in tensors) or forward_ad._current_level >= 0
            or torch.jit.is_tracing())


class _sla_core(torch.autograd.Function):
    """Sparse branch + linear branch + projection + sum as one differentiable operator.

    Same function as ``_attention`` followed by ``_linear_proj_add`` (reference core.py:88-100); fusing
    them lets the backward add the linear-branch gradients into the sparse-branch ones in place.
    """

    @staticmethod
    def forward(ctx, q, k, v, weight, bias, topk_ratio, BLKQ, BLKK, fmap, dtype, mask):
        assert q.is_contiguous() and k.is_contiguous() and v.is_contiguous()
        out, saved, T = _module_fwd(q, k, v, weight, bias, topk_ratio, BLKQ, BLKK, fmap, dtype, True, mask)
        if q.dtype == dtype:
            ctx.save_for_backward(weight, bias, saved, q, k, v)
        else:                                   # (the backward works on the 16-bit copies among what is kept)
            ctx.save_for_backward(weight, bias, saved)
            out = out.to(q.dtype)               # (fp32 inputs: out is fp32 already)
        in_dt = _lib.dtype_code(q.dtype) if mask is None else _lib.SLA_MASK_GIVEN
        ctx.cfg = (tuple(q.shape), in_dt, T, BLKQ, BLKK, fmap, dtype, q.dtype)
        return out

    @staticmethod
    def backward(ctx, d_out):
        weight, bias, saved, *qkv = ctx.saved_tensors
        shape, in_dt, T, BLKQ, BLKK, fmap, dtype, in_dtype = ctx.cfg
        off = _plan(in_dt, _lib.dtype_code(dtype), *shape, BLKQ, BLKK, T, True)[2]
        d_out = d_out.contiguous().to(dtype)
        # (an allocation per gradient: a caller may keep one of them, or detach it in place, without the others)
        grads = [torch.empty(shape, dtype=dtype, device=d_out.device) for _ in range(3)]
        if qkv:
            ptrs = [t.data_ptr() for t in qkv]
        else:
            step = grads[0].numel() * grads[0].element_size()
            ptrs = [saved.data_ptr() + off["cast"] + i * step for i in range(3)]
        dw, db = _module_bwd_saved(saved, off, *ptrs, None, d_out, None, weight, bias, [t.data_ptr() for t in grads], shape,
                                   dtype, T, BLKQ, BLKK, fmap)
        return (*(t.to(in_dtype) for t in grads), dw, db, None, None, None, None, None, None)


class _sla_complement(torch.autograd.Function):
    """Sparse branch + complement-mode linear branch (over the key blocks a query block did not select) + projection
    + sum.  The reference has no such variant; the definition is ``linear_complement_fwd``'s."""

    @staticmethod
    def forward(ctx, q, k, v, weight, bias, sparse_map, lut, topk, BLKQ, BLKK, fmap, keep):
        # (keep: a backward may follow.  ctx.needs_input_grad also says so of a parameter under no_grad)
        assert q.is_contiguous() and k.is_contiguous() and v.is_contiguous()
        assert sparse_map.is_contiguous() and lut.is_contiguous()
        assert BLKQ in (64, 128) and BLKK == 64
        qk_scale = q.shape[-1] ** -0.5
        weight, bias = weight.contiguous(), bias.contiguous()
        o_s, lse = sparse_attn_fwd(q, k, v, lut, topk, BLKQ, BLKK, qk_scale)
        out = linear_complement_fwd(q, k, v, lut, topk, weight, bias, o_s, fmap, BLKQ, BLKK, keep_states=keep)
        if keep:
            out, states = out
            ctx.save_for_backward(q, k, v, weight, bias, sparse_map, lut, lse, o_s, states)
            ctx.cfg = (topk, BLKQ, BLKK, fmap, qk_scale)
        return out

    @staticmethod
    def backward(ctx, d_out):
        q, k, v, weight, bias, sparse_map, lut, lse, o_s, states = ctx.saved_tensors
        topk, BLKQ, BLKK, fmap, qk_scale = ctx.cfg
        d_out = d_out.contiguous()
        dq, dk, dv = sparse_attn_bwd(q, k, v, o_s, d_out, lse, sparse_map, lut, topk, BLKQ, BLKK, qk_scale)
        _, _, _, dw, db = linear_complement_bwd(q, k, v, sparse_map, lut, topk, weight, bias, d_out, fmap, BLKQ, BLKK,
                                                accumulate_into=(dq, dk, dv), states=states)
        return dq, dk, dv, dw, db, None, None, None, None, None, None, None


class _sla_packed(torch.autograd.Function):
    """The same operator on a packed ``(B, L, 3, H, D)`` projection output, returning ``(B, L, H, D)``.

    A transformer block produces q, k, v as one packed tensor in token-major order and consumes the attention
    output in token-major order.  Fed to ``_sla_core`` through views, autograd would rebuild the packed gradient
    with three zero-fill-and-copy passes; here the kernels read q, k, v where they lie (row stride ``3*H*D``) and
    the backward kernels write dq, dk, dv straight into one packed gradient tensor, so neither direction copies.
    """

    @staticmethod
    def forward(ctx, qkv, weight, bias, topk_ratio, BLKQ, BLKK, fmap):
        assert qkv.dim() == 5 and qkv.shape[2] == 3 and qkv.is_contiguous()
        q, k, v = (qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3))          # (B, H, L, D) views
        out, saved, T = _module_fwd(q, k, v, weight, bias, topk_ratio, BLKQ, BLKK, fmap, qkv.dtype, True)
        ctx.save_for_backward(qkv, weight, bias, saved)
        ctx.cfg = (tuple(q.shape), T, BLKQ, BLKK, fmap)
        return out.permute(0, 2, 1, 3)                                            # (B, L, H, D), contiguous

    @staticmethod
    def backward(ctx, d_out):
        qkv, weight, bias, saved = ctx.saved_tensors
        shape, T, BLKQ, BLKK, fmap = ctx.cfg
        q = qkv[:, :, 0].permute(0, 2, 1, 3)
        d_out = d_out.permute(0, 2, 1, 3)                                         # (B, H, L, D) view
        if not _lib.row_strided(d_out):
            d_out = d_out.contiguous()
        d_qkv = torch.empty_like(qkv)
        dt = _lib.dtype_code(qkv.dtype)
        off = _plan(dt, dt, *shape, BLKQ, BLKK, T, True)[2]
        step = shape[1] * shape[3] * qkv.element_size()                           # from a token's q to its k, to its v
        p, g = qkv.data_ptr(), d_qkv.data_ptr()
        dw, db = _module_bwd_saved(saved, off, p, p + step, p + 2 * step, _lib.strides_arg(q), d_out, _lib.strides_arg(d_out),
                                   weight, bias, (g, g + step, g + 2 * step), shape, qkv.dtype, T, BLKQ, BLKK, fmap)
        return d_qkv, dw, db, None, None, None, None


class _StateBuild:
    """The k/v-only half of the linear branch, started on a side stream so that it runs beside the mask
    builder (both are short memory-bound kernels; neither fills the device on its own).  ``join`` makes
    the calling stream wait for it and hands over the workspace it filled."""

    _side = {}

    def __init__(self, k, v, weight, fmap):
        dev = k.device

        def build():
            self.ws = linear_state_fwd(k, v, weight, fmap)

        cur = torch.cuda.current_stream(dev)
        if torch.cuda.is_current_stream_capturing():
            side = None          # inside a graph capture the work stays on the capturing stream
        else:
            side = self._side.get(dev.index)
            if side is None:
                side = self._side[dev.index] = torch.cuda.Stream(device=dev)
        self.side = side
        if side is None:
            build()
            return
        side.wait_stream(cur)    # k, v and the weight were produced on the calling stream
        with torch.cuda.stream(side):
            build()

    def join(self):
        if self.side is not None:
            torch.cuda.current_stream(self.ws.device).wait_stream(self.side)
            # the workspace was allocated under the side stream; it is consumed on the calling one
            self.ws.record_stream(torch.cuda.current_stream(self.ws.device))
        return self.ws


class SparseLinearAttention(nn.Module):
    def __init__(self, head_dim, topk, feature_map="softmax", BLKQ=64, BLKK=64, use_bf16=True,
                 tie_feature_map_qk=True, linear_mode="global"):
        r"""
        Args:
            head_dim: dimension of each head.
            topk: ratio of keys selected for sparse attention, shared across all queries.
            feature_map: feature map for linear attention, one of ['elu', 'relu', 'softmax'].
            BLKQ: block size for query.
            BLKK: block size for key.
            use_bf16: bfloat16 (default) or float16 compute; inputs are converted inside the module.
            tie_feature_map_qk: kept for signature compatibility; q and k always use the same map
                (as in the reference, core.py:43-60).
            linear_mode: "global" (default, what the reference computes: the linear branch sees every key)
                or "complement" (extension: it sees only the key blocks the query block did not select).
        """
        super().__init__()
        self.dtype = torch.bfloat16 if use_bf16 else torch.float16
        self.topk = topk
        self.BLKQ = BLKQ
        self.BLKK = BLKK
        self.proj_l = nn.Linear(head_dim, head_dim, dtype=torch.float32)
        if feature_map not in FEATURE_MAPS:
            raise NotImplementedError(f"Not supported feature map {feature_map}.")
        self.feature_map = feature_map
        self.tie_feature_map_qk = tie_feature_map_qk
        if linear_mode not in ("global", "complement"):
            raise NotImplementedError(f"Not supported linear mode {linear_mode}.")
        self.linear_mode = linear_mode
        self.init_weights_()

    def init_weights_(self):
        with torch.no_grad():
            nn.init.zeros_(self.proj_l.weight)
            nn.init.zeros_(self.proj_l.bias)

    def forward(self, q, k, v, return_sparsity=False):
        r"""
        Args:
            q, k, v: (B, H, L, D).
            return_sparsity: also return real_topk / n_key_blocks (reference core.py:102-103).
        """
        proj = self.proj_l
        weight, bias = proj.weight, proj.bias
        _lib.check_operands(q, k, v, weight, bias)      # no CPU path: refuse loudly before anything touches a stream
        _lib.check_shapes(q, k, v)
        _lib.check_projection(weight, bias, q.shape[3])
        dtype = q.dtype
        needs_grad = _through_autograd(q, k, v, weight, bias)
        # Inference on activations that are not laid out as (B, H, L, D) -- a (B, L, H, D) tensor or the slices
        # of a packed QKV projection, viewed as (B, H, L, D) -- reads them where they are and writes the output
        # in the same dimension order, instead of copying three tensors in and one out (the reference makes
        # the copies: core.py:77-79).  Training and the other cases take the contiguous route.
        contiguous = q.is_contiguous() and k.is_contiguous() and v.is_contiguous()
        in_place = (not contiguous and not needs_grad and self.linear_mode == "global" and dtype == self.dtype
                    and _lib.row_strided(q, k, v))
        if not in_place and not contiguous:
            q = q.contiguous()
            k = k.contiguous()
            v = v.contiguous()

        if self.linear_mode == "complement":
            return self._forward_complement(q, k, q.to(self.dtype), k.to(self.dtype), v.to(self.dtype), dtype, return_sparsity,
                                            needs_grad)
        if not (weight.is_contiguous() and bias.is_contiguous()):
            weight, bias = weight.contiguous(), bias.contiguous()
        mask = None
        if not (q.dtype == k.dtype == v.dtype and (dtype == self.dtype or (dtype == torch.float32 and v.data_ptr() % 16 == 0))):
            # the mask is built from the inputs in their own dtype (reference core.py:83), the rest works on copies (which the
            # library makes itself of fp32 tensors that lie on 16 bytes)
            with torch.no_grad():
                mask = get_block_map(q, k, topk_ratio=self.topk, BLKQ=self.BLKQ, BLKK=self.BLKK)[:2]
            q, k, v = q.to(self.dtype), k.to(self.dtype), v.to(self.dtype)
        args = (q, k, v, weight, bias, self.topk, self.BLKQ, self.BLKK, self.feature_map, self.dtype)
        o = _sla_core.apply(*args, mask) if needs_grad else _module_fwd(*args, False, mask)[0]
        if o.dtype != dtype:
            o = o.to(dtype)
        if return_sparsity:
            N = -(-q.shape[2] // self.BLKK)
            return o, topk_count(N, self.topk) / N
        return o

    def forward_packed(self, qkv, return_sparsity=False):
        r"""
        The forward on a packed projection output, without layout copies in either direction (extension; the
        reference takes separate ``(B, H, L, D)`` tensors).

        Args:
            qkv: (B, L, 3, H, D), as ``nn.Linear(dim, 3 * dim)(x).view(B, L, 3, H, D)`` gives it.
        Returns:
            (B, L, H, D), ready for ``reshape(B, L, H * D)``.
        """
        if qkv.dtype != self.dtype or self.linear_mode != "global" or not _lib.row_strided(qkv[:, :, 0].permute(0, 2, 1, 3)):
            q, k, v = (qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3))
            res = self.forward(q, k, v, return_sparsity)
            o = res[0] if return_sparsity else res
            o = o.permute(0, 2, 1, 3)
            return (o, res[1]) if return_sparsity else o
        assert qkv.dim() == 5 and qkv.shape[2] == 3, f"the packed projection is (B, L, 3, H, D), got {tuple(qkv.shape)}"
        weight, bias = self.proj_l.weight, self.proj_l.bias
        _lib.check_operands(qkv, weight, bias)
        _lib.check_projection(weight, bias, qkv.shape[-1])
        args = (qkv.contiguous(), weight.contiguous(), bias.contiguous(), self.topk, self.BLKQ, self.BLKK, self.feature_map)
        if _through_autograd(*args[:3]):
            o = _sla_packed.apply(*args)
        else:
            q, k, v = (args[0][:, :, i].permute(0, 2, 1, 3) for i in range(3))
            o = _module_fwd(q, k, v, *args[1:], self.dtype, False)[0].permute(0, 2, 1, 3)
        if return_sparsity:
            N = (qkv.shape[1] + self.BLKK - 1) // self.BLKK
            return o, min(N, int(self.topk * N)) / N
        return o

    def _forward_complement(self, q, k, qc, kc, vc, dtype, return_sparsity, needs_grad):
        sparse_map, lut, real_topk = get_block_map(q, k, topk_ratio=self.topk, BLKQ=self.BLKQ, BLKK=self.BLKK)
        o = _sla_complement.apply(qc, kc, vc, self.proj_l.weight, self.proj_l.bias, sparse_map, lut, real_topk, self.BLKQ,
                                  self.BLKK, self.feature_map, needs_grad).to(dtype)
        if return_sparsity:
            return o, real_topk / sparse_map.shape[-1]
        return o
