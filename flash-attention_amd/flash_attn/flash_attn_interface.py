"""Public attention API, argument-for-argument the reference's
`flash_attn/flash_attn_interface.py` (functions at :551-1042 there), forward and backward
(autograd functions at :193-548 there).

The native module is `flash_attn._native` (ctypes over libfa_mi355x.so) in place of the
reference's `flash_attn_2_cuda`; its entry points keep the reference's positional
signatures, so the call sites below read like the reference's (:47, :79, :121, :165, :1024).

Dropout draws its mask from a counter-based hash seeded by torch's CUDA generator (not the reference's
Philox stream: masks differ from the reference's for the same seed, their statistics do not).
`return_attn_probs=True` returns `(out, softmax_lse, S_dmask)`; with dropout 0 S_dmask is None exactly
as in the reference, with dropout it holds the softmax probabilities in plain (row, key) order,
negated where dropped.

Gradients are deterministic: the same call gives the same bits.  Some backward calls borrow work space (at most 512 MiB,
freed in stream order); where it cannot be allocated another form runs, whose sums are in another order.

`grad_fn` of a result is a node of C++ for an ordinary call, and FlashAttnFuncBackward and its like for the others (see `_apply`): code
that reads a node's name, its `saved_tensors` or its attributes gets them from the latter only (hooks on saved tensors are such a call).
"""
from typing import Optional, Union

import torch

from flash_attn import _native as flash_attn_gpu


def _get_block_size(device, head_dim, is_dropout, is_causal):
    """(query rows per workgroup, keys per tile) of the general tiled forward kernel, the one that
    runs whenever dropout or return_attn_probs is in play.  The reference's helper of this name
    (flash_attn_interface.py:13-41) mirrors its CUDA tile table because its tests need it to decode
    S_dmask; here S_dmask is in plain (row, key) order and the value is informational.  Without
    dropout, sequences of 512 rows and more run on kernels with 128- or 256-row workgroups and 64-key
    tiles (32 above head dim 128)."""
    assert head_dim <= 256
    return (128, 64) if head_dim <= 128 else (128, 32)


def _maybe_contiguous(x):
    return x.contiguous() if x is not None and x.stride(-1) != 1 else x


def _flash_attn_forward(q, k, v, dropout_p, softmax_scale, causal, window_size, return_softmax):
    q, k, v = [_maybe_contiguous(x) for x in (q, k, v)]
    out, q, k, v, out_padded, softmax_lse, S_dmask, rng_state = flash_attn_gpu.fwd(
        q, k, v, None, dropout_p, softmax_scale, causal, window_size[0], window_size[1],
        return_softmax, None,
    )
    return out, q, k, v, out_padded, softmax_lse, S_dmask, rng_state


def _flash_attn_varlen_forward(q, k, v, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k,
                               dropout_p, softmax_scale, causal, window_size, return_softmax):
    q, k, v = [_maybe_contiguous(x) for x in (q, k, v)]
    out, q, k, v, out_padded, softmax_lse, S_dmask, rng_state = flash_attn_gpu.varlen_fwd(
        q, k, v, None, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, dropout_p,
        softmax_scale, False, causal, window_size[0], window_size[1], return_softmax, None,
    )
    return out, q, k, v, out_padded, softmax_lse, S_dmask, rng_state


def _flash_attn_backward(dout, q, k, v, out, softmax_lse, dq, dk, dv, dropout_p, softmax_scale, causal,
                         window_size, rng_state=None):
    # dq, dk, dv are allocated by the caller below and may be strided views of one packed tensor
    dout, q, k, v, out = [_maybe_contiguous(x) for x in (dout, q, k, v, out)]
    dq, dk, dv, softmax_d = flash_attn_gpu.bwd(
        dout, q, k, v, out, softmax_lse, dq, dk, dv, dropout_p, softmax_scale, causal,
        window_size[0], window_size[1], None, rng_state,
    )
    return dq, dk, dv, softmax_d


def _flash_attn_varlen_backward(dout, q, k, v, out, softmax_lse, dq, dk, dv, cu_seqlens_q, cu_seqlens_k,
                                max_seqlen_q, max_seqlen_k, dropout_p, softmax_scale, causal, window_size,
                                rng_state=None):
    dout, q, k, v, out = [_maybe_contiguous(x) for x in (dout, q, k, v, out)]
    dq, dk, dv, softmax_d = flash_attn_gpu.varlen_bwd(
        dout, q, k, v, out, softmax_lse, dq, dk, dv, cu_seqlens_q, cu_seqlens_k, max_seqlen_q,
        max_seqlen_k, dropout_p, softmax_scale, False, causal, window_size[0], window_size[1], None,
        rng_state,
    )
    return dq, dk, dv, softmax_d


flash_attn_gpu.host.watch(globals(), ("_flash_attn_forward", "_flash_attn_varlen_forward", "_flash_attn_backward", "_flash_attn_varlen_backward"))


def _save(ctx, tensors, dropout_p, softmax_scale, causal, window_size, **extra):
    ctx.save_for_backward(*tensors)
    ctx.dropout_p, ctx.softmax_scale, ctx.causal, ctx.window_size = dropout_p, softmax_scale, causal, window_size
    for name, value in extra.items():
        setattr(ctx, name, value)


class _NoGraph:
    """Stands in for the context of an autograd function where nothing will ask for it."""
    def save_for_backward(self, *tensors):
        pass


_fwd_ad = torch.autograd.forward_ad
_functorch_active = torch._C._are_functorch_transforms_active
_functorch_wrapped = torch._C._functorch.is_functorch_wrapped_tensor


def _apply(fn, tensors, *args):
    """fn.apply(*args), by the quickest route that the call can take.  The native host path (csrc/fa_host.cpp) takes the ordinary
    ones, node of autograd included: it left 6.9 us of host time of 14.6 for a prefill of 1 x 512 tokens, 32/8 heads, d 128, 44 of 86
    for a forward and backward pass of 2 x 512 tokens, 9.4 of 20.2 for a decoding step.  What it leaves (None) goes to the function's
    forward alone when autograd has no part in the call: `tensors` (its differentiable inputs) ask for no gradient and nothing
    that acts on autograd functions is active -- functorch transforms (or tensors they left behind), forward-mode levels, tracing,
    compilation; half the host time of a small call is the function's node that nobody reads."""
    native = getattr(fn, "native", None)
    if native is not None and _fwd_ad._current_level < 0 and not torch.compiler.is_compiling():
        out = native(*args)
        if out is not None:
            return out
    grad = torch.is_grad_enabled()
    for t in tensors:
        if (grad and t.requires_grad) or _functorch_wrapped(t):
            return fn.apply(*args)
    if _functorch_active() or _fwd_ad._current_level >= 0 or torch._C._get_tracing_state() is not None or torch.compiler.is_compiling():
        return fn.apply(*args)
    return fn.forward(_NoGraph(), *args)


class FlashAttnFunc(torch.autograd.Function):
    native = flash_attn_gpu.host.func

    @staticmethod
    def forward(ctx, q, k, v, dropout_p, softmax_scale, causal, window_size, return_softmax):
        if softmax_scale is None:
            softmax_scale = q.shape[-1] ** (-0.5)
        out, q, k, v, out_padded, softmax_lse, S_dmask, rng_state = _flash_attn_forward(
            q, k, v, dropout_p, softmax_scale, causal=causal, window_size=window_size,
            return_softmax=return_softmax and dropout_p > 0,
        )
        _save(ctx, (q, k, v, out_padded, softmax_lse, rng_state), dropout_p, softmax_scale, causal, window_size)
        return out if not return_softmax else (out, softmax_lse, S_dmask)

    @staticmethod
    def backward(ctx, dout, *args):
        q, k, v, out, softmax_lse, rng_state = ctx.saved_tensors
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        _flash_attn_backward(dout, q, k, v, out, softmax_lse, dq, dk, dv, ctx.dropout_p, ctx.softmax_scale,
                             ctx.causal, ctx.window_size, rng_state=rng_state)
        dq, dk, dv = dq[..., : dout.shape[-1]], dk[..., : dout.shape[-1]], dv[..., : dout.shape[-1]]
        return dq, dk, dv, None, None, None, None, None


class FlashAttnQKVPackedFunc(torch.autograd.Function):
    native = flash_attn_gpu.host.qkvpacked_func

    @staticmethod
    def forward(ctx, qkv, dropout_p, softmax_scale, causal, window_size, return_softmax):
        if softmax_scale is None:
            softmax_scale = qkv.shape[-1] ** (-0.5)
        out, q, k, v, out_padded, softmax_lse, S_dmask, rng_state = _flash_attn_forward(
            qkv[:, :, 0], qkv[:, :, 1], qkv[:, :, 2], dropout_p, softmax_scale, causal=causal,
            window_size=window_size, return_softmax=return_softmax and dropout_p > 0,
        )
        _save(ctx, (q, k, v, out_padded, softmax_lse, rng_state), dropout_p, softmax_scale, causal, window_size)
        return out if not return_softmax else (out, softmax_lse, S_dmask)

    @staticmethod
    def backward(ctx, dout, *args):
        q, k, v, out, softmax_lse, rng_state = ctx.saved_tensors
        qkv_shape = q.shape[:-2] + (3, *q.shape[-2:])
        dqkv = torch.empty(qkv_shape, dtype=q.dtype, device=q.device)
        _flash_attn_backward(dout, q, k, v, out, softmax_lse, dqkv[:, :, 0], dqkv[:, :, 1], dqkv[:, :, 2],
                             ctx.dropout_p, ctx.softmax_scale, ctx.causal, ctx.window_size, rng_state=rng_state)
        dqkv = dqkv[..., : dout.shape[-1]]
        return dqkv, None, None, None, None, None


class FlashAttnKVPackedFunc(torch.autograd.Function):
    native = flash_attn_gpu.host.kvpacked_func

    @staticmethod
    def forward(ctx, q, kv, dropout_p, softmax_scale, causal, window_size, return_softmax):
        if softmax_scale is None:
            softmax_scale = q.shape[-1] ** (-0.5)
        out, q, k, v, out_padded, softmax_lse, S_dmask, rng_state = _flash_attn_forward(
            q, kv[:, :, 0], kv[:, :, 1], dropout_p, softmax_scale, causal=causal,
            window_size=window_size, return_softmax=return_softmax and dropout_p > 0,
        )
        _save(ctx, (q, k, v, out_padded, softmax_lse, rng_state), dropout_p, softmax_scale, causal, window_size)
        return out if not return_softmax else (out, softmax_lse, S_dmask)

    @staticmethod
    def backward(ctx, dout, *args):
        q, k, v, out, softmax_lse, rng_state = ctx.saved_tensors
        dq = torch.empty_like(q)
        kv_shape = k.shape[:-2] + (2, *k.shape[-2:])
        dkv = torch.empty(kv_shape, dtype=k.dtype, device=k.device)
        _flash_attn_backward(dout, q, k, v, out, softmax_lse, dq, dkv[:, :, 0], dkv[:, :, 1], ctx.dropout_p,
                             ctx.softmax_scale, ctx.causal, ctx.window_size, rng_state=rng_state)
        dq, dkv = dq[..., : dout.shape[-1]], dkv[..., : dout.shape[-1]]
        return dq, dkv, None, None, None, None, None


class FlashAttnVarlenFunc(torch.autograd.Function):
    native = flash_attn_gpu.host.varlen_func

    @staticmethod
    def forward(ctx, q, k, v, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, dropout_p,
                softmax_scale, causal, window_size, return_softmax):
        if softmax_scale is None:
            softmax_scale = q.shape[-1] ** (-0.5)
        out, q, k, v, out_padded, softmax_lse, S_dmask, rng_state = _flash_attn_varlen_forward(
            q, k, v, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, dropout_p,
            softmax_scale, causal=causal, window_size=window_size,
            return_softmax=return_softmax and dropout_p > 0,
        )
        _save(ctx, (q, k, v, out_padded, softmax_lse, cu_seqlens_q, cu_seqlens_k, rng_state), dropout_p,
              softmax_scale, causal, window_size, max_seqlen_q=max_seqlen_q, max_seqlen_k=max_seqlen_k)
        return out if not return_softmax else (out, softmax_lse, S_dmask)

    @staticmethod
    def backward(ctx, dout, *args):
        q, k, v, out, softmax_lse, cu_seqlens_q, cu_seqlens_k, rng_state = ctx.saved_tensors
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        _flash_attn_varlen_backward(dout, q, k, v, out, softmax_lse, dq, dk, dv, cu_seqlens_q, cu_seqlens_k,
                                    ctx.max_seqlen_q, ctx.max_seqlen_k, ctx.dropout_p, ctx.softmax_scale,
                                    ctx.causal, ctx.window_size, rng_state=rng_state)
        dq, dk, dv = dq[..., : dout.shape[-1]], dk[..., : dout.shape[-1]], dv[..., : dout.shape[-1]]
        return dq, dk, dv, None, None, None, None, None, None, None, None, None


class FlashAttnVarlenQKVPackedFunc(torch.autograd.Function):
    native = flash_attn_gpu.host.varlen_qkvpacked_func

    @staticmethod
    def forward(ctx, qkv, cu_seqlens, max_seqlen, dropout_p, softmax_scale, causal, window_size,
                return_softmax):
        if softmax_scale is None:
            softmax_scale = qkv.shape[-1] ** (-0.5)
        out, q, k, v, out_padded, softmax_lse, S_dmask, rng_state = _flash_attn_varlen_forward(
            qkv[:, 0], qkv[:, 1], qkv[:, 2], cu_seqlens, cu_seqlens, max_seqlen, max_seqlen,
            dropout_p, softmax_scale, causal=causal, window_size=window_size,
            return_softmax=return_softmax and dropout_p > 0,
        )
        _save(ctx, (q, k, v, out_padded, softmax_lse, cu_seqlens, rng_state), dropout_p, softmax_scale, causal,
              window_size, max_seqlen=max_seqlen)
        return out if not return_softmax else (out, softmax_lse, S_dmask)

    @staticmethod
    def backward(ctx, dout, *args):
        q, k, v, out, softmax_lse, cu_seqlens, rng_state = ctx.saved_tensors
        qkv_shape = q.shape[:-2] + (3, *q.shape[-2:])
        dqkv = torch.empty(qkv_shape, dtype=q.dtype, device=q.device)
        _flash_attn_varlen_backward(dout, q, k, v, out, softmax_lse, dqkv[:, 0], dqkv[:, 1], dqkv[:, 2],
                                    cu_seqlens, cu_seqlens, ctx.max_seqlen, ctx.max_seqlen, ctx.dropout_p,
                                    ctx.softmax_scale, ctx.causal, ctx.window_size, rng_state=rng_state)
        dqkv = dqkv[..., : dout.shape[-1]]
        return dqkv, None, None, None, None, None, None, None


class FlashAttnVarlenKVPackedFunc(torch.autograd.Function):
    native = flash_attn_gpu.host.varlen_kvpacked_func

    @staticmethod
    def forward(ctx, q, kv, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, dropout_p,
                softmax_scale, causal, window_size, return_softmax):
        if softmax_scale is None:
            softmax_scale = q.shape[-1] ** (-0.5)
        out, q, k, v, out_padded, softmax_lse, S_dmask, rng_state = _flash_attn_varlen_forward(
            q, kv[:, 0], kv[:, 1], cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k,
            dropout_p, softmax_scale, causal=causal, window_size=window_size,
            return_softmax=return_softmax and dropout_p > 0,
        )
        _save(ctx, (q, k, v, out_padded, softmax_lse, cu_seqlens_q, cu_seqlens_k, rng_state), dropout_p,
              softmax_scale, causal, window_size, max_seqlen_q=max_seqlen_q, max_seqlen_k=max_seqlen_k)
        return out if not return_softmax else (out, softmax_lse, S_dmask)

    @staticmethod
    def backward(ctx, dout, *args):
        q, k, v, out, softmax_lse, cu_seqlens_q, cu_seqlens_k, rng_state = ctx.saved_tensors
        dq = torch.empty_like(q)
        kv_shape = k.shape[:-2] + (2, *k.shape[-2:])
        dkv = torch.empty(kv_shape, dtype=k.dtype, device=k.device)
        _flash_attn_varlen_backward(dout, q, k, v, out, softmax_lse, dq, dkv[:, 0], dkv[:, 1], cu_seqlens_q,
                                    cu_seqlens_k, ctx.max_seqlen_q, ctx.max_seqlen_k, ctx.dropout_p,
                                    ctx.softmax_scale, ctx.causal, ctx.window_size, rng_state=rng_state)
        dq, dkv = dq[..., : dout.shape[-1]], dkv[..., : dout.shape[-1]]
        return dq, dkv, None, None, None, None, None, None, None, None, None


def flash_attn_qkvpacked_func(qkv, dropout_p=0.0, softmax_scale=None, causal=False,
                              window_size=(-1, -1), return_attn_probs=False):
    """qkv: (batch_size, seqlen, 3, nheads, headdim).  Returns out (batch_size, seqlen, nheads,
    headdim), or (out, softmax_lse, None) if return_attn_probs.  Masks are bottom-right aligned;
    window_size=(left, right), -1 = unbounded."""
    return _apply(FlashAttnQKVPackedFunc, (qkv,), qkv, dropout_p, softmax_scale, causal, window_size,
                   return_attn_probs)


def flash_attn_kvpacked_func(q, kv, dropout_p=0.0, softmax_scale=None, causal=False,
                             window_size=(-1, -1), return_attn_probs=False):
    """q: (batch_size, seqlen, nheads, headdim); kv: (batch_size, seqlen_k, 2, nheads_k, headdim).
    MQA/GQA when nheads_k < nheads (nheads % nheads_k == 0)."""
    return _apply(FlashAttnKVPackedFunc, (q, kv), q, kv, dropout_p, softmax_scale, causal, window_size,
                   return_attn_probs)


def flash_attn_func(q, k, v, dropout_p=0.0, softmax_scale=None, causal=False, window_size=(-1, -1),
                    return_attn_probs=False):
    """q: (batch_size, seqlen, nheads, headdim); k, v: (batch_size, seqlen_k, nheads_k, headdim).

    softmax_scale defaults to 1/sqrt(headdim).  causal masks are aligned to the bottom right corner
    of the attention matrix; with window_size=(left, right) query i attends to keys in
    [i + seqlen_k - seqlen_q - left, i + seqlen_k - seqlen_q + right].  A row that sees no key
    gives an all-zero output.  Returns out (batch_size, seqlen, nheads, headdim), or
    (out, softmax_lse [batch_size, nheads, seqlen] fp32, None) if return_attn_probs."""
    return _apply(FlashAttnFunc, (q, k, v), q, k, v, dropout_p, softmax_scale, causal, window_size,
                   return_attn_probs)


def flash_attn_varlen_qkvpacked_func(qkv, cu_seqlens, max_seqlen, dropout_p=0.0, softmax_scale=None,
                                     causal=False, window_size=(-1, -1), return_attn_probs=False):
    """qkv: (total, 3, nheads, headdim); cu_seqlens: (batch_size + 1,) int32 prefix sums."""
    return _apply(FlashAttnVarlenQKVPackedFunc, (qkv,), qkv, cu_seqlens, max_seqlen, dropout_p,
                   softmax_scale, causal, window_size, return_attn_probs)


def flash_attn_varlen_kvpacked_func(q, kv, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k,
                                    dropout_p=0.0, softmax_scale=None, causal=False,
                                    window_size=(-1, -1), return_attn_probs=False):
    """q: (total_q, nheads, headdim); kv: (total_k, 2, nheads_k, headdim)."""
    return _apply(FlashAttnVarlenKVPackedFunc, (q, kv), q, kv, cu_seqlens_q, cu_seqlens_k,
                   max_seqlen_q, max_seqlen_k, dropout_p, softmax_scale, causal, window_size, return_attn_probs)


def flash_attn_varlen_func(q, k, v, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k,
                           dropout_p=0.0, softmax_scale=None, causal=False, window_size=(-1, -1),
                           return_attn_probs=False):
    """q: (total_q, nheads, headdim); k, v: (total_k, nheads_k, headdim); cu_seqlens_*:
    (batch_size + 1,) int32 prefix sums of the sequence lengths.  softmax_lse is
    (batch_size, nheads, max_seqlen_q)."""
    return _apply(FlashAttnVarlenFunc, (q, k, v), q, k, v, cu_seqlens_q, cu_seqlens_k, max_seqlen_q,
                   max_seqlen_k, dropout_p, softmax_scale, causal, window_size, return_attn_probs)


def flash_attn_with_kvcache(q, k_cache, v_cache, k=None, v=None, rotary_cos=None, rotary_sin=None,
                            cache_seqlens: Optional[Union[int, torch.Tensor]] = None,
                            cache_batch_idx: Optional[torch.Tensor] = None, softmax_scale=None,
                            causal=False, window_size=(-1, -1), rotary_interleaved=True,
                            num_splits=0):
    """Attention against a KV cache, optionally appending k / v (new keys rotated with
    rotary_cos / rotary_sin) in place first.

    q: (batch_size, seqlen, nheads, headdim); k_cache, v_cache: (batch_size_cache, seqlen_cache,
    nheads_k, headdim); k, v: (batch_size, seqlen_new, nheads_k, headdim) written at rows
    cache_seqlens[b] ...; rotary_cos/sin: (seqlen_ro, rotary_dim / 2); cache_seqlens: int or
    (batch_size,) int32; cache_batch_idx: (batch_size,) int32 cache rows to use.  New keys are
    rotated at positions cache_seqlens + t; q at cache_seqlens + i when causal or local, else at
    cache_seqlens.  num_splits: 0 = choose automatically, 1 = do not split, n = split the keys
    into at most n chunks.  Returns out: (batch_size, seqlen, nheads, headdim)."""
    if not torch.compiler.is_compiling():
        out = flash_attn_gpu.host.with_kvcache(q, k_cache, v_cache, k, v, rotary_cos, rotary_sin, cache_seqlens, cache_batch_idx,
                                               softmax_scale, causal, window_size, rotary_interleaved, num_splits)
        if out is not None:
            return out
    assert k_cache.stride(-1) == 1, "k_cache must have contiguous last dimension"
    assert v_cache.stride(-1) == 1, "v_cache must have contiguous last dimension"
    q, k, v = [_maybe_contiguous(x) for x in (q, k, v)]
    if softmax_scale is None:
        softmax_scale = q.shape[-1] ** (-0.5)
    if cache_seqlens is not None and isinstance(cache_seqlens, int):
        cache_seqlens = torch.full((k_cache.shape[0],), cache_seqlens, dtype=torch.int32,
                                   device=k_cache.device)
        cache_seqlens = _maybe_contiguous(cache_seqlens)
    cache_batch_idx = _maybe_contiguous(cache_batch_idx)
    out, softmax_lse = flash_attn_gpu.fwd_kvcache(
        q, k_cache, v_cache, k, v, cache_seqlens, rotary_cos, rotary_sin, cache_batch_idx, None,
        softmax_scale, causal, window_size[0], window_size[1], rotary_interleaved, num_splits,
    )
    return out
