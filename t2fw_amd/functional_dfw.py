"""Autograd boundary of the delta rule: same call as the reference's
``DFWFunction.apply(query, key, value, state)`` (t2fw/functional_dfw.py:29-65), backed by the
HIP kernels in libt2fw_hip.so.  As in the reference, backward consumes the per-step deltas
and the final state saved by forward (t2fw/functional_dfw.py:46-51)."""
import functools
import os

import torch

from . import _lib
from .functional_lfw import _check_input, _dtype_code, _flags, _on_device


def _dfw_flags(dtype):
    """Kernel-path flags of a call.  bfloat16 tensors take the matrix-core kernels' single-bf16-operand mode
    (include/t2fw_hip.h, T2FW_FLAG_BF16_OPERANDS): their inputs are bf16 numbers already, and rounding the
    intermediates to bf16 as well leaves the results at the accuracy that storing them in bf16 has anyway
    (measured against the fp64 oracle: 4e-3 .. 6e-3 of max|ref| per tensor, against 2e-3 .. 3.5e-3 for the exact
    per-step kernels), at 1.7 times the speed.  float32 and float16 tensors keep the split operands (results at
    the accuracy of the exact kernels for the type).  T2FW_FLAGS overrides this as everywhere."""
    if os.environ.get("T2FW_FLAGS"):
        return _flags()
    return _lib.FLAG_BF16_OPERANDS if dtype == torch.bfloat16 else _lib.FLAG_AUTO


def _dfw_forward(query, key, value, state):
    """The forward kernels on [B,T,M], [B,T,M], [B,T,D], [B,D,M]: (outputs, final_state, delta)"""
    dev = value.device
    with _on_device(dev):
        return _lib.host().dfw_forward(query, key, value, state, _dtype_code(value.dtype), _dfw_flags(value.dtype),
                                       _lib.current_stream(dev))


def _dfw_backward(grad_output, grad_state, query, key, delta, final_state):
    """The backward kernels: (d_q, d_k, d_v, d_s), the order of t2fw/csrc/dfw_kernel.cu:557"""
    dev = delta.device
    with _on_device(dev):
        return _lib.host().dfw_backward(grad_output, grad_state, query, key, delta, final_state, _dtype_code(delta.dtype),
                                        _dfw_flags(delta.dtype), _lib.current_stream(dev))


# ---- value widths that are multiples of 64 (key width 64) as independent blocks -----------------------------
# The rows of the state do not interact in the delta rule either: S[d, :] sees v[d], q, k only (the key side is
# coupled through delta_t = v_t - S_{t-1} k_t, a sum over all of M, so only the value side can be cut).  A
# [D, 64] state with D a multiple of 64 is D / 64 independent [64, 64] recurrences that share q and k.  The matrix-core
# kernels read and write the value side's [B,T,D] arrays in place; d_query and d_key are sums over the blocks, which the kernels
# make (float16 tensors: they come per block, and one more launch adds them up).  Arrays that those kernels do not take (not 16-byte aligned, T * D of 2^31 and more) are cut into copies that run as extra
# batch rows.  B=48, T=777, D=128 bf16, GPU time of a training step: 99 us, with copies 118 (kernels 85 and 78).
def _value_block_count(value, query):
    D, M = value.shape[-1], query.shape[-1]
    if M != 64 or D % 64 or D <= 64 or value.dtype not in (torch.float32, torch.float16, torch.bfloat16):
        return 0
    if _dfw_flags(value.dtype) & _lib.FLAG_FORCE_SCAN:
        return 0
    return D // 64


@functools.lru_cache(maxsize=256)
def _value_block_plans(B, T, nd):
    """Descriptors of the block copies (csrc/blocks.hip), one launch each way"""
    D = 64 * nd
    cut = ((B, nd, T), (T * D, 64, D))                       # [B,T,64 nd] -> [B nd,T,64]
    repeat = ((B, nd, T), (T * 64, 0, 64))                   # [B,T,64] -> [B nd,T,64]
    join = ((B, T, nd), (nd * T * 64, 64, T * 64))           # [B nd,T,64] -> [B,T,64 nd]
    total = ((B, T), (nd * T * 64, 64), nd, T * 64)          # [B nd,T,64] -> [B,T,64], the sum over the blocks
    kept = ((B * T,), (64,))                                 # q and k as they are
    return {"kept": _lib.block_plan(kept, kept), "inputs": _lib.block_plan(repeat, repeat, cut), "outputs": _lib.block_plan(join),
            "grads_in": _lib.block_plan(cut), "grads_out": _lib.block_plan(total, total, join),
            "key_grads": _lib.block_plan(total, total)}


def _dfw_forward_blocked(query, key, value, state, nd, need_grad=True):
    """(outputs, final_state, what the backward needs: q, k, delta and the final state, whole or of the blocks).  q and k
    are kept as copies: a caller may change its own before the backward."""
    B, D, M = state.shape
    T = value.shape[1]
    plans = _value_block_plans(B, T, nd)
    with _on_device(value.device):
        if value.is_cuda:
            res = _lib.host().dfw_forward_blocks(query, key, value, state, _dtype_code(value.dtype), _dfw_flags(value.dtype),
                                                 _lib.current_stream(value.device), plans["kept"] if need_grad else None)
            if res is not None:
                outputs, final_state, delta, q, k = res
                return outputs, final_state, (q, k, delta, final_state) if need_grad else ()
        qb, kb, vb = (value.new_empty((B * nd, T, 64)) for _ in range(3))
        _lib.block_copy(plans["inputs"], (query, key, value), (qb, kb, vb))
        out_b, fin_b, delta_b = _dfw_forward(qb, kb, vb, state.view(B * nd, 64, M))
        outputs = torch.empty_like(value)
        _lib.block_copy(plans["outputs"], (out_b,), (outputs,))
    return outputs, fin_b.view(B, D, M), (qb, kb, delta_b, fin_b)


def _dfw_backward_blocked(grad_output, grad_state, q, k, delta, final_state, nd):
    B, T, D = grad_output.shape
    M = q.shape[2]
    plans = _value_block_plans(B, T, nd)
    with _on_device(q.device):
        if delta.shape[2] == D and _dfw_flags(delta.dtype) & _lib.FLAG_FORCE_SCAN:      # asked for since: its kernels take blocks
            qb, kb, delta_b = (delta.new_empty((B * nd, T, 64)) for _ in range(3))
            _lib.block_copy(plans["inputs"], (q, k, delta), (qb, kb, delta_b))
            q, k, delta, final_state = qb, kb, delta_b, final_state.reshape(B * nd, 64, M)
        if delta.shape[2] == D:                               # whole arrays: the kernels took them as they are
            d_qb, d_kb, d_v, d_s = _lib.host().dfw_backward_blocks(grad_output, grad_state, q, k, delta, final_state,
                                                                   _dtype_code(delta.dtype), _dfw_flags(delta.dtype),
                                                                   _lib.current_stream(q.device))
            if d_qb.dim() == 3:
                return d_qb, d_kb, d_v, d_s
            d_q, d_k = torch.empty_like(q), torch.empty_like(k)
            _lib.block_copy(plans["key_grads"], (d_qb, d_kb), (d_q, d_k))
            return d_q, d_k, d_v, d_s
        go_b = torch.empty_like(delta)
        _lib.block_copy(plans["grads_in"], (grad_output,), (go_b,))
        d_qb, d_kb, d_vb, d_sb = _dfw_backward(go_b, grad_state.reshape(B * nd, 64, M), q, k, delta, final_state)
        d_q, d_k, d_v = q.new_empty((B, T, M)), q.new_empty((B, T, M)), q.new_empty((B, T, D))
        _lib.block_copy(plans["grads_out"], (d_qb, d_kb, d_vb), (d_q, d_k, d_v))
    return d_q, d_k, d_v, d_sb.view(B, D, M)


class DFWFunction(torch.autograd.Function):
    """Delta rule: out_t = S_{t-1} q_t, S_t = S_{t-1} + (v_t - S_{t-1} k_t) (x) k_t.
    Any scalar write strength is assumed to be absorbed into the key.
    D = M = 64 (fp32, fp16, bf16) runs on the matrix-core kernels, a value width that is another multiple of 64
    (with M = 64) as independent blocks on the same kernels, everything else on the exact per-step kernels."""

    @staticmethod
    def forward(ctx, query, key, value, state):
        """Return: (outputs [B,T,D], final state [B,D,M])"""
        # same asserts as t2fw/functional_dfw.py:38-40
        assert query.shape == key.shape
        assert query.dtype == value.dtype
        assert state.dtype == value.dtype
        assert key.dtype == value.dtype
        for t, n in ((query, "query"), (key, "key"), (value, "value"), (state, "state")):
            _check_input(t, n)
        if value.dim() != 3 or query.dim() != 3 or state.dim() != 3:
            raise RuntimeError("t2fw: expected query,key [B,T,M]; value [B,T,D]; state [B,D,M]")
        B, T, D = value.shape
        M = query.shape[2]
        if query.shape[0] != B or query.shape[1] != T or tuple(state.shape) != (B, D, M):
            raise RuntimeError("t2fw: inconsistent shapes query %s, value %s, state %s"
                               % (tuple(query.shape), tuple(value.shape), tuple(state.shape)))
        _dtype_code(value.dtype)
        ctx.value_blocks = _value_block_count(value, query)
        if ctx.value_blocks:
            outputs, final_state, kept = _dfw_forward_blocked(query, key, value, state, ctx.value_blocks, any(ctx.needs_input_grad))
            ctx.save_for_backward(*kept)
        else:
            outputs, final_state, delta = _dfw_forward(query, key, value, state)
            ctx.save_for_backward(query, key, delta, final_state)
        return outputs, final_state

    @staticmethod
    def backward(ctx, grad_output, grad_state):
        query, key, delta, final_state = ctx.saved_tensors
        # t2fw/functional_dfw.py:58-59
        assert grad_state.dtype == delta.dtype
        assert grad_output.dtype == delta.dtype
        grad_output = grad_output.contiguous()
        grad_state = grad_state.contiguous()
        if ctx.value_blocks:
            return _dfw_backward_blocked(grad_output, grad_state, query, key, delta, final_state, ctx.value_blocks)
        return _dfw_backward(grad_output, grad_state, query, key, delta, final_state)
