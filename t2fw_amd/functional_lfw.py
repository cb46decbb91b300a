"""Autograd boundary of the decay rule: same call as the reference's
``LFWFunction.apply(value, forget, query, key, f_key, state)``
(t2fw/functional_lfw.py:31-78), backed by the HIP kernels in libt2fw_hip.so.

Differences from the reference that a caller can observe:
  * the state is stored only every ``C`` steps (``[B, ceil(T/C), D, K]``) instead of
    every step (``[B, T, D, K]``, t2fw/csrc/lfw_kernel.cu:140-144); backward recomputes
    inside each chunk.  ``next_state`` is its own ``[B, D, K]`` tensor, not a view.
  * bf16 is accepted in addition to fp64/fp32/fp16.
  * kernels run on the current torch stream and on the inputs' device.
"""
import contextlib
import ctypes
import functools
import os

import torch

from . import _lib
from .path_hint import ForwardHints, choose_backward_flags

DEFAULT_CKPT_INTERVAL = 64


def _ckpt_interval():
    v = os.environ.get("T2FW_CKPT_INTERVAL")
    return int(v) if v else DEFAULT_CKPT_INTERVAL


def _flags():
    """Kernel-path flags (include/t2fw_hip.h): 0 = automatic, 1 = exact scan kernels only,
    2 = fp16 matrix-core operands for fp16 tensors, 8 = block-wise matrix-core kernels.
    Overridable with T2FW_FLAGS."""
    v = os.environ.get("T2FW_FLAGS")
    return int(v) if v else _lib.FLAG_AUTO


@functools.lru_cache(maxsize=256)
def _sizes(rows, T, D, K, C, code, flags):
    """(checkpoints per row, forward workspace bytes, forward + backward workspace bytes, flag regions)
    of a shape: calls into the library that a training loop would otherwise repeat every step"""
    lib = _lib.load()
    regions = (ctypes.c_int64 * 6)()
    _lib.check(lib.t2fw_lfw_flag_regions(rows, T, D, K, C, code, flags, regions))
    return (lib.t2fw_lfw_num_ckpt(T, C), lib.t2fw_lfw_forward_workspace_bytes(rows, T, D, K, C, code, flags),
            lib.t2fw_lfw_workspace_bytes(rows, T, D, K, C, code, flags), tuple(regions))


@functools.lru_cache(maxsize=256)
def _forward_plan(rows, T, D, K, C, dtype, flags, need_grad):
    """The flags a forward call of this shape runs with (and its backward after it), then _sizes with these flags"""
    flags = _exact_chunk_flags(rows, T, D, K, C, dtype, flags, need_grad)
    return (flags,) + _sizes(rows, T, D, K, C, _lib.DTYPE_CODE[dtype], flags)


def _host_hints_enabled():
    """T2FW_HOST_HINTS=0 keeps every workspace in device memory (the backward then decides on the device).  So does
    torch.use_deterministic_algorithms: whether the hints are there when the backward is issued depends on the host's
    pace, and for a batch with hinted rows the two backward kernels differ in the last bits."""
    return os.environ.get("T2FW_HOST_HINTS", "1") != "0" and not torch.are_deterministic_algorithms_enabled()


_AS_IT_IS = contextlib.nullcontext()      # may be entered any number of times, by any thread


def _on_device(dev):
    """Make ``dev`` current for the allocations and the launch, without the cost of switching when it already is."""
    if dev.index is None or dev.index == torch.cuda.current_device():      # (host memory has no index)
        return _AS_IT_IS
    return torch.cuda.device(dev)


def _check_input(t, name):
    # mirrors CHECK_INPUT of t2fw/csrc/lfw.cpp:24-26 (TORCH_CHECK -> RuntimeError)
    if not t.is_cuda:
        raise RuntimeError("%s must be a CUDA tensor" % name)
    if not t.is_contiguous():
        raise RuntimeError("%s must be contiguous" % name)


def _dtype_code(dtype):
    try:
        return _lib.DTYPE_CODE[dtype]
    except KeyError:
        raise RuntimeError("t2fw: unsupported dtype %s" % dtype)


# Where the chunk-parallel exact kernels (three launches per direction) take the place of the per-step ones (one launch
# forward, two backward): where a sequence is long enough for the launches, and the rows are few enough that the per-step
# kernels leave the chip idle.  Both sides in microseconds of GPU time, per-step / chunk-parallel.
#   Steps, forward + backward: 24 rows of 16 x 16, 224 steps 156 / 57 (a host that needs 180 for the launches: 180 / 190).
#   64 x 64 (float32; kernels of its own, on matrix instructions): 96 rows, 128 steps 148 / 78 (as issued by such a host 148 / 154),
#     224 steps 238 / 106, 1024 steps 1002 / 294; 256 rows x 256 steps 542 / 209, forward alone 123 / 76.  Fewer steps and more rows
#     would gain too (512 rows x 256 steps 958 / 392): the limits were measured for the step-by-step kernels that these replaced.
#   A width of 8 or less, where a workgroup of the per-step kernels takes several rows' worth of channels: 1024 rows of 8 x 8,
#     224 steps 1341 / 345; 64 x 8 forward alone, 128 rows x 224 steps 1.17 times as fast, 160 rows 1.00, 256 rows 0.75.
#   16 x 16: 384 rows x 224 steps 170 / 145, 512 rows 172 / 184, 768 rows 222 / 259, 1024 rows 248 / 332; x 448 steps 512 rows
#     321 / 323, 640 rows 414 / 394, 768 rows 419 / 456.
#   32 x 32: 384 rows x 224 steps 254 / 248, 512 rows 288 / 314.  33 x 17: 256 rows 257 / 250, 341 rows 288 / 325.
#   63 x 63: 160 rows x 224 steps 313 / 300, 192 rows 332 / 363, 256 rows 457 / 459; x 1024 steps 256 rows 1.07 times as fast.
#   Forward alone (one launch against three): up to 256 tiles of value channels 1.1 to 6 times as fast at every width; 384
#     tiles 0.82 (16 x 16) to 1.07 (33 x 17) at 224 steps, 1.06 to 1.33 at 1024; 512 tiles 0.68 to 0.88, where the per-step
#     kernel's workgroups come to two per CU; 640 and 768 tiles 1.02 to 1.48 from 448 steps on; 1024 tiles 0.72 to 1.0.
EXACT_CHUNKS_MIN_STEPS = 224


def _exact_chunks_faster(rows, T, D, K, need_grad):
    """Whether the chunk-parallel exact kernels take less time for ``rows`` states of D x K (up to 64 x 64) over T steps."""
    if T < EXACT_CHUNKS_MIN_STEPS:
        return False
    if D == 64 and K == 64:
        return rows <= 256
    if not need_grad:
        tiles = rows * -(-D // 16)
        if K <= 8:
            return tiles <= (1024 if D <= 16 else 512)
        return tiles <= 256 or (T >= 1024 and tiles <= 384) or (T >= 448 and 512 < tiles <= 768)
    narrow, wide = min(D, K), max(D, K)
    tiles = rows * -(-wide // 16)
    if narrow <= 8:
        return tiles <= 1024
    if wide <= 16:
        return tiles <= (384 if T < 448 else 640)
    if narrow <= 32:
        return tiles <= 768
    return tiles <= (640 if T < 448 else 1024)


def _exact_chunk_flags(rows, T, D, K, C, dtype, flags, need_grad):
    """``flags`` of a call that the 16-bit matrix-core kernels do not take, with FLAG_EXACT_CHUNKS added where the
    chunk-parallel exact kernels serve it (states of up to 64 x 64, checkpoints every 64 steps) and are faster; a caller's
    own flags stand."""
    if flags != _lib.FLAG_AUTO or C != 64 or D > 64 or K > 64 or dtype == torch.float64:
        return flags
    if (D == 64 and K == 64 and dtype != torch.float32) or not _exact_chunks_faster(rows, T, D, K, need_grad):
        return flags
    return flags | _lib.FLAG_EXACT_CHUNKS


# ---- widths that are multiples of 64 (other than 64 x 64) as independent 64 x 64 blocks -------------------
# The recurrence couples neither the rows of the state nor its columns: S[d, k] sees x[d], f[d], k[k], f_key[k]
# only, and o[d] is a sum over k.  A D x K state is (D / 64) (K / 64) independent 64 x 64 recurrences -- value
# channels 64 i .. 64 i + 63 with key channels 64 j .. 64 j + 63 -- whose outputs add up over j.  For fp16 / bf16
# tensors the blocks run as heads through the head-strided entry points, i.e. on the matrix-core
# kernels, which take 64 x 64 states only; the exact per-step kernels that would otherwise serve such widths take
# 4.2 ms for a forward + backward at B=24, T=1024, D=K=128 where the blocks take 0.16 ms.  The reference has one
# kernel for every shape (t2fw/csrc/lfw_kernel.cu:105-121).
def _block_counts(value, query, flags):
    """(D / 64, K / 64) if tensors of these widths run as blocks, else None"""
    D, K = value.shape[-1], query.shape[-1]
    if value.dim() not in (3, 4) or value.dtype not in (torch.float16, torch.bfloat16) or (flags & _lib.FLAG_FORCE_SCAN):
        return None
    if D % 64 or K % 64 or D == 0 or K == 0 or (D == 64 and K == 64):
        return None
    return D // 64, K // 64


# Tensors are [B,T,W] or, with a head axis, [B,T,H,W]; states [B,D,K] or [B,H,D,K].  Block (i, j) of head h becomes
# head (h * nd + i) * nk + j of the 64-wide call.  The blocks of a call's tensors are cut in one launch and its results
# put together in another (csrc/blocks.hip); what has only one block on the other side is a view and costs nothing.
@functools.lru_cache(maxsize=256)
def _block_plans(B, T, H, nd, nk):
    lines, rows, D, K = B * T * H, B * H, 64 * nd, 64 * nk
    value = ((lines, nd, nk), (D, 64, 0))
    key = ((lines, nd, nk), (K, 0, 64))
    state = ((rows, nd, nk, 64), (D * K, 64 * K, 64, K))
    whole_state = ((rows, nd, 64, nk), (D * K, nk * 4096, 64, 4096))
    key_sum = ((lines, nd), (nd * nk * 64, nk * 64), nk, 64)
    value_sum = ((lines, nk), (nd * nk * 64, 64), nd, nk * 64)
    inputs = [p for p, kept in ((value, nk > 1), (value, nk > 1), (key, nd > 1), (key, nd > 1), (key, nd > 1),
                                (state, nk > 1)) if kept]
    grads = [p for p, kept in ((key_sum, nk > 1), (key_sum, nk > 1), (value_sum, nd > 1), (value_sum, nd > 1),
                               (value_sum, nd > 1), (whole_state, nk > 1)) if kept]
    return {"inputs": _lib.block_plan(*inputs),
            "outputs": _lib.block_plan(key_sum, whole_state) if nk > 1 else None,
            "grads_in": _lib.block_plan(value, state) if nk > 1 else None,
            "grads_out": _lib.block_plan(*grads)}


def _block_dims(value, blocks):
    """(B, T, H, blocks along the value side, along the key side) of [B,T,W] or [B,T,H,W] tensors"""
    return value.shape[0], value.shape[1], value.shape[2] if value.dim() == 4 else 1, blocks[0], blocks[1]


def _run_plan(plan, srcs, dsts, copied):
    """dsts from srcs in one launch; an entry that is not ``copied`` is a view of its source, of the shape of dsts"""
    if srcs[0].is_cuda:
        outs = _lib.host().blocks_of(plan, tuple(srcs), tuple(dsts), tuple(copied), _dtype_code(srcs[0].dtype),
                                     _lib.current_stream(srcs[0].device))
        if outs is not None:
            return outs
    outs, cs, cd = [], [], []
    for s, shape, c in zip(srcs, dsts, copied):
        if c:
            t = torch.empty(shape, dtype=s.dtype, device=s.device)
            cs.append(s)
            cd.append(t)
            outs.append(t)
        else:
            outs.append(s.view(shape))
    if cs:
        _lib.block_copy(plan, cs, cd)
    return outs


def _input_blocks(tensors, B, T, H, nd, nk):
    """x, f, q, k, f_key [B,T,(H,)W] -> [B,T,H nd nk,64], state -> [B,H nd nk,64,64]"""
    v, k = nk > 1, nd > 1
    tok, st = (B, T, H * nd * nk, 64), (B, H * nd * nk, 64, 64)
    with _on_device(tensors[0].device):
        return _run_plan(_block_plans(B, T, H, nd, nk)["inputs"], tensors, (tok,) * 5 + (st,), (v, v, k, k, k, v))


class _BlockedCall:
    """What a forward call on blocks leaves for its backward call: the block copies of the six inputs (made once,
    not again in the backward) and the hints of the call underneath.  Travels in the ``hints`` slot."""
    __slots__ = ("tensors", "hints")

    def __init__(self, tensors, hints):
        self.tensors = tensors
        self.hints = hints


def _lfw_forward_blocked(value, forget, query, key, f_key, state, need_grad, blocks):
    dims = _block_dims(value, blocks)
    tensors = _input_blocks((value, forget, query, key, f_key, state), *dims)
    out_b, nxt_b, ckpt, C, flags, hints = _lfw_forward(*tensors, need_grad, heads=True)
    kept = _BlockedCall(tensors, hints) if need_grad else None
    summed = blocks[1] > 1
    with _on_device(value.device):
        out, nxt = _run_plan(_block_plans(*dims)["outputs"], (out_b, nxt_b), (value.shape, state.shape), (summed, summed))
    return out, nxt, ckpt, C, flags, kept


def _lfw_backward_blocked(grad_output, grad_state, value, forget, query, key, f_key, state, ckpt, C, flags, kept, blocks):
    """The adjoint of the copies is the sum over the blocks that share a channel (fp32 sums)."""
    B, T, H, nd, nk = dims = _block_dims(value, blocks)
    if isinstance(kept, _BlockedCall):
        tensors, hints = kept.tensors, kept.hints
    else:
        tensors, hints = _input_blocks((value, forget, query, key, f_key, state), *dims), None
    plans = _block_plans(*dims)
    v, k = nk > 1, nd > 1
    with _on_device(value.device):
        go_b, gs_b = _run_plan(plans["grads_in"], (grad_output, grad_state), (tensors[0].shape, tensors[5].shape), (v, v))
        grads = _lfw_backward(go_b, gs_b, *tensors, ckpt, C, flags, heads=True, hints=hints)
        return tuple(_run_plan(plans["grads_out"], grads, (value.shape, value.shape, query.shape, query.shape, query.shape,
                                                           state.shape), (v, v, k, k, k, v)))


def _checked_shape(value, forget, query, key, f_key, state, heads):
    """(B, T, H, D, K) of a call, or the error that it is: checks as in t2fw/functional_lfw.py:42-49 and
    t2fw/csrc/lfw.cpp:24-26,36-41 (``lfw_shape`` of csrc/host.cpp only tells whether there is one)"""
    assert value.shape == forget.shape
    assert query.shape == key.shape
    assert query.shape == f_key.shape
    assert forget.dtype == value.dtype
    assert query.dtype == value.dtype
    assert f_key.dtype == value.dtype
    assert state.dtype == value.dtype
    assert key.dtype == value.dtype
    for t, n in ((value, "x"), (forget, "f"), (query, "query"), (key, "key"),
                 (f_key, "f_key"), (state, "state")):
        _check_input(t, n)
    nd = 4 if heads else 3
    if value.dim() != nd or query.dim() != nd or state.dim() != nd:
        raise RuntimeError("t2fw: expected x,f [B,T,H,D]; q,k,f_key [B,T,H,K]; state [B,H,D,K]" if heads else
                           "t2fw: expected x,f [B,T,D]; q,k,f_key [B,T,K]; state [B,D,K]")
    B, T = value.shape[:2]
    H = value.shape[2] if heads else 1
    D, K = value.shape[-1], query.shape[-1]
    if tuple(query.shape[:-1]) != tuple(value.shape[:-1]) or \
            tuple(state.shape) != ((B, H, D, K) if heads else (B, D, K)):
        raise RuntimeError("t2fw: inconsistent shapes x %s, query %s, state %s"
                           % (tuple(value.shape), tuple(query.shape), tuple(state.shape)))
    return B, T, H, D, K


def _lfw_forward(value, forget, query, key, f_key, state, need_grad, heads=False, logits=False):
    """The checks, then the forward kernels.  heads=False: x,f [B,T,D]; q,k,f_key [B,T,K]; state [B,D,K].
    heads=True: x,f [B,T,H,D]; q,k,f_key [B,T,H,K]; state [B,H,D,K].  Returns (outputs, next_state, ckpt or
    None, checkpoint interval, flags, hints): ``hints`` is None, or the forward's verdict on which backward
    path the gates allow, readable from the host once the forward has run (path_hint.py).  logits=True: ``forget`` and
    ``f_key`` are gate logits, and the gates follow what is returned."""
    host = _lib.host() if _lib.loaded() else None
    dims = host.lfw_shape(value, forget, query, key, f_key, state, heads) if host is not None else None
    B, T, H, D, K = dims if dims is not None else _checked_shape(value, forget, query, key, f_key, state, heads)
    code = _dtype_code(value.dtype)
    flags = _flags()
    blocks = _block_counts(value, query, flags)
    if blocks is not None:
        if logits:
            forget, f_key = sigmoid_gates(forget, f_key)
        res = _lfw_forward_blocked(value, forget, query, key, f_key, state, need_grad, blocks)
        return (*res, forget, f_key) if logits else res
    if host is None:
        host = _lib.host()
    C = _ckpt_interval()
    dev = value.device
    flags, nc, ws_bytes, _, regions = _forward_plan(B * H, T, D, K, C, value.dtype, flags, need_grad)
    with _on_device(dev):
        hints = None
        ws_address = event = 0                             # the workspace is allocated for the call
        if need_grad and ws_bytes and regions[3] and regions[5] and _host_hints_enabled() and ForwardHints.usable(dev):
            # a backward on the matrix cores will follow: the workspace goes to pinned host memory
            hints = ForwardHints(dev, ws_bytes, regions[2], regions[3], B * H)
            ws_address, event = hints.workspace()[0].value, hints.event()
        res = host.lfw_forward(value, forget, query, key, f_key, state, heads, nc if need_grad else -1, C, code, flags, ws_address, ws_bytes,
                               _lib.current_stream(dev), logits, event)
        if hints is not None:
            hints.launched()
    if logits:
        return *res[:3], C, flags, hints, *res[3:]
    outputs, next_state, ckpt = res
    return outputs, next_state, ckpt, C, flags, hints


def _lfw_backward(grad_output, grad_state, value, forget, query, key, f_key, state, ckpt, C, flags, heads=False,
                  hints=None):
    """The backward kernels; gradients in the order of t2fw/csrc/lfw.cpp:95, laid out as their inputs.
    ``hints``: what the forward call on the same gates left for this call (path_hint.py), or None."""
    # t2fw/functional_lfw.py:71-72
    assert grad_state.dtype == value.dtype
    assert grad_output.dtype == value.dtype
    grad_output = grad_output.contiguous()
    grad_state = grad_state.contiguous()
    blocks = _block_counts(value, query, flags)
    if blocks is not None:
        return _lfw_backward_blocked(grad_output, grad_state, value, forget, query, key, f_key, state, ckpt, C,
                                     flags, hints, blocks)
    B, T = value.shape[:2]
    H = value.shape[2] if heads else 1
    D, K = value.shape[-1], query.shape[-1]
    code = _dtype_code(value.dtype)
    host = _lib.host()
    dev = value.device
    if hints is not None:
        flags = choose_backward_flags(flags, hints.hinted_rows(), B * H, value.dtype == torch.float16)
    ws_bytes = _sizes(B * H, T, D, K, C, code, flags)[2]
    with _on_device(dev):
        grads, args, ws = host.lfw_backward_arguments(grad_output, grad_state, value, forget, query, key, f_key, state, ckpt, heads,
                                                      C, code, flags, ws_bytes, _lib.current_stream(dev))
        lib = _lib.load()
        _lib.check((lib.t2fw_lfw_backward_heads if heads else lib.t2fw_lfw_backward)(*args))
    return grads


class LFWFunction(torch.autograd.Function):
    """Decay update rule S_t = S_{t-1} * (f_t (x) f_key_t) + x_t (x) k_t, o_t = S_t q_t.
    Inputs are already gated (no sigmoid is applied here), as in the reference.
    fp16 / bf16 tensors with D = K = 64 run on the matrix-core kernels, those whose widths are other multiples
    of 64 as independent 64 x 64 blocks on the same kernels (``_block_counts`` above), everything else on the
    exact kernels (per-step, or with the chunks of a row side by side: ``_exact_chunk_flags``); T2FW_FLAGS=1 keeps
    the per-step kernels for every shape.

    Which kernels run depends on the whole call: the number of rows and steps, and whether gradients are wanted.  The
    results of a row are then equal to rounding and not to the bit, for instance the first pass of activation
    checkpointing, which has no gradients, and its recomputation, which does.  torch.use_deterministic_algorithms(True) keeps
    the forward of 16-bit 64 x 64 states (and of blocks of them) on one kernel, whose bits depend on the row alone."""

    @staticmethod
    def forward(ctx, value, forget, query, key, f_key, state):
        """Return: (outputs [B,T,D], final state [B,D,K])"""
        need_grad = any(ctx.needs_input_grad)
        outputs, next_state, ckpt, C, flags, hints = _lfw_forward(value, forget, query, key, f_key, state, need_grad)
        if need_grad:
            ctx.save_for_backward(value, forget, query, key, f_key, state, ckpt)
            ctx.ckpt_interval = C
            ctx.flags = flags
            ctx.hints = hints
        return outputs, next_state

    @staticmethod
    def backward(ctx, grad_output, grad_state):
        value, forget, query, key, f_key, state, ckpt = ctx.saved_tensors
        return _lfw_backward(grad_output, grad_state, value, forget, query, key, f_key, state, ckpt,
                             ctx.ckpt_interval, ctx.flags, hints=ctx.hints)


def sigmoid_gates(f_logit, fk_logit, out_f=None, out_fk=None):
    """f = sigmoid(f_logit), f_key = sigmoid(fk_logit) in one launch (no autograd)."""
    for t, n in ((f_logit, "f_logit"), (fk_logit, "fk_logit")):
        _check_input(t, n)
    assert f_logit.dtype == fk_logit.dtype
    dev = f_logit.device
    with _on_device(dev):
        return _lib.host().gate_forward(f_logit, fk_logit, out_f, out_fk, _dtype_code(f_logit.dtype), _lib.current_stream(dev))


def _gate_backward_inplace(d_f, d_fk, forget, f_key):
    """d_f, d_fk: gate gradients on entry, logit gradients d_gate * gate * (1 - gate) on return."""
    dev = d_f.device
    with _on_device(dev):
        _lib.host().gate_backward(d_f, d_fk, forget, f_key, _dtype_code(d_f.dtype), _lib.current_stream(dev))


def _lfw_forward_logits(value, f_logit, query, key, fk_logit, state, need_grad, heads):
    """_lfw_forward on gate logits.  Where the call is an error, the gates come first, which may be one by themselves."""
    if _lib.loaded() and value.dtype != torch.float64 and _lib.host().lfw_shape(value, f_logit, query, key, fk_logit, state, heads) is not None:
        return _lfw_forward(value, f_logit, query, key, fk_logit, state, need_grad, heads, True)
    forget, f_key = sigmoid_gates(f_logit, fk_logit)
    return (*_lfw_forward(value, forget, query, key, f_key, state, need_grad, heads), forget, f_key)


class LFWGatedFunction(torch.autograd.Function):
    """``LFWFunction`` on gate *logits*: f = sigmoid(f_logit), f_key = sigmoid(fk_logit) are computed
    by one streaming kernel for both gates, the gates (not the logits) are kept for backward, and
    the gate gradients are turned into logit gradients in place by one more kernel.  The reference
    leaves the non-linearity to the caller (t2fw/functional_lfw.py:25-30), where it costs two
    elementwise passes forward and several backward, plus a second saved tensor per gate."""

    @staticmethod
    def forward(ctx, value, f_logit, query, key, fk_logit, state):
        assert value.shape == f_logit.shape and query.shape == fk_logit.shape
        assert f_logit.dtype == value.dtype and fk_logit.dtype == value.dtype
        need_grad = any(ctx.needs_input_grad)
        outputs, next_state, ckpt, C, flags, hints, forget, f_key = _lfw_forward_logits(value, f_logit, query, key, fk_logit, state, need_grad,
                                                                                        False)
        if need_grad:
            ctx.save_for_backward(value, forget, query, key, f_key, state, ckpt)
            ctx.ckpt_interval = C
            ctx.flags = flags
            ctx.hints = hints
        return outputs, next_state

    @staticmethod
    def backward(ctx, grad_output, grad_state):
        value, forget, query, key, f_key, state, ckpt = ctx.saved_tensors
        d_x, d_f, d_q, d_k, d_fk, d_s = _lfw_backward(grad_output, grad_state, value, forget, query, key, f_key,
                                                      state, ckpt, ctx.ckpt_interval, ctx.flags, hints=ctx.hints)
        _gate_backward_inplace(d_f, d_fk, forget, f_key)
        return d_x, d_f, d_q, d_k, d_fk, d_s


class LFWHeadsFunction(torch.autograd.Function):
    """The decay rule on tensors that keep the head axis next to the channels: x, f ``[B,T,H,D]``;
    q, k, f_key ``[B,T,H,K]``; state ``[B,H,D,K]``; returns outputs ``[B,T,H,D]`` and the final state
    ``[B,H,D,K]``.  Every (batch, head) pair is one recurrence.  The reference needs the folded,
    contiguous ``[B*H,T,D]`` layout (t2fw/csrc/lfw.cpp:24-26), i.e. ``transpose(1, 2).contiguous()``
    on five inputs and the inverse on the outputs and on six gradients; here the kernels stride
    over the head axis and those copies disappear.

    ``logits=True``: ``f`` and ``f_key`` are gate logits and the sigmoid is applied here (as in
    ``LFWGatedFunction``); the gradients returned for them are then logit gradients."""

    @staticmethod
    def forward(ctx, value, forget, query, key, f_key, state, logits=False):
        if logits:
            assert value.shape == forget.shape and query.shape == f_key.shape
            assert forget.dtype == value.dtype and f_key.dtype == value.dtype
        need_grad = any(ctx.needs_input_grad)
        if logits:
            outputs, next_state, ckpt, C, flags, hints, forget, f_key = _lfw_forward_logits(value, forget, query, key, f_key, state, need_grad,
                                                                                            True)
        else:
            outputs, next_state, ckpt, C, flags, hints = _lfw_forward(value, forget, query, key, f_key, state, need_grad, heads=True)
        if need_grad:
            ctx.save_for_backward(value, forget, query, key, f_key, state, ckpt)
            ctx.ckpt_interval = C
            ctx.flags = flags
            ctx.hints = hints
            ctx.logits = bool(logits)
        return outputs, next_state

    @staticmethod
    def backward(ctx, grad_output, grad_state):
        value, forget, query, key, f_key, state, ckpt = ctx.saved_tensors
        d_x, d_f, d_q, d_k, d_fk, d_s = _lfw_backward(grad_output, grad_state, value, forget, query, key, f_key,
                                                      state, ckpt, ctx.ckpt_interval, ctx.flags, heads=True,
                                                      hints=ctx.hints)
        if ctx.logits:
            _gate_backward_inplace(d_f, d_fk, forget, f_key)
        return d_x, d_f, d_q, d_k, d_fk, d_s, None


def _narrow_copies(tensors, dtype, stream):
    """``dtype`` copies of float32 tensors: one allocation, one launch."""
    dev = tensors[0].device
    offs, total = [], 0
    for t in tensors:
        offs.append(total)
        total += (t.numel() + 127) // 128 * 128          # every copy starts 256 bytes aligned
    buf = torch.empty(total, dtype=dtype, device=dev)
    outs = [buf[o:o + t.numel()].view(t.shape) for o, t in zip(offs, tensors)]
    _lib.cast_tensors(list(tensors), outs, stream)
    return outs


class LFW16Function(torch.autograd.Function):
    """The recurrence on float32 tensors through the 16-bit matrix-core kernels (see lfw_apply_16bit).  The
    16-bit copies of the inputs, not the float32 tensors, are what is kept for the backward."""

    @staticmethod
    def forward(ctx, value, forget, query, key, f_key, state, dtype):
        ins = (value, forget, query, key, f_key, state)
        for t, n in zip(ins, ("x", "f", "query", "key", "f_key", "state")):
            _check_input(t, n)
            if t.dtype != torch.float32:
                raise RuntimeError("t2fw: lfw_apply_16bit takes float32 tensors, %s is %s" % (n, t.dtype))
        need_grad = any(ctx.needs_input_grad)
        dev = value.device
        with _on_device(dev):
            stream = _lib.current_stream_handle(dev)
            narrow = _narrow_copies(ins, dtype, stream)
            out16, nxt16, ckpt, C, flags, hints = _lfw_forward(*narrow, need_grad)
            outputs, next_state = torch.empty_like(value), torch.empty_like(state)
            _lib.cast_tensors([out16, nxt16], [outputs, next_state], stream)
        if need_grad:
            ctx.save_for_backward(*narrow, ckpt)
            ctx.ckpt_interval, ctx.flags, ctx.hints, ctx.narrow = C, flags, hints, dtype
        return outputs, next_state

    @staticmethod
    def backward(ctx, grad_output, grad_state):
        *narrow, ckpt = ctx.saved_tensors
        dev = grad_output.device
        with _on_device(dev):
            stream = _lib.current_stream_handle(dev)
            go16, gs16 = _narrow_copies((grad_output.contiguous().float(), grad_state.contiguous().float()), ctx.narrow, stream)
            grads16 = _lfw_backward(go16, gs16, *narrow, ckpt, ctx.ckpt_interval, ctx.flags, hints=ctx.hints)
            grads = [torch.empty(g.shape, dtype=torch.float32, device=dev) for g in grads16]
            _lib.cast_tensors(list(grads16), grads, stream)
        return (*grads, None)


def lfw_apply_16bit(value, forget, query, key, f_key, state, dtype=torch.float16):
    """``LFWFunction.apply`` for float32 tensors at the speed of the 16-bit matrix-core kernels: the six
    inputs are converted to ``dtype`` (float16 or bfloat16) in one launch, the recurrence and its backward
    run in that type, outputs and gradients come back as float32.  An explicit choice of the caller: the
    results carry the 16-bit kernels' accuracy (within 1e-2 of max|ref| per tensor; gates are rounded to
    ``dtype`` before they are multiplied up, 2^-11 relative per step in float16, so bfloat16 is for short
    memories only), where ``LFWFunction.apply`` on float32 tensors runs the exact kernels.  The reference
    has one kernel for every dtype (t2fw/csrc/lfw_kernel.cu:157-168) and no counterpart of this."""
    assert dtype in (torch.float16, torch.bfloat16)
    return LFW16Function.apply(value, forget, query, key, f_key, state, dtype)


def lfw_apply_padded(value, forget, query, key, f_key, state):
    """``LFWFunction.apply`` for fp16 / bf16 tensors whose value or key width is not a multiple of 64, on the
    matrix-core kernels: the widths are padded up to the next multiple of 64 (values, keys, queries and the state
    with zeros, gates with ones -- the padded channels stay zero and add nothing), the padded tensors run as
    64 x 64 blocks (``LFWFunction.apply`` does that by itself for multiples of 64), and the results are cut back.
    Correct for any width, and as expensive as the padded width: a 32 x 32 state costs what a 64 x 64 one costs
    (forward + backward at B=96, T=1024: 201 us of GPU time where the exact kernels take 278; 33 x 17: 207 and
    414).  An explicit choice of the caller, because the results carry the matrix-core kernels' accuracy where ``LFWFunction.apply`` runs the exact
    kernels for such widths.  Padding, cutting and their gradients are plain tensor operations."""
    assert value.dtype in (torch.float16, torch.bfloat16), "the matrix-core kernels take fp16 / bf16 tensors"
    assert value.shape == forget.shape and query.shape == key.shape and query.shape == f_key.shape
    B, T, D = value.shape
    K = query.shape[2]
    assert tuple(state.shape) == (B, D, K)
    Dp, Kp = 64 * -(-D // 64), 64 * -(-K // 64)
    if Dp == D and Kp == K:
        return LFWFunction.apply(value, forget, query, key, f_key, state)
    pad = torch.nn.functional.pad
    out, nxt = LFWFunction.apply(pad(value, (0, Dp - D)), pad(forget, (0, Dp - D), value=1.0), pad(query, (0, Kp - K)),
                                 pad(key, (0, Kp - K)), pad(f_key, (0, Kp - K), value=1.0),
                                 pad(state, (0, Kp - K, 0, Dp - D)))
    return out[..., :D].contiguous(), nxt[:, :D, :K].contiguous()


def lfw_step(x, f, query, key, f_key, state, out=None, inplace=True):
    """One generation step (T = 1) without autograd: x,f [B,D]; query,key,f_key [B,K];
    state [B,D,K] updated in place when ``inplace``.  Returns (out [B,D], state).
    The reference does this through the T=1 forward (tests/benchmark.py:104-105), which
    allocates a new state tensor per step."""
    if _lib.loaded() and x.is_cuda:
        with _on_device(x.device):
            done = _lib.host().lfw_step(x, f, query, key, f_key, state, out, bool(inplace), _lib.current_stream(x.device))
        if done is not None:
            return done
    # which error it is, or what the step above leaves to the caller
    for t, n in ((x, "x"), (f, "f"), (query, "query"), (key, "key"), (f_key, "f_key"), (state, "state")):
        _check_input(t, n)
        assert t.dtype == x.dtype
    B, D = x.shape
    K = query.shape[1]
    assert tuple(state.shape) == (B, D, K) and f.shape == x.shape
    assert key.shape == query.shape and f_key.shape == query.shape
    lib = _lib.load()
    dev = x.device
    with _on_device(dev):
        if out is None:
            out = torch.empty_like(x)
        nxt = state if inplace else torch.empty_like(state)
        _lib.check(lib.t2fw_lfw_step(
            _lib.ptr(x), _lib.ptr(f), _lib.ptr(query), _lib.ptr(key), _lib.ptr(f_key), _lib.ptr(state),
            _lib.ptr(out), _lib.ptr(nxt), B, D, K, _dtype_code(x.dtype), _lib.current_stream_handle(dev)))
    return out, nxt
