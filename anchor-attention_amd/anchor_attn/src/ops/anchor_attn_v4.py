"""The AnchorAttention prefill operator on MI355X.

Same entry points, argument meaning, assertions and return arity as the reference's
``anchor_attn/src/ops/anchor_attn_v4.py`` (``anchor_attn`` :291-324, ``anchor_attn_test_time``
:328-354, ``anchor_attn_without_anchor`` :275-289); the three stages underneath are hand-written
gfx950 kernels reached through the C ABI in ``include/anchor_attn_hip.h``.

Beyond the reference: K and V may be passed with their native (un-repeated) KV heads, any
``[B,H,N,D]`` view with unit last stride is taken without a copy, and ``out`` may be supplied.
There is no CPU or eager fallback - tensors must be bf16 (or fp16, which the reference's kernels also take) on the GPU.
"""
from __future__ import annotations

import ctypes
import threading
import time

import my_utils
import torch

from . import _hip
from .anchor_step_1_2_v2 import (_check_inputs, _row_major, _stream, anchor_attn_step_1,
                                 select_stripes_packed)

LOG2E = 1.44269504


def _ratio_denominator(B, H, N, block_size, step):
    return B * H * N * N / (block_size * step) // 2


def _ratio(true_counts, B, H, N, block_size, step):
    # same expression as the reference (anchor_attn_v4.py:271); stays a 0-dim device tensor
    denominator = _ratio_denominator(B, H, N, block_size, step)
    if torch.get_default_dtype() != torch.float32 or not true_counts.is_contiguous():
        return true_counts.sum() / denominator  # (the quotient of whole numbers has the default type)
    ratio = torch.empty((), dtype=torch.float32, device=true_counts.device)
    _hip.check(_hip.lib().aa_sparsity_ratio(true_counts.data_ptr(), true_counts.numel(), denominator, ratio.data_ptr(), _stream()))
    return ratio


_UNSET = -1.0
_host_ratios = threading.local()
_left_words, _left_lock = [], threading.Lock()


def _host_ratio(device):
    """This thread's word of pinned host memory for ratios of calls on ``device``, unset; None if the ratio of a call cannot be
    waited for.  One word is enough: a call that uses it returns when the GPU has written it, or leaves it (:func:`_leave_host_ratio`)."""
    if not (my_utils.Logger.enabled and device.type == "cuda" and torch.get_default_dtype() == torch.float32) or torch.cuda.is_current_stream_capturing():
        return None
    words = _host_ratios.__dict__
    word = words.get(str(device))
    if word is None:
        tensor = torch.empty((), dtype=torch.float32, pin_memory=True)
        word = words[str(device)] = (tensor, ctypes.c_float.from_address(tensor.data_ptr()))
    word[1].value = _UNSET
    return word[1]


def _leave_host_ratio(device):
    """After a call that ended early, with its launch perhaps on the way: what that still stores is not the next call's, which gets
    another word.  This one is kept until the stream has come to here."""
    word, done = _host_ratios.__dict__.pop(str(device)), torch.cuda.Event()
    with _left_lock:
        done.record(torch.cuda.current_stream(device))
        _left_words[:] = [left for left in _left_words if not left[1].query()] + [(word, done)]


def _log_ratio(sparse_ratio, host_ratio=None):
    """The reference logs the ratio on every call (anchor_attn_v4.py:321-323).  Formatting the 0-dim device tensor
    copies it to the host, i.e. waits for the whole operator; a ``host_ratio`` that the operator was given is there as soon as
    stage 2 is done (a single big block: when its first rows are), and the call returns while the GPU is at work.  Calls in a row: 2048 tokens, 14/2
    heads of 64 63 us each against 28; 4096 tokens, 32/8 heads of 128 190 against 165.  (One call until its output is complete gains less
    from it: with all the steps that this was one of 81 -> 50 and 218 -> 187.)"""
    text = None

    def message():
        nonlocal text
        there = host_ratio is not None and _hip.lib().aa_wait_ratio(ctypes.addressof(host_ratio), _UNSET, 100000)
        text = f"anchor sparse_ratio:{host_ratio.value if there else sparse_ratio}"
        return text
    log = my_utils.Logger.log
    try:
        if my_utils.Logger.enabled:
            # (the own logger opens its file first, while the GPU works; one that a program put in its place is given the line)
            log(message if getattr(log, "takes_function", False) else message())
    finally:
        if text is None and host_ratio is not None:  # (not written: the GPU still has to have stored the word before the next call uses it)
            message()


def _workspace(B, H, N, D, block_size, step, device):
    nbytes = _hip.lib().aa_workspace_bytes(B, H, N, D, block_size, step)
    if nbytes == 0:
        raise _hip.AnchorAttnHipError(f"unsupported problem shape B={B} H={H} N={N} D={D} block_size={block_size} step={step}")
    return torch.empty((nbytes,), dtype=torch.uint8, device=device)


def _anchor_attn(Q, K, V, sm_scale=None, block_size=64, step=16, difference=100, return_sparsity_ratio=False,
                 BLOCK_SIZE_M=128, BLOCK_SIZE_N=128, out=None, scale_mode=_hip.AA_SCALE_BF16_CHAIN,
                 geometry=_hip.AA_GEOMETRY_AS_RUN, host_ratio=None, rows=None):
    """All three stages on the current stream, one C call (``difference`` is in the log2 domain
    here, as in the reference's private function, anchor_attn_v4.py:226-273)."""
    B, H, N, D = Q.shape
    assert N % block_size == 0
    assert block_size in [16, 32, 64, 128, 256], "BLOCK_SIZE must be a power of 2 and ≥16"  # get_mask_test.py:133
    _check_inputs(Q, K, V)
    output = torch.empty_like(Q) if out is None else out
    assert output.shape == Q.shape and output.dtype == Q.dtype and output.stride(-1) == 1
    sizes = (B, H, K.shape[1], N, D, block_size, step)
    if rows is None:
        ws, beside = _workspace(B, H, N, D, block_size, step, Q.device), ()
    else:
        problem, row_tensors, row_sizes, row_scale = rows
        assert problem == (B, H, K.shape[1], D, Q.dtype), "rows beside the operator have its batch, heads, head dimension and type"
        nbytes = _hip.lib().aa_anchor_attn_rows_workspace_bytes(*sizes, *row_sizes)
        ws, beside = torch.empty((nbytes,), dtype=torch.uint8, device=Q.device), (*row_tensors, *row_sizes, row_scale)
    tensors = (*_hip.t3(Q), *_hip.t3(K), *_hip.t3(V), *_hip.t3(output), *beside, ws.data_ptr(), ws.numel())
    options = (*sizes, float(sm_scale), float(difference), scale_mode, int(geometry), _hip.dtype_code(Q), _stream())
    counts = ratio = None
    if return_sparsity_ratio and torch.get_default_dtype() == torch.float32:
        ratio = torch.empty((), dtype=torch.float32, device=Q.device)
    elif return_sparsity_ratio:
        counts = torch.empty((B, H, N // (block_size * step), 1), dtype=torch.int32, device=Q.device)
    counts_ptr = counts.data_ptr() if counts is not None else None
    ratio_args = (None, None, 1.0)
    if ratio is not None:
        ratio_args = (ratio.data_ptr(), ctypes.addressof(host_ratio) if host_ratio is not None else None, _ratio_denominator(B, H, N, block_size, step))
    if rows is not None:
        _hip.check(_hip.lib().aa_anchor_attn_rows_fwd(*tensors, counts_ptr, *ratio_args, *options))
    elif ratio is not None:
        _hip.check(_hip.lib().aa_anchor_attn_ratio_fwd(*tensors, *ratio_args, *options))
    else:
        _hip.check(_hip.lib().aa_anchor_attn_fwd(*tensors, counts_ptr, *options))
    if counts is not None:
        ratio = _ratio(counts, B, H, N, block_size, step)
    return output, ratio if return_sparsity_ratio else 1.0


def _stage3(Q, K, V, coords, counts, L, M, Acc, sm_scale, block_size, step, out=None):
    B, H, N, D = Q.shape
    output = torch.empty_like(Q) if out is None else out
    _hip.check(_hip.lib().aa_stage3_sparse_fwd(
        *_hip.t3(Q), *_hip.t3(K), *_hip.t3(V), coords.data_ptr(), counts.data_ptr(),
        M.data_ptr(), L.data_ptr(), Acc.data_ptr(), *_hip.t3(output),
        B, H, K.shape[1], N, D, block_size, step, float(sm_scale), _hip.dtype_code(Q), _stream()))
    return output


def _anchor_attn_staged(Q, K, V, sm_scale, block_size, step, difference, timed):
    B, H, N, D = Q.shape
    assert N % block_size == 0
    _check_inputs(Q, K, V)
    if timed:
        torch.cuda.synchronize()
        t0 = time.time()
    L, M, Acc = anchor_attn_step_1(Q, K, V, 1, 1, block_size, step, B, H, N, D, sm_scale)
    coords, counts = select_stripes_packed(Q, K, M, block_size, step, difference, B, H, N, D, sm_scale)
    if timed:
        torch.cuda.synchronize()
        t1 = time.time()
    output = _stage3(Q, K, V, coords, counts, L, M, Acc, sm_scale, block_size, step)
    if timed:
        torch.cuda.synchronize()
        t2 = time.time()
        return output, counts, (t1 - t0) * 1000, (t2 - t1) * 1000
    return output, counts, None, None


def _prepare(Q, K, V):
    return _row_major(Q), _row_major(K), _row_major(V)


def anchor_attn_without_anchor(Q, K, V, sm_scale: float = None, block_size: int = 128, step: int = 16,
                               difference: float = 12):
    difference *= LOG2E
    Q, K, V = _prepare(Q, K, V)
    assert Q.size(-2) % block_size == 0
    B, H, N, D = Q.shape
    sm_scale = sm_scale if sm_scale else 1.0 / (D ** 0.5)
    output, counts, _, _ = _anchor_attn_staged(Q, K, V, sm_scale, block_size, step, difference, timed=False)
    return output, _ratio(counts, B, H, N, block_size, step)


def anchor_attn(Q, K, V, sm_scale: float = None, block_size: int = 128, step: int = 16, difference: float = 12,
                return_computational_ratio: bool = True, out: torch.Tensor = None, strict_reference: bool = True, rows=None):
    """Sparse prefill attention.  ``Q`` ``[B,H,N,D]`` bf16 or fp16; ``K``/``V`` ``[B,H or H_kv,N,D]`` of the same type;
    returns ``out`` or ``(out, ratio)`` exactly like the reference.

    ``strict_reference=False`` (analysis only, never the default) lets stage 2 choose from ``[S, bb*S)``
    - the range of the reference's fused variant, anchor_fuse_step_1_2_v2.py:152 - instead of the as-run
    ``[block_size, bb*S - block_size)``: no key is attended twice and none is left out.

    With the ratio, a call waits for that number where the logger is on, and not for the output, which is ordered by the stream like any
    GPU result.

    ``rows``: dense attention of other rows that is computed with the operator's first launch (:func:`rows_beside`)."""
    difference *= LOG2E
    Q, K, V = _prepare(Q, K, V)
    assert Q.stride(-1) == 1 and K.stride(-1) == 1 and V.stride(-1) == 1, \
        "Q, K, V must be contiguous. Please call .contiguous() before passing."

    assert step in [16, 32], \
        f"Invalid step size: {step}. Only step sizes 16 or 32 are supported."

    assert Q.size(-2) % (block_size * step) == 0, \
        f"Sequence length {Q.size(-2)} must be divisible by (block_size * step = {block_size * step})."

    B, H, N, D = Q.shape
    sm_scale = sm_scale if sm_scale else 1.0 / (D ** 0.5)
    host_ratio = _host_ratio(Q.device) if return_computational_ratio else None
    try:
        sparse_output, sparse_ratio = _anchor_attn(Q, K, V, sm_scale, block_size, step, difference,
                                                   return_computational_ratio, out=out, host_ratio=host_ratio, rows=rows,
                                                   geometry=_hip.AA_GEOMETRY_AS_RUN if strict_reference else _hip.AA_GEOMETRY_INTENDED)
        if return_computational_ratio:
            _log_ratio(sparse_ratio, host_ratio)
            return sparse_output, sparse_ratio
        return sparse_output
    except BaseException:  # (an interrupt among them)
        if host_ratio is not None:
            _leave_host_ratio(Q.device)
        raise


def anchor_attn_test_time(Q, K, V, sm_scale: float = None, block_size: int = 128, step: int = 16,
                          difference: float = 12, return_computational_ratio: bool = True):
    """Same result as :func:`anchor_attn` plus the wall-clock of (stage 1 + stage 2) and of stage 3
    in milliseconds, each bracketed by device synchronisation (anchor_attn_v4.py:107-169)."""
    difference *= LOG2E
    Q, K, V = _prepare(Q, K, V)
    assert Q.size(-2) % block_size == 0
    B, H, N, D = Q.shape
    sm_scale = sm_scale if sm_scale else 1.0 / (D ** 0.5)
    output, counts, search_time, compute_time = _anchor_attn_staged(Q, K, V, sm_scale, block_size, step, difference, timed=True)
    if return_computational_ratio:
        sparse_ratio = _ratio(counts, B, H, N, block_size, step)
        _log_ratio(sparse_ratio)
        return output, sparse_ratio, search_time, compute_time
    return output, search_time, compute_time


def _function_modes():
    """The ``TorchFunctionMode`` stack without ``torch.device(...)`` blocks, which only concern factory functions."""
    return [m for m in torch.overrides._get_current_function_mode_stack() if type(m) is not torch.utils._device.DeviceContext]


def _called_plainly() -> bool:
    """False while something other than eager execution watches the operations (vmap, forward-mode differentiation, tracing,
    compilation, a dispatch or function mode): it would not see what happens behind the C interface.  The framework has no
    public names for most of these; a release in which they have moved counts as watched."""
    try:
        return (not torch.compiler.is_compiling() and torch._C._functorch.peek_interpreter_stack() is None
                and torch.autograd.forward_ad._current_level < 0 and not torch.jit.is_tracing()
                and torch._C._len_torch_dispatch_stack() == 0
                and (torch._C._len_torch_function_stack() == 0 or not _function_modes()))
    except AttributeError:
        return False


def _no_backend_chosen() -> bool:
    """Whether all of library attention's backends are allowed: who rules one out (``torch.nn.attention.sdpa_kernel``,
    ``torch.backends.cuda.enable_*_sdp``) has chosen what computes the attention."""
    return torch.backends.cuda.flash_sdp_enabled() and torch.backends.cuda.mem_efficient_sdp_enabled() and torch.backends.cuda.math_sdp_enabled()


def _rows_tensors(Q, K, V, mask=None, out=None):
    """``data_ptr, stride_b, stride_h, stride_n`` of ``Q``, ``K``, ``V`` and ``out`` (not given: ``Q``'s) for the launch; None
    where the kernels do not take them: their types, head dimensions, alignment, sizes of one launch and 32-bit addressing
    of one head.  All of them hold for ``out`` too, whose strides can be wider than ``Q``'s."""
    dtype, device, q_shape, kv_shape = Q.dtype, Q.device, Q.shape, K.shape
    if not (Q.is_cuda and dtype in (torch.bfloat16, torch.float16) and K.dtype == V.dtype == dtype and K.device == V.device == device):
        return None
    if not (len(q_shape) == len(kv_shape) == 4 and V.shape == kv_shape):
        return None
    B, H, N, D = q_shape
    kv_batch, kv_heads, n_keys, kv_dim = kv_shape
    if D not in (64, 128) or kv_dim != D or kv_batch != B or not B or not kv_heads or H % kv_heads or not H:
        return None
    if out is None:
        out = Q
    elif out.shape != q_shape or out.dtype != dtype or out.device != device:
        return None
    tensors = []
    for t, rows in ((Q, N), (K, n_keys), (V, n_keys), (out, N)):
        ptr, (sb, sh, sn, sd) = t.data_ptr(), t.stride()
        if sd != 1 or (sb | sh | sn) & 7 or ptr & 15 or not D <= sn <= 1 << 14 or not 0 < rows <= 1 << 20 or rows * sn * 2 >= 1 << 32:
            return None
        tensors += (ptr, sb, sh, sn)
    col_blocks = (N * (H // kv_heads) + 127) // 128
    # (that many column blocks are one chunk each; but a decode step's chunk holds 2^13 keys, a masked one 2^16)
    if B * kv_heads * col_blocks * (1 if col_blocks > 1 and mask is None else (n_keys >> 13) + 1) >= 1 << 24:
        return None
    if mask is not None:
        if type(mask) is not torch.Tensor or mask.device != device or mask.dtype != torch.bool or mask.dim() != 4:
            return None
        if mask.shape[0] not in (1, B) or tuple(mask.shape[1:]) != (1, N, n_keys):
            return None
        if B >= 1 << 16 or col_blocks >= 1 << 16 or N * ((n_keys + 63) // 64) * 8 >= 1 << 32:
            return None
    return tensors


def _rows_dispatch(Q, K, V, mask=None, out=None):
    """:func:`_rows_tensors` where the attention of these tensors is to be computed by the own kernels: they take them, and
    nothing about the call asks for the framework's own operations; otherwise None."""
    if not (type(Q) is type(K) is type(V) is torch.Tensor and _called_plainly() and _no_backend_chosen()):
        return None
    if torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") != Q.dtype:  # (attention is computed in that type)
        return None
    # Thousands of padded prompts of a few tokens: a work-group per (prompt, KV head) has one tile to do, and library attention, where it
    # need not repeat heads, is faster: 128 prompts of 16 tokens, 32 heads of 128, 37 us against 64 (32 tokens 68 against 71; 16 prompts 36
    # against 28; 32/8 heads 241 against 30).
    if mask is not None and 1 < Q.shape[2] and K.shape[2] < 32 and Q.shape[1] == K.shape[1] and Q.shape[0] * Q.shape[1] > 2048:
        return None
    return _rows_tensors(Q, K, V, mask, out)


def dense_rows_supported(Q, K, V, mask=None, out=None) -> bool:
    """Whether the attention of these tensors is to be computed by :func:`dense_rows_attention`."""
    return _rows_dispatch(Q, K, V, mask, out) is not None


def dense_rows_attention(Q, K, V, causal_offset: int = 0, sm_scale: float = None, out: torch.Tensor = None, mask: torch.Tensor = None):
    """Attention of ``Q`` ``[B,H,n_rows,D]`` over ``K``/``V`` ``[B,H_kv,n_keys,D]`` on the same MFMA core: query row ``i``
    sees keys ``0 .. causal_offset + i``, or, with a boolean ``mask`` ``[B or 1, 1, n_rows, n_keys]``, the keys it is True for.
    Any row and key count (:func:`_rows_tensors` names the rest)."""
    tensors = _rows_tensors(Q, K, V, mask, out)
    if tensors is None:
        raise _hip.AnchorAttnHipError("dense_rows_attention: unsupported tensors (bf16 or fp16 on one GPU, head dimension 64 or 128, rows of at "
                                      "most 16384 elements on 16-byte boundaries, a boolean mask [B or 1, 1, n_rows, n_keys], out like Q)")
    return _dense_rows(tensors, Q, K, causal_offset, sm_scale, out, mask)


def rows_beside(tensors, Q, K, causal_offset, sm_scale):
    """``rows`` of :func:`anchor_attn` for the attention that ``_dense_rows`` computes of the same arguments (``tensors`` with ``out``)."""
    B, H, N, D = Q.shape
    return (B, H, K.shape[1], D, Q.dtype), tensors, (N, K.shape[2], int(causal_offset)), float(sm_scale if sm_scale else 1.0 / (D ** 0.5))


def _dense_rows(tensors, Q, K, causal_offset, sm_scale, out, mask):
    # (`tensors` comes from _rows_tensors for this very call, which has looked at them: the launch trusts their shapes)
    B, H, N, D = Q.shape
    _, kv_heads, n_keys, _ = K.shape
    sm_scale = sm_scale if sm_scale else 1.0 / (D ** 0.5)
    output = out
    if out is None:
        output = torch.empty_like(Q)
        tensors[12:] = _hip.t3(output)
    mask_args = (None, 0, 0)
    if mask is not None:
        mask = mask if mask.stride(3) == 1 else mask.contiguous()
        mask_args = (mask.data_ptr(), mask.stride(0) if mask.shape[0] > 1 else 0, mask.stride(2))
    lib = _hip.lib()
    sizes = (B, H, kv_heads, N, n_keys, D, int(causal_offset))
    dtype = _hip.dtype_code(Q)
    nbytes = lib.aa_dense_rows_workspace_bytes_of(*sizes, mask is not None, dtype)
    ws = torch.empty((nbytes,), dtype=torch.uint8, device=Q.device) if nbytes else None
    args = (*tensors, *mask_args, ws.data_ptr() if nbytes else None, nbytes, *sizes, float(sm_scale), dtype)
    if Q.device.index == torch.cuda.current_device():
        _hip.check(lib.aa_dense_rows_fwd(*args, _stream()))
    else:  # (a pipeline's later layers lie on other GPUs than the current one)
        with torch.cuda.device(Q.device):
            _hip.check(lib.aa_dense_rows_fwd(*args, _stream()))
    return output


def dense_causal_attention(Q, K, V, sm_scale: float = None, out: torch.Tensor = None):
    """Plain causal attention on the same MFMA core (the dense baseline the sparse operator is
    compared with; GQA-aware like the reference's flash_attn_triton.py:129-132)."""
    Q, K, V = _prepare(Q, K, V)
    _check_inputs(Q, K, V)
    B, H, N, D = Q.shape
    sm_scale = sm_scale if sm_scale else 1.0 / (D ** 0.5)
    output = torch.empty_like(Q) if out is None else out
    _hip.check(_hip.lib().aa_dense_causal_fwd(*_hip.t3(Q), *_hip.t3(K), *_hip.t3(V), *_hip.t3(output),
                                              B, H, K.shape[1], N, D, float(sm_scale), _hip.dtype_code(Q), _stream()))
    return output
