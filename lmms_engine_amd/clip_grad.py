"""Gradient-norm clipping on one GPU, the call that precedes `optimizer.step()`.

Mirror of `fsdp2_clip_grad_norm_` (src/lmms_engine/utils/fsdp2_utils.py:234-255) when no process
group is active: torch's `_get_total_norm` followed by `_clip_grads_with_norm_`.  The norm of every
gradient, the norm of those norms and the in-place scaling each run as one multi-tensor kernel per
dtype; nothing synchronises the host unless `error_if_nonfinite` asks for the value.
"""
from __future__ import annotations

from collections import OrderedDict

import torch
from torch import Tensor

from . import _abi
from .multi_tensor import TensorListTable


@torch.no_grad()
def clip_grad_norm_(parameters, max_norm, norm_type=2.0, error_if_nonfinite=False, foreach=None) -> Tensor:
    """Same signature and return value (the total norm, a 0-d tensor on the gradients' device) as
    fsdp2_clip_grad_norm_.  `norm_type` is any order torch.linalg.vector_norm takes: 2 (the default), 1, 0, inf and
    -inf have reductions of their own, every other p is (sum |x|^p)^(1/p) accumulated in fp32 as torch does.
    `foreach` is accepted and ignored (every call is one launch per dtype)."""
    if isinstance(parameters, Tensor):
        parameters = [parameters]
    else:
        parameters = list(parameters)
    norm_type = float(norm_type)
    if norm_type != norm_type:
        raise ValueError("norm_type is NaN")
    held = []  # the gradients' memory, until this call has launched everything
    plain = _abi.scan().grads(parameters, _abi.MULTI_CHUNK, held)
    if plain is not None:
        index, lists = plain
        dev = torch.device("cuda", index)
        return _clip(dev, sum(n for _, n, _, _ in lists), [code for code, *_ in lists],
                     lambda: [TensorListTable.of_words(words, 1, n, chunks, dev, _abi.DTYPES[code]) for code, n, chunks, words in lists],
                     max_norm, norm_type, error_if_nonfinite)
    grads = [g for g in [p.grad for p in parameters] if g is not None]
    if len(grads) == 0:
        return torch.tensor(0.0)  # what _get_total_norm returns for an empty list
    for g in grads:
        if not g.is_cuda:
            raise _abi.MuonHipError(f"gradients must live on a GPU: this build has no CPU path (got {g.device})")
    dev, index = grads[0].device, grads[0].get_device()
    groups: "OrderedDict[torch.dtype, list]" = OrderedDict()
    strided = []  # gradients with other than row-major strides are scaled through a row-major copy that is written back
    for g in grads:
        if g.get_device() != index:
            raise NotImplementedError("gradients on several devices")
        c = g
        if not g.is_contiguous():
            c = g.contiguous()
            strided.append((g, c))
        same = groups.get(g.dtype)
        if same is None:
            same = groups[g.dtype] = []
        same.append(c)
    total = _clip(dev, len(grads), [_abi.dtype_code(dt) for dt in groups], lambda: [TensorListTable([gs]) for gs in groups.values()], max_norm,
                  norm_type, error_if_nonfinite)
    for g, c in strided:
        g.copy_(c)
    return total


def _clip(dev, n_total, codes, make_tables, max_norm, norm_type, error_if_nonfinite) -> Tensor:
    """The norm of the lists that make_tables() describes, one per dtype code, and their scaling."""
    lib = _abi.lib()
    # torch stacks the per-tensor norms of all dtype groups; stacking promotes, so the total has the widest dtype
    out_dtype = torch.float32 if _abi.F32 in codes else torch.bfloat16
    with torch.cuda.device(dev):
        s = _abi.stream_ptr(dev)
        norms = torch.empty(n_total, dtype=torch.float32, device=dev)
        total_f32 = torch.empty(1, dtype=torch.float32, device=dev)
        total = torch.empty((), dtype=out_dtype, device=dev)
        tables, off = make_tables(), 0
        for code, tab in zip(codes, tables):
            if tab.chunks > 0:
                partials = torch.empty(tab.chunks, dtype=torch.float32, device=dev)
                _abi.check(lib.muon_hip_grad_norms(tab.role_ptrs[0], tab.numel_ptr, tab.chunk_start_ptr, tab.n, tab.chunks,
                                                   code, norm_type, partials.data_ptr(), norms.data_ptr() + 4 * off, s),
                           "grad_norms")
            else:
                norms[off:off + tab.n].zero_()
            off += tab.n
        _abi.check(lib.muon_hip_total_norm(norms.data_ptr(), n_total, _abi.dtype_code(out_dtype), norm_type, total_f32.data_ptr(),
                                           total.data_ptr(), s), "total_norm")
        if error_if_nonfinite and not bool(torch.isfinite(total)):
            raise RuntimeError(
                f"The total norm of order {norm_type} for gradients from `parameters` is non-finite, so it "
                "cannot be clipped. To disable this error and scale the gradients by the non-finite norm anyway, "
                "set `error_if_nonfinite=False`")
        for code, tab in zip(codes, tables):
            if tab.chunks > 0:
                _abi.check(lib.muon_hip_clip_scale(tab.role_ptrs[0], tab.numel_ptr, tab.chunk_start_ptr, tab.n, tab.chunks,
                                                   code, total_f32.data_ptr(), _abi.dtype_code(out_dtype),
                                                   float(max_norm), s), "clip_scale")
    return total


fsdp2_clip_grad_norm_ = clip_grad_norm_
