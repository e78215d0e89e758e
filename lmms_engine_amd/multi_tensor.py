"""Device-side description of a list of tensors for the multi-tensor kernels of libmuon_hip.

One pinned host buffer holds, as int64 words, the base pointers of every tensor role (one row
per role: parameters, grads, ...), the element counts, the first-chunk index of every tensor
(n + 1 entries) and any per-tensor doubles (bit patterns); one asynchronous copy puts it on
the device.  The layout is the one include/muon_hip.h documents for muon_hip_adamw_multi,
muon_hip_grad_norms and muon_hip_clip_scale.
"""
from __future__ import annotations

from array import array
from typing import Sequence

import torch
from torch import Tensor

from . import _abi


def _reject(t: Tensor, first: Tensor, numel: int) -> None:
    if not t.is_cuda:
        raise _abi.MuonHipError(f"tensors must live on a GPU: this build has no CPU path (got {t.device})")
    if t.device != first.device or t.dtype != first.dtype or t.numel() != numel:
        raise ValueError("a tensor list holds tensors of one device and dtype; roles must match in size")
    raise NotImplementedError("multi-tensor kernels need contiguous tensors")


class TensorListTable:
    def __init__(self, roles: Sequence[Sequence[Tensor]], doubles: Sequence[Sequence[float]] = ()):
        n = len(roles[0])
        assert n > 0 and all(len(r) == n for r in roles) and all(len(d) == n for d in doubles)
        first = roles[0][0]
        index, dtype = first.get_device(), first.dtype  # -1 for a tensor that is not on a GPU
        numel = [t.numel() for t in roles[0]]
        for r in roles:
            for t, ne in zip(r, numel):
                if index < 0 or t.get_device() != index or t.dtype != dtype or t.numel() != ne or not t.is_contiguous():
                    _reject(t, first, ne)
        self.n = n
        self.device = first.device
        self.dtype = dtype
        starts = [0]
        at = 0
        for ne in numel:
            at += (ne + _abi.MULTI_CHUNK - 1) // _abi.MULTI_CHUNK
            starts.append(at)
        self.chunks = at
        words = array("q")
        for r in roles:
            words.extend([t.data_ptr() for t in r])
        words.extend(numel)
        words.extend(starts)
        self._put(bytearray(words.tobytes()), len(roles), doubles)
        self._keep += ([list(r) for r in roles],)  # the tensors stay alive while kernels may read them

    @classmethod
    def of_words(cls, words: bytearray, roles: int, n: int, chunks: int, device, dtype, doubles: Sequence[Sequence[float]] = ()):
        """A table whose rows `_abi.scan()` has put together: pointers of `roles` roles, element counts, first chunks."""
        self = cls.__new__(cls)
        self.n, self.chunks, self.device, self.dtype = n, chunks, device, dtype
        self._put(words, roles, doubles)
        return self

    def _put(self, words: bytearray, k: int, doubles) -> None:
        n = self.n
        for d in doubles:
            words += array("d", d).tobytes()
        host = torch.empty(len(words) // 8, dtype=torch.int64, pin_memory=True)
        host.copy_(torch.frombuffer(words, dtype=torch.int64))
        self.table = host.to(self.device, non_blocking=True)
        self._keep = (host,)
        base = self.table.data_ptr()
        self.role_ptrs = [base + 8 * n * i for i in range(k)]
        self.numel_ptr = base + 8 * n * k
        self.chunk_start_ptr = self.numel_ptr + 8 * n
        self.double_ptrs = [self.chunk_start_ptr + 8 * (n + 1) + 8 * n * i for i in range(len(doubles))]
