"""Python face of the fused GroupGEMM launch: device pointer tables + one C-ABI call per launch.

Host-side counterpart of `moe_mxmoe_share_fused` (mxmoe/kernels/src/ref_bind.cu:312-431): it builds the same
five pointer arrays, the problem sizes and the QParams list, but once, into one device buffer that is reused by
every launch (the reference re-allocates and re-copies them on every call, ref_bind.cu:395-404,426-428).
"""
from __future__ import annotations

import ctypes as C
import struct
from array import array
from functools import lru_cache

import numpy as np
import torch

from . import _lib
from .weights import PackedWeight  # noqa: F401  (re-export for callers)


@lru_cache(maxsize=256)
def _qparams_bytes(q: tuple) -> bytes:
    a, w, g, s = q
    return struct.pack("=4i", int(a), int(w), int(g), 1 if s else 0)  # (a_bits, w_bits, gsize, sym byte): the QParams layout


@lru_cache(maxsize=256)
def _array_types(p: int):
    return _lib.Dim3 * p, _lib.QParams * p


def _upload(host: np.ndarray, device) -> torch.Tensor:
    """`host` (contiguous) as a device tensor of bytes.  The bytes travel in kernel arguments (mxmoe_upload): unlike a copy from pageable
    memory, which first waits for everything enqueued on the stream, the host goes on at once."""
    d = torch.empty(max(host.nbytes, 8), dtype=torch.uint8, device=device)
    lib = _lib.load()
    _lib.check(lib, lib.mxmoe_upload(d.data_ptr(), host.ctypes.data, host.nbytes, _lib.current_stream()))
    return d


class GroupGemmLaunch:
    """A prepared problem list: `run()` is a single allocation-free, sync-free kernel launch."""

    def __init__(self, As, Bs, scale_a, scale_b, Cs, sizes, qparams, kernel_id: int = -1, acc=None, lib=None):
        self.lib = lib or _lib.load()
        p = len(As)
        assert len(Bs) == len(Cs) == len(sizes) == len(qparams) == p
        self.count = p
        self.kernel_id = kernel_id
        self._keep = (As, Bs, scale_a, scale_b, Cs, acc)  # keep the tensors alive
        dev = Cs[0].device if p else torch.device("cuda")

        # host tables as arrays: the six pointer rows and the sizes go to the device as one block, sizes and QParams also stay for the launcher
        # (one conversion of all pointers, not one per row, and QParams as bytes)
        block = np.empty(6 * p * 8 + p * 12 + 12, np.uint8)
        ptrs = []
        for ts in (As, Bs, scale_a, scale_b, Cs, acc):
            if not ts:
                ptrs += [0] * p
                continue
            if len(ts) != p:
                raise ValueError(f"a list of {len(ts)} tensors for {p} problems")
            ptrs += [0 if t is None else t.data_ptr() for t in ts]  # (0 for a tensor without elements)
        if p:
            block[:6 * p * 8] = np.frombuffer(array("q", ptrs), np.uint8)
        block[6 * p * 8 + p * 12:] = 0
        h_sizes = block[6 * p * 8:6 * p * 8 + p * 12].view(np.uint32).reshape(p, 3)
        h_sizes[:] = (sizes if isinstance(sizes, np.ndarray) else np.array(sizes, np.int32)).reshape(p, 3)
        sizes_t, qparams_t = _array_types(max(p, 1))
        self.h_sizes = sizes_t.from_buffer(block, 6 * p * 8)
        self.h_q = qparams_t.from_buffer_copy(b"".join([_qparams_bytes(q if type(q) is tuple else tuple(q)) for q in qparams]) or bytes(16))
        self.d_block = _upload(block, dev)
        self._base = self.d_block.data_ptr()
        self.has_acc = acc is not None
        self._host_sizes = h_sizes

    @property
    def sizes(self) -> list:
        return [tuple(s) for s in self._host_sizes.tolist()]

    @property
    def ops(self) -> int:
        return int(2 * self._host_sizes.astype(np.int64).prod(axis=1).sum())

    def _ptr(self, row: int) -> int:
        return self._base + row * self.count * 8

    def run(self, stream=None) -> None:
        if self.count == 0:
            return
        s = stream if stream is not None else _lib.current_stream()
        rc = self.lib.mxmoe_group_gemm(
            self.kernel_id, self._ptr(0), self._ptr(1), self._ptr(2), self._ptr(3), self._ptr(4), self._ptr(4),
            None, None, None, None, self._ptr(6), self.h_sizes, None, self.h_q, self.count,
            self._ptr(5) if self.has_acc else None, s,
        )
        _lib.check(self.lib, rc)

    def plan(self):
        """(kernel id, branch per problem, total tiles) the launcher would use."""
        br = (C.c_int32 * max(self.count, 1))()
        tiles = C.c_int32(0)
        rc = self.lib.mxmoe_group_gemm_plan(self.kernel_id, self.h_sizes, self.h_q, self.count, br, C.byref(tiles))
        if rc < 1000:
            _lib.check(self.lib, rc or 1)
        return rc - 1000, list(br)[: self.count], tiles.value
