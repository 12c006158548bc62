"""Torch-tensor front end of the C ABI (``include/msa_amd.h``).

PyTorch is used here only to own device / pinned memory and to name streams; every computation
below happens in the HIP library.  All functions enqueue on the current torch stream unless a
stream is given, and raise :class:`msa_amd._lib.MsaError` on any failure.
"""
from __future__ import annotations

import ctypes as C
import os
from dataclasses import dataclass
from typing import List, Optional, Sequence, Tuple

import torch
from torch.nn.modules.module import _has_any_global_hook

from . import _lib
from ._lib import MODE_COSINE, MODE_SCALED_DOT, check, dtype_code, ptr

MODES = {"cosine": MODE_COSINE, "scaled_dot": MODE_SCALED_DOT}


def _stream(stream: Optional[torch.cuda.Stream] = None) -> int:
    # (current_stream() takes 9 us a call)
    return stream.cuda_stream if stream is not None else torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


class _Scratch:
    """Bytes of the caching allocator on the current stream, given back when the call that holds them returns (a tensor of them takes the
    host 1.4 us, this 0.5)."""
    __slots__ = ("at",)

    def __init__(self, at: int):
        self.at = at

    def __del__(self, free=torch._C._cuda_cudaCachingAllocator_raw_delete):
        free(self.at)

    def data_ptr(self) -> int:
        return self.at


def scratch(need: int, device):
    """Scratch of one call, from the allocator each time: calls on other streams and threads have their own, and inside a capture it
    belongs to the graph, whose replays then share it with nothing."""
    if not need:
        return None
    if device.type != "cuda" or device.index != torch._C._cuda_getDevice():
        return torch.empty(need, dtype=torch.uint8, device=device)
    return _Scratch(torch._C._cuda_cudaCachingAllocator_raw_alloc(need, torch._C._cuda_getCurrentRawStream(device.index)))


def _need_cuda(*ts):
    for t in ts:
        if t is None or (t.is_cuda and t.is_contiguous()):
            continue
        if not t.is_cuda:
            raise ValueError("expected a device tensor (the HIP path has no CPU fallback)")
        raise ValueError("expected a contiguous tensor")


# ------------------------------------------------------------------------------ chunk table
@dataclass
class ChunkTable:
    """Device-side chunking of one packed block (all int32 tensors)."""
    doc_start: torch.Tensor       # [n_docs + 1] token offsets
    doc_chunk_off: torch.Tensor   # [n_docs + 1]
    chunk_start: torch.Tensor     # [C]
    chunk_len: torch.Tensor       # [C]
    chunk_doc: torch.Tensor       # [C] 0-based
    n_chunks: torch.Tensor        # [1] int64, written by the kernel
    P: int
    max_doc_len: int

    @property
    def C(self) -> int:
        return self.chunk_start.numel()


def chunk_table(doc_lens: Sequence[int], P: int, first_token: int = 0, device="cuda", doc_start: Optional[torch.Tensor] = None) -> ChunkTable:
    """Builds the chunk table on the device from host-side document lengths (the host only sizes
    the outputs: ``C = sum(ceil(len / P))``, as src/prefill.py:225 does).  ``doc_start``: the documents' first tokens and the end
    (int32) where the device has them already; without it they are copied there, which waits for the device."""
    lib = _lib.load()
    lens = [int(x) for x in doc_lens]
    if not lens or min(lens) <= 0:
        raise ValueError("every document needs at least one token")
    n_chunks = sum((n + P - 1) // P for n in lens)
    n_docs = len(lens)
    if doc_start is None:
        doc_start = torch.tensor([first_token] + lens, dtype=torch.int64).cumsum(0).to(torch.int32).to(device)
    elif doc_start.dtype != torch.int32 or doc_start.numel() != n_docs + 1 or not doc_start.is_contiguous() or not doc_start.is_cuda:
        raise ValueError(f"doc_start: {n_docs + 1} contiguous int32 values on the device")
    i32 = dict(dtype=torch.int32, device=device)
    t = ChunkTable(doc_start, torch.empty(n_docs + 1, **i32), torch.empty(n_chunks, **i32),
                   torch.empty(n_chunks, **i32), torch.empty(n_chunks, **i32),
                   torch.zeros(1, dtype=torch.int64, device=device), P, max(lens))
    check(lib.msa_chunk_table(ptr(t.doc_start), n_docs, P, n_chunks, ptr(t.doc_chunk_off), ptr(t.chunk_start),
                              ptr(t.chunk_len), ptr(t.chunk_doc), ptr(t.n_chunks), _stream()), "msa_chunk_table")
    return t


class BlockSegments:
    """The segments of one packed block ``[template | documents]`` for all layers of a forward pass: found on the device in one launch,
    read by the host once (``read``), behind work that has been enqueued meanwhile."""
    HOST = 4096                      # documents in the first copy

    def __init__(self, ids: torch.Tensor, mask: Optional[torch.Tensor], pos: Optional[torch.Tensor]):
        """``ids [1, T]``, ``mask`` and ``pos`` (of that shape, or None): contiguous int64 on the device."""
        self.ids, self.mask, self.T = ids, mask, ids.numel()
        _need_cuda(ids, mask, pos)
        if any(t is not None and (t.dtype != torch.int64 or t.shape != ids.shape) for t in (ids, mask, pos)) or ids.shape != (1, self.T):
            raise ValueError("block segments: ids, mask and positions must be int64 [1, T]")
        self._words = torch.empty(8 + self.T + 2, dtype=torch.int32, device=ids.device)      # head, cu
        self._start = torch.empty(self.T + 8, dtype=torch.int64, device=ids.device)
        self._len = torch.empty(self.T + 1, dtype=torch.int32, device=ids.device)
        check(_lib.load().msa_block_segments(ptr(ids), ptr(mask), ptr(pos), self.T, ptr(self._words), ptr(self._words[8:]), ptr(self._start),
                                             ptr(self._len), _stream()), "msa_block_segments")
        n = min(8 + self.T + 2, 8 + self.HOST)
        self._host = torch.empty(n, dtype=torch.int32, pin_memory=True)
        self._host.copy_(self._words[:n], non_blocking=True)
        self._copied = torch.cuda.Event()
        self._copied.record()
        self._tables = {}
        self.done = False

    def read(self) -> "BlockSegments":
        if self.done:
            return self
        self._copied.synchronize()
        n_template, n_docs, bad, last, low, high = self._host[:6].tolist()
        n = n_docs + (n_template > 0)
        words = self._host[8:9 + n] if 9 + n <= self._host.numel() else self._words[8:9 + n].cpu()
        cu = words.tolist()
        self.n_template, self.bad, self.last_position, self.mask_sum = n_template, bool(bad), last, (low & 0xffffffff) | high << 32
        self.lens = [b - a for a, b in zip(cu, cu[1:])]                    # of all segments
        self.doc_lens = self.lens[n_template > 0:]
        self.cu, self.start, self.len = self._words[8:9 + n], self._start[:n], self._len[:n]
        self.done = True
        return self

    def table(self, P: int) -> ChunkTable:
        if P not in self._tables:
            self._tables[P] = chunk_table(self.doc_lens, P, first_token=self.n_template, device=self.ids.device,
                                          doc_start=self.cu[self.n_template > 0:])
        return self._tables[P]


# ------------------------------------------------------------------------------ pooling
def rope_tables(n_rows: int, D: int, theta: float, device="cuda") -> Tuple[torch.Tensor, torch.Tensor]:
    """fp32 ``[n_rows, D/2]`` cos / sin tables, computed the way Qwen3RotaryEmbedding does (fp32
    inv_freq, fp32 angles)."""
    inv_freq = 1.0 / (theta ** (torch.arange(0, D, 2, dtype=torch.int64).float() / D))
    ang = torch.arange(n_rows, dtype=torch.float32)[:, None] * inv_freq[None, :]
    return ang.cos().contiguous().to(device), ang.sin().contiguous().to(device)


def pool_chunks(k: Optional[torch.Tensor], v: Optional[torch.Tensor], kr: Optional[torch.Tensor], table: ChunkTable,
                rope: Optional[Tuple[torch.Tensor, torch.Tensor]] = None, normalize_kr: bool = False):
    """Chunk means of token-major ``[T, H, D]`` tensors -> chunk-major ``[C, H, D]`` (same dtype).
    ``rope=(cos, sin)`` rotates K at per-document positions while reading it."""
    lib = _lib.load()
    ref = next(t for t in (k, v, kr) if t is not None)
    _need_cuda(k, v, kr)
    T, H, D = ref.shape
    for t in (k, v, kr):
        if t is not None and (t.shape != ref.shape or t.dtype != ref.dtype):
            raise ValueError("K, V and K_r must share shape and dtype")
    outs = [None if t is None else torch.empty((table.C, H, D), dtype=ref.dtype, device=ref.device) for t in (k, v, kr)]
    cos, sin = rope if rope is not None else (None, None)
    if rope is not None:
        _need_cuda(cos, sin)
        if cos.dtype != torch.float32 or cos.shape != sin.shape or cos.shape[1] != D // 2:
            raise ValueError("rotary tables must be fp32 [rows, D/2]")
    check(lib.msa_pool_chunks(ptr(k), ptr(v), ptr(kr), dtype_code(ref.dtype), T, H, D, ptr(table.chunk_start),
                              ptr(table.chunk_len), ptr(table.chunk_doc), table.C, ptr(table.doc_start), ptr(cos),
                              ptr(sin), 0 if cos is None else cos.shape[0], table.max_doc_len, int(normalize_kr),
                              ptr(outs[0]), ptr(outs[1]), ptr(outs[2]), _stream()), "msa_pool_chunks")
    return tuple(outs)


# ------------------------------------------------------------------------------ bank + routing
class Bank:
    """Owner of an ``msa_bank`` handle plus the tensors it borrows."""

    def __init__(self, n_layers: int, doc_chunk_off: Sequence[int], doc_global_id: Sequence[int], Hkv: int, D: int,
                 dtype: torch.dtype):
        lib = _lib.load()
        self.off_host = torch.as_tensor(doc_chunk_off, dtype=torch.int32).contiguous()
        self.gid_host = torch.as_tensor(doc_global_id, dtype=torch.int64).contiguous()
        self.n_docs = self.gid_host.numel()
        if self.off_host.numel() != self.n_docs + 1:
            raise ValueError("doc_chunk_off must have n_docs + 1 entries")
        self.C = int(self.off_host[-1])
        self.max_doc_chunks = int((self.off_host[1:] - self.off_host[:-1]).max())
        self.n_layers, self.Hkv, self.D, self.dtype = n_layers, Hkv, D, dtype
        self._keep = {}
        h = C.c_void_p()
        check(lib.msa_bank_create(C.byref(h), n_layers, self.C, Hkv, D, dtype_code(dtype), ptr(self.off_host),
                                  ptr(self.gid_host), self.n_docs), "msa_bank_create")
        self.handle = h

    def set_layer(self, layer: int, kr: torch.Tensor, k_host: Optional[torch.Tensor] = None,
                  v_host: Optional[torch.Tensor] = None):
        want = (self.C, self.Hkv, self.D)
        _need_cuda(kr)
        for t in (kr, k_host, v_host):
            if t is not None and (tuple(t.shape) != want or t.dtype != self.dtype or not t.is_contiguous()):
                raise ValueError(f"bank tensors must be contiguous {want} {self.dtype}")
        for t in (k_host, v_host):
            if t is not None and (t.is_cuda or not t.is_pinned()):
                raise ValueError("pooled K / V must live in pinned host memory")
        check(_lib.load().msa_bank_set_layer(self.handle, layer, ptr(kr), ptr(k_host), ptr(v_host)),
              "msa_bank_set_layer")
        self._keep[layer] = (kr, k_host, v_host)

    def workspace_bytes(self, B: int, S: int, Hq: int, topk: int, chunk_plane: bool = False) -> int:
        """Scratch of ``route_topk`` (pre-summed queries, row masks, one key per document, candidate lists);
        with ``chunk_plane`` also room for the ``[B, C]`` key plane ``chunk_scores`` needs."""
        lib = _lib.load()
        return (lib.msa_route_workspace_bytes(B, S, Hq, self.Hkv, self.D, self.C, self.n_docs, topk) if chunk_plane
                else lib.msa_route_topk_workspace_bytes(B, S, Hq, self.Hkv, self.D, self.n_docs, topk))

    def workspace(self, B: int, S: int, Hq: int, topk: int, device, chunk_plane: bool = False) -> torch.Tensor:
        return torch.empty(self.workspace_bytes(B, S, Hq, topk, chunk_plane), dtype=torch.uint8, device=device)

    def close(self):
        if getattr(self, "handle", None):
            _lib.load().msa_bank_destroy(self.handle)
            self.handle = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def _route_args(bank: Bank, q: torch.Tensor, qmask: Optional[torch.Tensor], mode: str):
    _need_cuda(q, qmask)
    if q.dim() != 4 or q.shape[3] != bank.D or q.dtype != bank.dtype:
        raise ValueError(f"q must be [B, S, Hq, {bank.D}] {bank.dtype}")
    B, S, Hq, _ = q.shape
    if qmask is not None:
        if tuple(qmask.shape) != (B, S):
            raise ValueError("qmask must be [B, S]")
        qmask = qmask.to(torch.uint8).contiguous()
    if mode not in MODES:
        raise NotImplementedError(f"unsupported scoring mode {mode!r}")
    return B, S, Hq, qmask


def chunk_scores(bank: Bank, layer: int, q: torch.Tensor, qmask: Optional[torch.Tensor] = None, mode: str = "cosine",
                 scale: float = 1.0) -> torch.Tensor:
    """fp32 ``[B, C]`` chunk scores (mean over heads, max over scored tokens)."""
    B, S, Hq, qm = _route_args(bank, q, qmask, mode)
    need = bank.workspace_bytes(B, S, Hq, 16, chunk_plane=True)
    ws = scratch(need, q.device)
    out = torch.empty((B, bank.C), dtype=torch.float32, device=q.device)
    check(_lib.load().msa_chunk_scores(bank.handle, layer, ptr(q), ptr(qm), B, S, Hq, MODES[mode], scale, ptr(out),
                                       ptr(ws), need, _stream()), "msa_chunk_scores")
    return out


QUERY_REDUCE = {"max": 0, "mean": 1, "last": 2}     # the reference's query_reduce_method (src/msa_service.py:749-780)
CHUNK_REDUCE = {"max": 0, "mean": 1}                # chunk_reduce_method (:787-811)


def route_topk(bank: Bank, layer: int, q: torch.Tensor, qmask: Optional[torch.Tensor] = None, mode: str = "cosine",
               scale: float = 1.0, topk: int = 16, query_reduce: str = "max", chunk_reduce: str = "max"):
    """``(scores [B, k] fp32, doc [B, k] int32 0-based, doc_global [B, k] int64)``.  ``query_reduce`` / ``chunk_reduce``
    other than "max" take the reference's other reductions (``msa_route_topk_reduce``)."""
    B, S, Hq, qm = _route_args(bank, q, qmask, mode)
    if query_reduce not in QUERY_REDUCE:
        raise NotImplementedError(f"Unsupported query reduce method: {query_reduce}")
    if chunk_reduce not in CHUNK_REDUCE:
        raise ValueError(f"Invalid chunk reduction method: {chunk_reduce}")
    scores = torch.empty((B, topk), dtype=torch.float32, device=q.device)
    doc = torch.empty((B, topk), dtype=torch.int32, device=q.device)
    gid = torch.empty((B, topk), dtype=torch.int64, device=q.device)
    need = bank.workspace_bytes(B, S, Hq, topk, chunk_plane=chunk_reduce != "max")
    ws = scratch(need, q.device)
    if query_reduce == "max" and chunk_reduce == "max":
        check(_lib.load().msa_route_topk(bank.handle, layer, ptr(q), ptr(qm), B, S, Hq, MODES[mode], scale, topk,
                                         ptr(scores), ptr(doc), ptr(gid), ptr(ws), need, _stream()),
              "msa_route_topk")
    else:
        check(_lib.load().msa_route_topk_reduce(bank.handle, layer, ptr(q), ptr(qm), B, S, Hq, MODES[mode], scale,
                                                QUERY_REDUCE[query_reduce], CHUNK_REDUCE[chunk_reduce], topk, ptr(scores),
                                                ptr(doc), ptr(gid), ptr(ws), need, _stream()),
              "msa_route_topk_reduce")
    return scores, doc, gid


# ------------------------------------------------------------------------------ gather
def gather_kv(bank: Bank, layer: int, doc_sel_host: torch.Tensor, device, stream: Optional[torch.cuda.Stream] = None):
    """Copies the selected documents' pooled K / V rows from pinned host memory on ``stream``.
    Returns ``(K [sum, Hkv, D], V, cu_sel int64 [B + 1] (host))``; the copies are merely enqueued."""
    lib = _lib.load()
    sel = doc_sel_host.to(torch.int32).contiguous()
    if sel.is_cuda or sel.dim() != 2:
        raise ValueError("doc_sel_host must be a host tensor [B, k]")
    B, k = sel.shape
    cu = torch.empty(B + 1, dtype=torch.int64)
    check(lib.msa_gather_plan(bank.handle, ptr(sel), B, k, ptr(cu)), "msa_gather_plan")
    total = int(cu[-1])
    with torch.cuda.stream(stream) if stream is not None else _null_ctx():
        k_out = torch.empty((total, bank.Hkv, bank.D), dtype=bank.dtype, device=device)
        v_out = torch.empty_like(k_out)
    check(lib.msa_gather_kv(bank.handle, layer, ptr(sel), B, k, ptr(k_out), ptr(v_out), total, _stream(stream)),
          "msa_gather_kv")
    return k_out, v_out, cu


def gather_kv_device(bank: Bank, layer: int, doc_sel: torch.Tensor, capacity_chunks: int,
                     out: Optional[Tuple[torch.Tensor, torch.Tensor]] = None):
    """Device-side gather: ``doc_sel [B, k]`` int32 on the device (e.g. ``route_topk``'s documents).  Returns
    ``(K [capacity, Hkv, D], V, cu_sel int32 [B + 1] on the device)``; rows ``cu_sel[b] .. cu_sel[b + 1]`` belong to
    sample ``b``.  No host synchronisation."""
    _need_cuda(doc_sel)
    if doc_sel.dtype != torch.int32 or doc_sel.dim() != 2:
        raise ValueError("doc_sel must be int32 [B, k]")
    B, k = doc_sel.shape
    lib = _lib.load()
    dev = doc_sel.device
    if out is None:
        k_out = torch.empty((capacity_chunks, bank.Hkv, bank.D), dtype=bank.dtype, device=dev)
        v_out = torch.empty_like(k_out)
    else:
        k_out, v_out = out
    cu = torch.empty(B + 1, dtype=torch.int32, device=dev)
    need = lib.msa_gather_device_workspace_bytes(B, k)
    ws = scratch(need, dev)
    check(lib.msa_gather_kv_device(bank.handle, layer, ptr(doc_sel), B, k, ptr(k_out), ptr(v_out), capacity_chunks, ptr(cu),
                                   ptr(ws), need, _stream()), "msa_gather_kv_device")
    return k_out, v_out, cu


def route_topk_gather(bank: Bank, layer: int, q: torch.Tensor, qmask: Optional[torch.Tensor], mode: str, scale: float,
                      topk: int, gather_layer: int, gather_doc_sel: torch.Tensor, capacity_chunks: int,
                      out: Optional[Tuple[torch.Tensor, torch.Tensor]] = None):
    """``route_topk`` of ``layer`` with ``gather_kv_device`` of (``gather_layer``, ``gather_doc_sel``) in the same
    launch (one workgroup of the scan copies while the others score).  Returns the two calls' results:
    ``(scores, doc, doc_global), (K, V, cu_sel)``."""
    B, S, Hq, qm = _route_args(bank, q, qmask, mode)
    _need_cuda(gather_doc_sel)
    if gather_doc_sel.dtype != torch.int32 or gather_doc_sel.dim() != 2:
        raise ValueError("gather_doc_sel must be int32 [B, k]")
    gB, gk = gather_doc_sel.shape
    lib = _lib.load()
    dev = q.device
    need, gneed = bank.workspace_bytes(B, S, Hq, topk), lib.msa_gather_device_workspace_bytes(gB, gk)
    ws, gws = scratch(need, dev), scratch(gneed, dev)
    scores = torch.empty((B, topk), dtype=torch.float32, device=dev)
    doc = torch.empty((B, topk), dtype=torch.int32, device=dev)
    gid = torch.empty((B, topk), dtype=torch.int64, device=dev)
    if out is None:
        k_out = torch.empty((capacity_chunks, bank.Hkv, bank.D), dtype=bank.dtype, device=dev)
        v_out = torch.empty_like(k_out)
    else:
        k_out, v_out = out
    cu = torch.empty(gB + 1, dtype=torch.int32, device=dev)
    check(lib.msa_route_topk_gather(bank.handle, layer, ptr(q), ptr(qm), B, S, Hq, MODES[mode], scale, topk, ptr(scores),
                                    ptr(doc), ptr(gid), ptr(ws), need, gather_layer, ptr(gather_doc_sel), gB, gk,
                                    ptr(k_out), ptr(v_out), capacity_chunks, ptr(cu), ptr(gws), gneed, _stream()),
          "msa_route_topk_gather")
    return (scores, doc, gid), (k_out, v_out, cu)


class _null_ctx:
    def __enter__(self):
        return None

    def __exit__(self, *a):
        return False


# ------------------------------------------------------------------------------ cache + attention
def assemble_context(prefix_k, prefix_v, mem_k, mem_v, cu_sel, local_k, local_v, cu_local, B: int, Lcap: int):
    """Builds ``kcache / vcache [B, Lcap, Hkv, D]`` and ``kv_len [B]`` from
    ``[prefix | memory rows of b | local rows of b]``."""
    ref = next(t for t in (prefix_k, mem_k, local_k) if t is not None)
    Hkv, D = ref.shape[-2], ref.shape[-1]
    _need_cuda(prefix_k, prefix_v, mem_k, mem_v, cu_sel, local_k, local_v, cu_local)
    kc = torch.empty((B, Lcap, Hkv, D), dtype=ref.dtype, device=ref.device)
    vc = torch.empty_like(kc)
    kv_len = torch.empty(B, dtype=torch.int32, device=ref.device)
    n_prefix = 0 if prefix_k is None else prefix_k.shape[0]
    check(_lib.load().msa_assemble_context(ptr(prefix_k), ptr(prefix_v), n_prefix, ptr(mem_k), ptr(mem_v),
                                           ptr(cu_sel), ptr(local_k), ptr(local_v), ptr(cu_local), B, Hkv, D,
                                           dtype_code(ref.dtype), ptr(kc), ptr(vc), Lcap, ptr(kv_len), _stream()),
          "msa_assemble_context")
    return kc, vc, kv_len


def cache_append(k_new, v_new, kcache, vcache, kv_len):
    """Writes one ``[B, Hkv, D]`` row per sample at ``kv_len[b]`` and increments it, in place."""
    _need_cuda(k_new, v_new, kcache, vcache, kv_len)
    B, Lcap, Hkv, D = kcache.shape
    check(_lib.load().msa_cache_append(ptr(k_new), ptr(v_new), B, Hkv, D, dtype_code(kcache.dtype), ptr(kcache),
                                       ptr(vcache), Lcap, ptr(kv_len), _stream()), "msa_cache_append")


def cache_append_rows(k_new, v_new, cu_new, max_new: int, kcache, vcache, kv_len):
    """Ragged append: sample ``b`` gets rows ``cu_new[b]:cu_new[b+1]`` of ``k_new / v_new [total, Hkv, D]`` at
    ``kv_len[b]``, which grows by that count (clamped to the capacity), in place."""
    _need_cuda(k_new, v_new, cu_new, kcache, vcache, kv_len)
    B, Lcap, Hkv, D = kcache.shape
    if cu_new.dtype != torch.int32 or cu_new.numel() != B + 1 or k_new.shape[1:] != (Hkv, D) or k_new.shape != v_new.shape:
        raise ValueError("cu_new int32 [B + 1]; k_new / v_new [total, Hkv, D]")
    check(_lib.load().msa_cache_append_rows(ptr(k_new), ptr(v_new), ptr(cu_new), max_new, B, Hkv, D,
                                            dtype_code(kcache.dtype), ptr(kcache), ptr(vcache), Lcap, ptr(kv_len),
                                            _stream()), "msa_cache_append_rows")


FLASH_MIN_ROWS = 16     # bf16 query blocks at least this long go to the MFMA flash kernel


def sparse_attn(q, k, v, kv_off, kv_len, max_kv: int, cu_q=None, max_sq: int = 1, scale: Optional[float] = None,
                causal: bool = True):
    """GQA attention of ``q [total_q, Hq, D]`` over per-sample key ranges of ``k / v [rows, Hkv, D]``."""
    _need_cuda(q, k, v, kv_off, kv_len, cu_q)
    total_q, Hq, D = q.shape
    Hkv = k.shape[-2]
    B = kv_len.numel()
    if kv_off.dtype != torch.int64 or kv_len.dtype != torch.int32 or (cu_q is not None and cu_q.dtype != torch.int32):
        raise ValueError("kv_off int64, kv_len / cu_q int32")
    lib = _lib.load()
    sc = D ** -0.5 if scale is None else scale
    # bf16 query blocks: the one-pass MFMA flash kernel, except where its few workgroups (tiles of 128 columns) would each walk over many
    # keys: there the split-KV entry point below, which runs the same kernel per key range and combines.  A key range less costs 2.3 us in 128
    # keys, the combining 3 us and the way of the partials, which grows with the rows and heads.  Where both take as long, and the line: 16 rows of 8
    # heads over 8 370 keys and 278, of 32 over 32 370 and 336, 128 rows of 32 over 8 560 and 515, 4 x 60 of 16 over 8 500 and 503, 16 x 60 of 8 over 8 900 and
    # 848, 400 of 32 over 8 1400 and 1066 (us there, flash and split: 1024 keys 24.4 and 30.1, 1536 34.1 and 32.8); within 0.2 % of the better one in the
    # mean of 600 sizes, 13 % behind at most (without keys: zeros from as many rows as fill the chip, refused below)
    tiles = Hkv * max(B, -(-total_q * (Hq // max(1, Hkv)) // 128))
    one_pass = tiles > 128 or max_kv <= 260 + total_q * Hq // 20 + 8 * tiles // 5 if max_kv > 0 else total_q * Hkv >= 32 * 512
    if q.dtype == torch.bfloat16 and max_sq >= FLASH_MIN_ROWS and one_pass:
        out = torch.empty_like(q)
        check(lib.msa_flash_attn_fit(ptr(q), ptr(cu_q), ptr(k), ptr(v), ptr(kv_off), ptr(kv_len), B, total_q, Hq, Hkv, D,
                                     sc, int(causal), ptr(out), int(max_sq), _stream()), "msa_flash_attn")
        return out
    need = lib.msa_attn_workspace_bytes(total_q, Hq, Hkv, D, max_kv)
    ws = scratch(need, q.device)
    out = torch.empty_like(q)
    check(lib.msa_sparse_attn(ptr(q), ptr(cu_q), ptr(k), ptr(v), ptr(kv_off), ptr(kv_len), B, total_q, max_sq, max_kv,
                              Hq, Hkv, D, dtype_code(q.dtype), sc, int(causal),
                              ptr(out), ptr(ws), need, _stream()), "msa_sparse_attn")
    return out


# ------------------------------------------------------------------------------ fused layer helpers
def qk_norm_rope(qkv: torch.Tensor, Hq: int, Hkv: int, D: int, positions: torch.Tensor, q_norm_w, k_norm_w, eps: float,
                 rope: Tuple[torch.Tensor, torch.Tensor]):
    """``qkv [N, (Hq + 2 Hkv) * D]`` (fused projection output) -> ``q [N, Hq, D]`` and ``k [N, Hkv, D]``
    normalised per head and rotated at ``positions [N]``, plus ``v [N, Hkv, D]`` copied dense."""
    _need_cuda(qkv, positions, q_norm_w, k_norm_w, rope[0], rope[1])
    N, W = qkv.shape
    if W != (Hq + 2 * Hkv) * D or positions.dtype != torch.int64 or positions.numel() != N:
        raise ValueError("qkv must be [N, (Hq + 2 Hkv) D] and positions int64 [N]")
    q = torch.empty((N, Hq, D), dtype=qkv.dtype, device=qkv.device)
    k = torch.empty((N, Hkv, D), dtype=qkv.dtype, device=qkv.device)
    v = torch.empty((N, Hkv, D), dtype=qkv.dtype, device=qkv.device)
    es = qkv.element_size()
    base = qkv.data_ptr()
    check(_lib.load().msa_qk_norm_rope(base, base + Hq * D * es, base + (Hq + Hkv) * D * es, W, W, W, ptr(positions),
                                       ptr(q_norm_w), ptr(k_norm_w), eps, ptr(rope[0]), ptr(rope[1]), rope[0].shape[0],
                                       dtype_code(qkv.dtype), N, Hq, Hkv, D, ptr(q), ptr(k), ptr(v), _stream()),
          "msa_qk_norm_rope")
    return q, k, v


def qkv_proj(x: torch.Tensor, w: torch.Tensor, Hq: int, Hkv: int, positions: torch.Tensor, q_norm_w, k_norm_w, eps: float,
             rope: Tuple[torch.Tensor, torch.Tensor], router_front: int = 0, router_back: int = 0):
    """Fused projection of ``x [T, K]`` (bf16) through ``w [(router_front + Hq + 2 Hkv + router_back) * 128, K]``:
    returns ``q [T, Hq, 128]`` and ``k [T, Hkv, 128]`` (per-head RMSNorm + rotary at ``positions [T]`` done in the
    GEMM's epilogue), ``v [T, Hkv, 128]`` and the router heads ``r [T, router_front + router_back, 128]`` (``None``
    without router heads), all dense."""
    _need_cuda(x, w, positions, q_norm_w, k_norm_w, rope[0], rope[1])
    T, K = x.shape
    D = 128
    heads = router_front + Hq + 2 * Hkv + router_back
    if x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16 or tuple(w.shape) != (heads * D, K):
        raise ValueError(f"qkv_proj: x [T, K] and w [{heads * D}, K] in bf16")
    if positions.dtype != torch.int64 or positions.numel() != T:
        raise ValueError("qkv_proj: positions int64 [T]")
    for name, nw in (("q_norm_w", q_norm_w), ("k_norm_w", k_norm_w)):
        if nw.dtype != torch.bfloat16 or nw.numel() != D or not nw.is_contiguous():
            raise ValueError(f"qkv_proj: {name} must be {D} contiguous bf16 weights, got {nw.dtype} x {nw.numel()}")
    for name, tab in (("cos", rope[0]), ("sin", rope[1])):
        if tab.dtype != torch.float32 or tab.dim() != 2 or tab.shape[1] != D // 2 or not tab.is_contiguous():
            raise ValueError(f"qkv_proj: the {name} table must be contiguous fp32 [rows, {D // 2}], got {tab.dtype} "
                             f"{tuple(tab.shape)}")
    if rope[0].shape != rope[1].shape:
        raise ValueError("qkv_proj: cos / sin tables differ in shape")
    if not (x.is_contiguous() and w.is_contiguous()) or x.data_ptr() % 16 or w.data_ptr() % 16:
        raise ValueError("qkv_proj: x and w must be contiguous and 16-byte aligned")
    dev = x.device
    q = torch.empty((T, Hq, D), dtype=x.dtype, device=dev)
    k = torch.empty((T, Hkv, D), dtype=x.dtype, device=dev)
    v = torch.empty((T, Hkv, D), dtype=x.dtype, device=dev)
    r = torch.empty((T, router_front + router_back, D), dtype=x.dtype, device=dev) if router_front + router_back else None
    need = _lib.load().msa_tile_workspace_bytes(T, K, heads * D)
    ws = scratch(need, dev)
    check(_lib.load().msa_qkv_proj_ws(ptr(x), T, K, ptr(w), Hq, Hkv, router_front, router_back, ptr(positions), ptr(q_norm_w),
                                      ptr(k_norm_w), eps, ptr(rope[0]), ptr(rope[1]), rope[0].shape[0], ptr(q), ptr(k), ptr(v),
                                      ptr(r), ptr(ws), need, _stream()), "msa_qkv_proj")
    return q, k, v, r


def tile_linear(x: torch.Tensor, w: torch.Tensor, out: Optional[torch.Tensor] = None, add: bool = False,
                silu_mul: bool = False, glu: Optional[Tuple[float, float, float]] = None, gelu_n: int = 0) -> torch.Tensor:
    """``x @ w.T`` of a block of bf16 rows ``x [T, K]`` (unit column stride, K a multiple of 64) with a dense ``w [N, K]``, into ``out``
    where given.  At most one of: ``add`` adds the product to ``out``; ``silu_mul`` takes ``w`` from ``interleave_gate_up`` and returns
    ``silu(gate) * up`` of width ``N / 2``; ``glu`` (limit, alpha, shift) takes rows in (gate, up) pairs and returns the clamped gated
    unit; ``gelu_n`` puts the first columns through gelu."""
    _need_cuda(w)
    if x.dim() != 2 or w.dim() != 2 or x.shape[1] != w.shape[1] or x.stride(1) != 1 or not x.is_cuda or w.device != x.device:
        raise ValueError("tile_linear: x [T, K] with unit column stride, w [N, K] contiguous, both on one device")
    if x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16:
        raise ValueError("tile_linear: x and w in bf16")
    if add + silu_mul + (glu is not None) + (gelu_n != 0) > 1 or (add and out is None):
        raise ValueError("tile_linear: one of add (with out), silu_mul, glu and gelu_n")
    (T, K), N = x.shape, w.shape[0]
    width = N // 2 if silu_mul or glu is not None else N
    if out is None:
        out = torch.empty((T, width), dtype=x.dtype, device=x.device)
    elif tuple(out.shape) != (T, width) or out.dtype != x.dtype or out.stride(1) != 1 or out.device != x.device:
        raise ValueError(f"tile_linear: out must be bf16 [{T}, {width}] on x's device with unit column stride")
    if not T:
        return out
    need = _lib.load().msa_tile_workspace_bytes(T, K, N)
    ws = scratch(need, x.device)
    mode = (_lib.TILE_ADD if add else _lib.TILE_SILU_MUL if silu_mul else _lib.TILE_GLU if glu is not None
            else _lib.TILE_GELU if gelu_n else _lib.TILE_STORE)
    end = _lib.TileEnd(mode, gelu_n, *(glu or (0.0, 0.0, 0.0)))
    rows = lambda t: t.stride(0) if T > 1 else t.shape[1]
    check(_lib.load().msa_tile_linear(ptr(x), rows(x), T, K, ptr(w), N, C.byref(end), ptr(out), rows(out), ptr(ws), need,
                                      _stream()), "msa_tile_linear")
    return out


TILE_MIN = 144 << 16    # outputs (144 tiles of 256 x 256) from which tile_linear with an end is at least the equal of the vendor's two launches
TILE_PLAIN = 256 << 16  # without one, where the vendor's tiles fit the columns
DEEP, DEEP_ROWS, DEEP_TILES = 8192, 448, (20, 110)
TILE_ROWS = 256         # no matrix of the models has outputs enough for fewer rows


def tile_linear_ok(x: torch.Tensor, w: torch.Tensor, matrices: int = 1, end: bool = True) -> bool:
    """Whether ``x [..., K] @ w.T`` (``matrices`` of w's shape in one; with an ``end`` besides the store) is ``tile_linear``'s: operands as it
    takes them, nothing but their values asked for (no gradients in either direction, no vmap or trace), and outputs enough to fill the compute units.  us in a loop of 60 ms, the vendor's (and its second
    launch) and here, rows x K x N: with an end 573 x 2560 x 19456 glu and 1600 x 1024 x 6144 glu level, 900 x 2560 x 19456 1.06 times, 6001 1.26
    times the speed; without one and N no multiple of 256 1600 x 1024 x 6176 1.10, 900 x 2560 x 14944 1.17 times.  Where N is one, a single
    round of tiles is behind the vendor's smaller ones (6001 x 9728 x 2560 199 and 217, 6001 x 4096 x 2560 86 and 93, 10000 x 3072 x 1024 53 and
    63), and several are level or ahead (7000 x 2560 x 2560 1.14 times, 6001 x 4096 x 12288 1.28, but 4096 x 2560 x 6144 0.87).  Padding does not
    count.  Deep products whose tiles are less than half a round, cut into pieces of K, are ahead as well (``DEEP``; weights not in the caches: 500 x 9728 x 2560 51.1 and 46.2,
    769 76 and 58, 1492 89 and 78, 2340 189 and 116; a third of a round deeper or half as deep they are level or behind: 3200 x 9728 x 2560 130 and 150, 1492 x
    4096 x 2560 42 and 47).  A step's products ask ``flow_linear`` first up to ``FLOW_FIRST`` rows, modules (``linear``) come here from ``DEEP_ROWS`` on.  Depths under 1024 were not measured and stay where they were."""
    N = matrices * w.shape[0]
    K = x.shape[-1]
    if x.numel() * N < (TILE_MIN if end or N % 256 else TILE_PLAIN) * max(K, 1):   # (most calls end here: steps of few tokens wait for the host)
        if end or N % 256 or K < DEEP or x.numel() < DEEP_ROWS * K or not DEEP_TILES[0] <= -(-x.numel() // (256 * K)) * (N // 256) <= DEEP_TILES[1]:
            return False
    T = x.numel() // K
    return (x.is_cuda and x.dtype == w.dtype == torch.bfloat16 and host().ordinary(x, w) and w.dim() == 2 and w.is_contiguous() and w.shape[1] == K
            and (x.is_contiguous() or (x.dim() == 2 and x.stride(1) == 1 and x.stride(0) % 8 == 0 and K <= x.stride(0) < 1 << 21))
            and K % 64 == 0 and 1024 <= K <= 32768 and N % 8 == 0 and N < 1 << 20 and T < 1 << 22
            and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0 and w.device == x.device
            and not (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad)))


BLOCK_US, BLOCK_ROWS, BLOCK_DEPTH = 23.0, 2048, 128
CAPTURED_US, CAPTURED_ROWS, CAPTURED_DEPTH = 12.5, 1024, 2048


def block_linear_ok(x: torch.Tensor, w: torch.Tensor, end: bool = False) -> bool:
    """Whether ``x [T, K] @ w.T`` (with an ``end``: behind which the vendor's product needs another launch) is ``block_linear``'s: operands
    as it takes them, no gradients asked for, and about as fast there or faster.  The host takes about 21 us to hand a product to the
    vendor's library and 5 to this, so up to ``BLOCK_ROWS`` rows, where a prompt waits for the host, products of about that length are here
    also where the vendor's kernel alone is a little faster (us, the vendor's and here, rows x K x N: 64 x 1024 x 1024 6.6 and 5.0, 1000 x
    1024 x 6176 24.2 and 20.5, 2048 x 1024 x 4096 20.6 and 22; behind the line 300 x 2560 x 8192, 25.8 and 27.4).  Of more rows those of a depth up to ``BLOCK_DEPTH`` (6001 x 128 x 4096 25.9 and 18.5; 8192 x 256 x 2048 16.7 and 19.0).  A captured
    call pays for no host: there the kernels alone decide (17 x 1024 x 6176 9.0 and 5.7, 64 x 1024 x 1024 7.0 and 5.4, 1000 x 2048 x 1024 11.8
    and 11.0; behind the lines 32 x 2560 x 2560 7.7 and 9.9, 17 x 4096 x 2560 11.8 and 13.8, 1500 x 128 x 4096 9.0 and 10.4, 573 x 1024 x 8192
    16.4 and 21.0)."""
    if x.is_cuda and (took := host().block_ok(x, w, end)) is not None:
        return took
    (T, K), N = (x.shape if x.dim() == 2 else (0, 0)), w.shape[0]
    if not (T > 0 and w.dim() == 2 and x.is_cuda and x.dtype == w.dtype == torch.bfloat16 and w.is_contiguous() and w.shape[1] == K
            and K % 64 == 0 and 64 <= K <= 32768 and N % 16 == 0 and 0 < N < 1 << 20 and T < 1 << 22 and (T <= BLOCK_ROWS or K <= BLOCK_DEPTH)):
        return False
    us = _lib.load().msa_block_linear_us(T, K, N)
    if us > BLOCK_US or (not end and (us > CAPTURED_US or T > CAPTURED_ROWS or K > CAPTURED_DEPTH)
                         and torch.cuda.is_current_stream_capturing()):
        return False
    return ((x.is_contiguous() or (x.stride(1) == 1 and x.stride(0) % 8 == 0 and K <= x.stride(0) < 1 << 21))
            and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0 and w.device == x.device
            and not (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad)))


def block_linear(x: torch.Tensor, w: torch.Tensor, glu: Optional[Tuple[float, float, float]] = None, gelu_n: int = 0) -> torch.Tensor:
    """``tile_linear`` of few rows (``x`` and ``w`` as ``block_linear_ok`` has them), with ``glu``, ``gelu_n`` or neither."""
    out = host().linear(x, w, _lib.TILE_GLU if glu is not None else _lib.TILE_GELU if gelu_n else _lib.TILE_STORE, gelu_n, *(glu or _NO_GLU))
    if out is None:
        raise ValueError("block_linear: x [T, K] and w [N, K] on the device")
    if type(out) is int:
        check(out, "msa_block_linear")
    return out


_NO_GLU = (0.0, 0.0, 0.0)
FLOW_FIRST = 896        # rows up to which deep products are flow_linear's (weights from memory, there and here: 700 x 9728 x 2560 53 and 49 us, 1000 61.5 and 64)


def flow_linear(x: torch.Tensor, w: torch.Tensor, glu: Optional[Tuple[float, float, float]] = None, gelu_n: int = 0) -> Optional[torch.Tensor]:
    """``tile_linear`` of some hundred rows, ``x [T, K]`` and ``w [N, K]``, with ``glu``, ``gelu_n`` or neither, where one round of mid-sized
    tiles fills the chip; None where another form is the better one or has to take the operands (gradients, strides, types)."""
    if not x.is_cuda:
        return None
    out = host().flow(x, w, _lib.TILE_GLU if glu is not None else _lib.TILE_GELU if gelu_n else _lib.TILE_STORE, gelu_n, *(glu or _NO_GLU))
    if type(out) is int:
        check(out, "msa_flow_linear")
    return out


_host = None


def host():
    """The module of ``csrc/host.cpp``, bound to the libraries; raises if it is missing."""
    global _host
    if _host is None:
        module = _lib.load_host()
        module.bind(_lib.LIB_PATH if os.path.exists(_lib.LIB_PATH) else None, _lib.SEQ_LIB_PATH, (BLOCK_ROWS, BLOCK_DEPTH, CAPTURED_ROWS, CAPTURED_DEPTH, BLOCK_US, CAPTURED_US))
        _host = module
    return _host


def plain_module(module: torch.nn.Module, base: type) -> bool:
    """Whether ``base``'s own ``forward`` and nothing else runs when the module is called: no forward of a subclass or of the instance, and
    no hooks, the module's or global ones."""
    return (getattr(type(module), "forward", None) is base.forward and "forward" not in module.__dict__
            and not (module._forward_hooks or module._forward_pre_hooks or module._backward_hooks or module._backward_pre_hooks)
            and not _has_any_global_hook())


def embed_ok(table: torch.Tensor, tokens: torch.Tensor) -> bool:
    """Whether ``embed_rows`` takes the lookup (torch's own takes the others)."""
    return (table.is_cuda and tokens.device == table.device and table.dim() == 2 and table.dtype in (torch.bfloat16, torch.float32)
            and tokens.dtype == torch.int64 and tokens.numel() > 0 and table.shape[1] % 8 == 0 and table.is_contiguous()
            and tokens.is_contiguous() and table.data_ptr() % 16 == 0 and not (torch.is_grad_enabled() and table.requires_grad))


def embed_rows(table: torch.Tensor, tokens: torch.Tensor, f32: bool = False, wrap: bool = False, lib=None):
    """``table[tokens]`` and, with ``f32``, the same in fp32 (``(rows, rows in fp32)``).  ``wrap``: negative tokens count from the end."""
    _need_cuda(table, tokens)
    out = torch.empty((*tokens.shape, table.shape[1]), dtype=table.dtype, device=table.device)
    wide = torch.empty(out.shape, dtype=torch.float32, device=table.device) if f32 else None
    lib = lib or _lib.load()
    check(lib.msa_embed_rows(ptr(tokens), tokens.numel(), ptr(table), table.shape[0], wrap, table.shape[1], dtype_code(table.dtype), ptr(out),
                             ptr(wide), _stream()), "msa_embed_rows", lib)
    return (out, wide) if f32 else out


def linear_ok(module: torch.nn.Module, x: torch.Tensor, end: bool = False) -> bool:
    if type(module) is not torch.nn.Linear or not tile_linear_ok(x, module.weight, end=end):
        return False
    return module.bias is None and x.is_contiguous() and type(module.weight) is torch.nn.Parameter and plain_module(module, torch.nn.Linear)


def linear(module: torch.nn.Module, x: torch.Tensor) -> torch.Tensor:
    """``module(x)``, by ``tile_linear`` where that is the faster form."""
    if linear_ok(module, x):
        return tile_linear(x.view(-1, x.shape[-1]), module.weight).view(*x.shape[:-1], -1)
    return module(x)


def qk_norm_rope_append(qkv: torch.Tensor, Hq: int, Hkv: int, D: int, positions: torch.Tensor, q_norm_w, k_norm_w,
                        eps: float, rope: Tuple[torch.Tensor, torch.Tensor], kcache: torch.Tensor, vcache: torch.Tensor,
                        kv_len: torch.Tensor) -> torch.Tensor:
    """Decode-step form of :func:`qk_norm_rope` (one new token per sample): returns ``q [B, Hq, D]`` and writes
    the k / v rows into ``kcache / vcache [B, Lcap, Hkv, D]`` at ``kv_len[b]``, which is incremented in place."""
    _need_cuda(qkv, positions, q_norm_w, k_norm_w, rope[0], rope[1], kcache, vcache, kv_len)
    B, W = qkv.shape
    if W != (Hq + 2 * Hkv) * D or positions.dtype != torch.int64 or positions.numel() != B:
        raise ValueError("qkv must be [B, (Hq + 2 Hkv) D] and positions int64 [B]")
    if (kcache.shape != vcache.shape or kcache.dim() != 4 or kcache.shape[0] != B or tuple(kcache.shape[2:]) != (Hkv, D)
            or kcache.dtype != qkv.dtype or not (kcache.is_contiguous() and vcache.is_contiguous())):
        raise ValueError("kcache / vcache must be contiguous [B, Lcap, Hkv, D] of qkv's dtype")
    if kv_len.dtype != torch.int32 or kv_len.numel() != B:
        raise ValueError("kv_len must be int32 [B]")
    q = torch.empty((B, Hq, D), dtype=qkv.dtype, device=qkv.device)
    es, base = qkv.element_size(), qkv.data_ptr()
    check(_lib.load().msa_qk_norm_rope_append(base, base + Hq * D * es, base + (Hq + Hkv) * D * es, W, W, W,
                                              ptr(positions), ptr(q_norm_w), ptr(k_norm_w), eps, ptr(rope[0]),
                                              ptr(rope[1]), rope[0].shape[0], dtype_code(qkv.dtype), B, Hq, Hkv, D,
                                              ptr(q), ptr(kcache), ptr(vcache), kcache.shape[1], ptr(kv_len), _stream()),
          "msa_qk_norm_rope_append")
    return q


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float, residual: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Row RMSNorm of ``x [..., H]``; with ``residual`` (same shape) does ``residual += x`` in place first
    and normalises the sum."""
    _need_cuda(x, weight, residual)
    H = x.shape[-1]
    out = torch.empty_like(x)
    check(_lib.load().msa_rmsnorm(ptr(x), ptr(residual), ptr(weight), dtype_code(x.dtype), x.numel() // H, H, eps,
                                  ptr(out), _stream()), "msa_rmsnorm")
    return out


def silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    """``silu(gate) * up`` for a fused ``[..., 2 I]`` projection output (gate first)."""
    _need_cuda(gate_up)
    I = gate_up.shape[-1] // 2
    out = torch.empty(gate_up.shape[:-1] + (I,), dtype=gate_up.dtype, device=gate_up.device)
    check(_lib.load().msa_silu_mul(ptr(gate_up), dtype_code(gate_up.dtype), gate_up.numel() // (2 * I), I, ptr(out),
                                   _stream()), "msa_silu_mul")
    return out


def decode_attn_fused(qkv: torch.Tensor, Hq: int, Hkv: int, D: int, positions: torch.Tensor, q_norm_w, k_norm_w,
                      eps: float, rope: Tuple[torch.Tensor, torch.Tensor], kcache: torch.Tensor, vcache: torch.Tensor,
                      kv_len: torch.Tensor, scale: Optional[float] = None) -> torch.Tensor:
    """One decode step from the fused projection output ``qkv [B, (Hq + 2 Hkv) D]`` (bf16) to the attention output
    ``[B, Hq, D]``: q / k norm + rotary, in-place append of the new K / V row to ``kcache / vcache [B, Lcap, Hkv, D]``
    at ``kv_len`` (advanced by one) and attention over ``[cache | new token]``, in two launches."""
    _need_cuda(qkv, positions, q_norm_w, k_norm_w, rope[0], rope[1], kcache, vcache, kv_len)
    B, W = qkv.shape
    if qkv.dtype != torch.bfloat16 or W != (Hq + 2 * Hkv) * D or positions.dtype != torch.int64 or positions.numel() != B:
        raise ValueError("qkv must be bf16 [B, (Hq + 2 Hkv) D] and positions int64 [B]")
    if kcache.shape != vcache.shape or kcache.dim() != 4 or kcache.shape[0] != B or tuple(kcache.shape[2:]) != (Hkv, D) \
            or kcache.dtype != torch.bfloat16 or kv_len.dtype != torch.int32 or kv_len.numel() != B:
        raise ValueError("caches must be bf16 [B, Lcap, Hkv, D] and kv_len int32 [B]")
    Lcap = kcache.shape[1]
    lib = _lib.load()
    need = lib.msa_attn_workspace_bytes(B, Hq, Hkv, D, Lcap)
    ws = scratch(need, qkv.device)
    out = torch.empty((B, Hq, D), dtype=qkv.dtype, device=qkv.device)
    check(lib.msa_decode_attn_fused(ptr(qkv), W, ptr(positions), ptr(q_norm_w), ptr(k_norm_w), eps, ptr(rope[0]),
                                    ptr(rope[1]), rope[0].shape[0], B, Hq, Hkv, D, ptr(kcache), ptr(vcache), Lcap,
                                    ptr(kv_len), D ** -0.5 if scale is None else scale, ptr(out), ptr(ws), need,
                                    _stream()), "msa_decode_attn_fused")
    return out


def greedy_sample(logits: torch.Tensor, tok: torch.Tensor, pos: Optional[torch.Tensor] = None,
                  out: Optional[torch.Tensor] = None, col: Optional[torch.Tensor] = None,
                  scratch: Optional[torch.Tensor] = None, lib=None) -> torch.Tensor:
    """Row-wise argmax of ``logits [B, V]`` written to ``tok`` (int64, ``B`` elements) with the bookkeeping of a
    greedy decode step done in place: ``pos += 1``; ``out[b, col[b]] = tok[b]``; ``col += 1``.  Returns ``tok``."""
    _need_cuda(logits, tok, pos, out, col)
    B, V = logits.shape
    if not logits.is_contiguous() or tok.dtype != torch.int64 or tok.numel() != B:
        raise ValueError("logits must be contiguous [B, V] and tok int64 with B elements")
    for t in (pos, col):
        if t is not None and (t.dtype != torch.int64 or t.numel() != B or not t.is_contiguous()):
            raise ValueError("pos / col must be contiguous int64 with B elements")
    if (out is None) != (col is None) or (out is not None and (out.dtype != torch.int64 or out.stride(-1) != 1)):
        raise ValueError("out [B, max_new] int64 and col go together")
    if scratch is None:
        scratch = torch.empty(B * 32, dtype=torch.int64, device=logits.device)
    lib = lib or _lib.load()              # either library holds it
    check(lib.msa_greedy_sample(ptr(logits), dtype_code(logits.dtype), B, V, ptr(scratch), ptr(tok), ptr(pos),
                                        ptr(out), out.stride(0) if out is not None else 0, ptr(col),
                                        out.shape[1] if out is not None else 0, _stream()), "msa_greedy_sample", lib)
    return tok


SKINNY_MAX_ROWS = 16


def interleave_gate_up(gate_w: torch.Tensor, up_w: torch.Tensor) -> torch.Tensor:
    """``[2 I, K]`` weight with alternating 8-row groups of gate and up rows (rows ``16 i .. 16 i + 7`` are gate
    rows ``8 i .. 8 i + 7``, the next 8 the same up rows): the layout the silu-mul epilogue of ``skinny_linear``
    expects (``I`` a multiple of 8)."""
    I, K = gate_w.shape
    if I % 8 or up_w.shape != gate_w.shape:
        raise ValueError("gate / up weights must be [I, K] with I a multiple of 8")
    return torch.stack([gate_w.view(I // 8, 8, K), up_w.view(I // 8, 8, K)], dim=1).reshape(2 * I, K).contiguous()


def skinny_linear(x: torch.Tensor, w: torch.Tensor, residual: Optional[torch.Tensor] = None,
                  silu_mul: bool = False, norm_weight: Optional[torch.Tensor] = None, eps: float = 1e-6) -> torch.Tensor:
    """``x @ w.T`` for up to 16 rows of bf16 ``x [M, K]`` against ``w [N, K]``, streaming ``w`` once.
    ``residual [M, N]`` is added to the bf16-rounded product; ``silu_mul`` takes ``w`` from ``interleave_gate_up``
    and returns ``silu(gate) * up`` of width ``N / 2``; ``norm_weight [K]`` applies RMSNorm to ``x`` first."""
    _need_cuda(x, w)
    if x.dim() != 2 or w.dim() != 2 or x.shape[1] != w.shape[1] or not x.is_contiguous() or not w.is_contiguous():
        raise ValueError("skinny_linear: x [M, K] and w [N, K], both contiguous")
    if residual is not None and silu_mul:
        raise ValueError("skinny_linear: residual and silu_mul are exclusive")
    M, K = x.shape
    N = w.shape[0]
    out = torch.empty((M, N // 2 if silu_mul else N), dtype=x.dtype, device=x.device)
    if residual is not None and (residual.shape != out.shape or not residual.is_contiguous() or residual.dtype != x.dtype):
        raise ValueError("skinny_linear: residual must be a contiguous [M, N] tensor of x's dtype")
    epi = 2 if silu_mul else (1 if residual is not None else 0)
    if norm_weight is not None and (norm_weight.shape != (K,) or norm_weight.dtype != x.dtype or not norm_weight.is_contiguous()):
        raise ValueError("skinny_linear: norm_weight must be a contiguous [K] tensor of x's dtype")
    lib = _lib.load()
    need = lib.msa_skinny_linear_workspace_bytes(M, N, K)
    ws = scratch(need, x.device)
    check(lib.msa_skinny_linear_ws(ptr(x), ptr(w), ptr(residual) if residual is not None else None,
                                   ptr(norm_weight) if norm_weight is not None else None, float(eps), epi,
                                   dtype_code(x.dtype), M, N, K, ptr(out), ptr(ws), need, _stream()), "msa_skinny_linear_ws")
    return out
