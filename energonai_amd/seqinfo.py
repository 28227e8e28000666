"""Per-batch sequence bookkeeping shared by every kernel call of a forward pass.

The reference recomputes the prefix of ``seq_lens`` inside every block of every
kernel (csrc/transpose_pad_fusion_kernel.cu:24-27,70-73).  Here the prefix is
computed once per batch by one small kernel and reused by every op of every
layer; the public functions still accept the plain ``seq_lens`` tensor of the
reference API (int32 or int64, examples/bert/bert.py:100-103) and find the
cached offsets through :func:`seq_info`.
"""
from __future__ import annotations

from collections import OrderedDict
from typing import Optional

import torch

from . import _lib

_CACHE_SIZE = 16
PER_THREAD_STREAMS = (2,)                 # hipStreamPerThread
TILES_FIRST_MAX_KV_BYTES = 256 << 10     # see tiles_first
TILES_FIRST_MAX_TOTAL_BYTES = 96 << 20
TILES_FIRST_FEW_UNITS = 256
TILES_FIRST_FEW_UNITS_TOTAL_BYTES = 160 << 20


def tiles_first(units: int, unit_kv_bytes: int, causal: Optional[bool] = None) -> bool:
    """Whether the last query tiles of all (batch, head) units run before any unit's others, or a unit's tiles stay together
    (``en_attn_tile_table``).  ``unit_kv_bytes``: K and V of a unit at full length; ``causal`` ``None``: by these alone.

    Under a causal mask a unit's tiles differ in length, last tile longest, and a launch of few units ends on the long tiles of the
    units that came last; the last tiles first, nothing long is left for the end.  The tiles of a unit then no longer share its
    K and V in the XCD's L2, which costs nothing while the memory-side cache holds them all beside what else it holds, or with
    units so few that the tiles running at any time (about 96 an XCD) are several of each.  us a layer, units together / last
    tiles first: 7 sequences of up to 1531, 20 heads x 80, bf16 82 / 78; 1 of 2048, 64 x 128 123 / 102; 3 of up to 1100, 24 x 96
    47 / 39; 8 of up to 2048, 16 x 64 100 / 90; 16 of up to 1024, 16 x 128 (256 units, 128 MB) 93 / 91; 64 of up to 1100, 5 x 64 (320, 85
    MB) 60 / 58; 32 of up to 512, 16 x 64 (512, 64 MB) 38.5 / 37.4.  Beyond: 24 of up to 900, 24 x 64 (576, 126 MB) 69 / 75; 24 of
    768, 16 x 128 (384, 144 MB) 134 / 146; 64 of up to 256, 20 x 128 (1280, 160 MB) 71 / 74; 4 of up to 2048, 72 x 128 (288, 288 MB)
    298 / 322; 16 of up to 2048, 12 x 128 (192, 192 MB) 244 / 247.  Without the mask all tiles of a unit are as long, and its K and V
    are what counts: 32 of up to 512, 16 x 64 44.1 / 46.5, 5 of up to 1300, 20 x 128 66.5 / 71.4."""
    if causal is None:
        return unit_kv_bytes <= TILES_FIRST_MAX_KV_BYTES
    total = units * unit_kv_bytes
    return causal and (total <= TILES_FIRST_MAX_TOTAL_BYTES or
                       (units <= TILES_FIRST_FEW_UNITS and total <= TILES_FIRST_FEW_UNITS_TOTAL_BYTES))


class SeqInfo:
    """Device-resident int32 lengths and exclusive prefix for one batch."""

    __slots__ = ("lens", "cu_seqlens", "batch_size", "_total", "_source", "_row_offsets", "_tile_tables", "_arrivals", "_ready",
                 "_last_tables", "_last_table", "_ordered", "ephemeral", "_lens_host")

    def __init__(self, lens: torch.Tensor, cu_seqlens: torch.Tensor, batch_size: int, total: Optional[int], source):
        self.lens = lens                # int32 [B] on the device
        self.cu_seqlens = cu_seqlens    # int32 [B+1] on the device
        self.batch_size = batch_size
        self._total = total
        self._source = source           # keeps the caller's tensor alive while cached
        self._row_offsets = {}          # (max_seq_len, left_padded, version of lens) -> int32 [T]
        self._tile_tables = {}          # (head_num, q_seq_len, order, version of lens, tile height) -> int32 workgroup order
        self._last_tables = None        # (what layer_tables was asked for, row offsets, tile table): the last it found
        self._last_table = None         # (what tile_table was asked for, tile table): the last it found
        self._arrivals = {}             # (bucket, stream) -> int64 meeting words of en_attn_fused_norm
        self._ready = []                # events recorded behind the kernels that produced the arrays above
        self._ordered = set()           # raw streams already ordered behind every event of _ready
        self.ephemeral = False          # built for one call only (lengths that cannot be cached): see tile_table_ptr
        self._lens_host = None          # (version of lens, the lengths as a Python list)

    def produced_on_current_stream(self) -> None:
        """Call right after launching a kernel that writes one of this object's arrays: remembers the point
        in the launching stream where they are complete."""
        if not self.lens.is_cuda:
            return
        self._ready.append(_lib.front.record_event(self.lens))
        del self._ready[:-8]            # lengths that change every step rebuild their tables every step
        self._ordered = {_lib.stream_of(self.lens)}

    def order_current_stream(self) -> None:
        """Makes torch's current stream wait for the kernels that produced the offsets when they were launched
        on another stream (the arrays are cached and reused by later calls, whichever stream those run on)."""
        if not self._ready:
            return
        raw, ordered = _lib.stream_of(self.lens), self._ordered
        if raw in ordered:
            return
        for ev in self._ready:
            _lib.front.wait_event(ev, self.lens)
        ordered.add(raw)                # of no consequence where another thread's launch has begun a new set meanwhile

    @property
    def device(self) -> torch.device:
        return self.lens.device

    @property
    def total(self) -> int:
        """Sum of the lengths as a Python int.  The first use copies one int from
        the device (a sync), like ``valid_word_num[0].item()`` in the reference
        callers (examples/gpt/gpt.py:303); later uses are free."""
        if self._total is None:
            self._total = int(self.cu_seqlens[self.batch_size].item())
        return self._total


    def lens_host(self):
        """The lengths as a list of Python ints.  The first use copies them from the device (a sync, like
        ``total``); later uses of the same lengths are free, so every layer of a stack can ask."""
        version = self._lens_version()
        if self._lens_host is None or version is None or self._lens_host[0] != version:
            self.order_current_stream()
            self._lens_host = (version, [int(n) for n in self.lens.tolist()])
        return list(self._lens_host[1])

    def _lens_version(self):
        """Version counter of the lengths, part of every key under which something derived from them is kept:
        a caller that owns ``lens`` may change it in place (the K/V cache advances its lengths every step), and
        what was derived from the old lengths must then not be found again.  Tensors created under
        ``torch.inference_mode()`` have no counter; ``None`` then means "do not keep"."""
        try:
            return self.lens._version
        except RuntimeError:
            return None

    def row_offsets(self, max_seq_len: int, left_padded: bool) -> torch.Tensor:
        """``off[t]`` = row of token ``t`` in the padded ``[B*S]`` numbering minus ``t``; computed once per
        batch and bucket by one small kernel (the reference's ft offsets, csrc/transpose_pad_fusion_kernel.cu:
        112-131, made aware of left padding)."""
        version = self._lens_version()
        key = (int(max_seq_len), bool(left_padded), version)
        off = None if version is None and self._mutable() else self._row_offsets.get(key)
        self.order_current_stream()
        if off is None:
            off = torch.empty(max(self.total, 1), dtype=torch.int32, device=self.lens.device)
            with _lib.device_guard(self.lens):
                _lib.check(_lib.fn.en_padding_offsets(self.lens.data_ptr(), self.batch_size, key[0], int(key[1]),
                                                      off.data_ptr(), _lib.stream_of(self.lens)), "padding_offsets")
                self.produced_on_current_stream()
            if version is not None or not self._mutable():
                self._row_offsets = {k: o for k, o in self._row_offsets.items() if k[2] == version}
                self._row_offsets[key] = off
        return off

    def layer_tables(self, max_seq_len: int, left_padded: bool, head_num: int, unit_kv_bytes: int, causal: Optional[bool] = None):
        """``(row_offsets, tile_table)`` of a layer step (128-row tiles), built by one launch when the batch has neither; the
        launch clears the words of ``arrivals`` as well."""
        version = self._lens_version()
        call = (max_seq_len, left_padded, head_num, unit_kv_bytes, causal, version)
        found = self._last_tables       # the layers of a batch ask for the same ones in turn
        if found is not None and found[0] == call:
            self.order_current_stream()
            return found[1], found[2]
        first = tiles_first(self.batch_size * head_num, unit_kv_bytes, causal)
        if self.cu_seqlens is None or (version is None and self._mutable()):
            return self.row_offsets(max_seq_len, left_padded), self.tile_table(head_num, max_seq_len, unit_kv_bytes, causal=causal)
        off_key, tab_key = (max_seq_len, left_padded, version), (head_num, max_seq_len, first, version, 128)
        off, tab = self._row_offsets.get(off_key), self._tile_tables.get(tab_key)
        self.order_current_stream()     # behind the lookup: what it found may be another thread's, on another stream
        if off is not None and tab is not None:
            self._last_tables = (call, off, tab)
            return off, tab
        if off is not None or tab is not None:
            return self.row_offsets(max_seq_len, left_padded), self.tile_table(head_num, max_seq_len, unit_kv_bytes, causal=causal)
        off, tab, arrivals = _lib.front.layer_tables(self.lens, self.cu_seqlens, self.batch_size, max_seq_len, left_padded,
                                                     self.total, head_num, first)
        self.produced_on_current_stream()
        self._row_offsets = {k: o for k, o in self._row_offsets.items() if k[2] == version}
        self._row_offsets[off_key] = off
        self._tile_tables = {k: t for k, t in self._tile_tables.items() if k[3] == version}
        self._tile_tables[tab_key] = tab
        raw = _lib.stream_of(self.lens)
        if raw not in PER_THREAD_STREAMS and not torch.cuda.is_current_stream_capturing():
            self._arrivals[(max_seq_len, raw)] = arrivals
        return off, tab

    def arrivals(self, max_seq_len: int):
        """The meeting words of ``en_attn_fused_norm`` for launches on the current stream, or ``None``.  They belong to the
        stream they were cleared on, whose order keeps launches apart that share them; a handle that names another stream
        in every thread has none.  (A layer step does this lookup natively, where one launch is for it.)"""
        return self._arrivals.get((max_seq_len, _lib.stream_of(self.lens)))

    def _mutable(self) -> bool:
        """True when the lengths belong to a caller that may edit them in place (no prefix was computed from
        them, or they are the caller's own tensor)."""
        return self.cu_seqlens is None or self._source is self.lens


    def tile_table(self, head_num: int, q_seq_len: int, unit_kv_bytes: int = 1 << 30, query_tile: int = 128,
                   causal: Optional[bool] = None) -> torch.Tensor:
        """Workgroup order of the attention kernels for this batch (``en_attn_tile_table``): the query tiles the
        sequences really have, longest sequence first.  ``unit_kv_bytes`` is what one (batch, head) unit's K and V
        hold at full length and ``causal`` the mask of the call it is for (``None``: by ``unit_kv_bytes`` alone); they decide
        whether the last tiles of all units run first or a unit's tiles stay together (``tiles_first``).  ``query_tile`` is the
        tile height of the kernel that will read the table (128; 256 for the fused kernel's 64-queries-per-wave form).  Computed
        once per batch, head count, bucket, order and tile height by one small kernel and reused by every layer."""
        version = self._lens_version()
        call = (head_num, q_seq_len, unit_kv_bytes, query_tile, causal, version)
        found = self._last_table        # QK^T and PV of every layer ask for the same one
        if found is not None and found[0] == call:
            self.order_current_stream()
            return found[1]
        first = tiles_first(self.batch_size * int(head_num), int(unit_kv_bytes), causal)
        key = (int(head_num), int(q_seq_len), first, version, int(query_tile))
        tab = None if version is None and self._mutable() else self._tile_tables.get(key)
        self.order_current_stream()
        if tab is None:
            n = int(_lib.fn.en_attn_tile_table_elems(self.batch_size, key[0], key[1], key[4]))
            tab = torch.empty(max(n, 1), dtype=torch.int32, device=self.lens.device)
            with _lib.device_guard(self.lens):
                _lib.check(_lib.fn.en_attn_tile_table(self.lens.data_ptr(), self.batch_size, key[0], key[1], int(key[2]),
                                                      key[4], tab.data_ptr(), _lib.stream_of(self.lens)), "attn_tile_table")
                self.produced_on_current_stream()
            if version is not None or not self._mutable():
                # tables of older versions of the lengths can never be found again: drop them
                self._tile_tables = {k: t for k, t in self._tile_tables.items() if k[3] == version}
                self._tile_tables[key] = tab
        if version is not None or not self._mutable():
            self._last_table = (call, tab)
        return tab


    def tile_table_ptr(self, head_num: int, q_seq_len: int, unit_kv_bytes: int = 1 << 30, query_tile: int = 128,
                       causal: Optional[bool] = None):
        """Raw pointer of the workgroup order for an attention call, or ``None`` (the kernels then compute their
        own order) when this object lives for one call only: building the table is a launch of its own, which pays
        off when every layer reuses it, not when every call would rebuild it (lengths given as Python lists or as
        tensors made under ``torch.inference_mode()`` are never cached -- pass a ``SeqInfo`` to keep one)."""
        if self.ephemeral:
            return None
        return self.tile_table(head_num, q_seq_len, unit_kv_bytes, query_tile, causal).data_ptr()


_cache: "OrderedDict[tuple, SeqInfo]" = OrderedDict()


def build_seq_info(seq_lens, batch_size: int, device=None, total: Optional[int] = None) -> SeqInfo:
    """Runs the prefix-sum kernel.  ``seq_lens`` is a CUDA int32/int64 tensor, or
    a CPU tensor / list (then the total is known without a sync)."""
    if not isinstance(seq_lens, torch.Tensor):
        seq_lens = torch.as_tensor(list(seq_lens), dtype=torch.int32)
    if seq_lens.dtype not in (torch.int32, torch.int64):
        raise RuntimeError(f"seq_lens must be int32 or int64, got {seq_lens.dtype}")
    if seq_lens.numel() < batch_size:
        raise RuntimeError(f"seq_lens has {seq_lens.numel()} entries, batch_size is {batch_size}")
    source = seq_lens
    if not seq_lens.is_cuda:
        if total is None:
            total = int(seq_lens[:batch_size].sum())
        if device is None:
            device = torch.device("cuda", torch.cuda.current_device())
        seq_lens = seq_lens.to(device, non_blocking=False)
    cu, lens32 = _lib.front.prefix_sum(seq_lens.contiguous(), batch_size)
    info = SeqInfo(lens32, cu, batch_size, total, source)
    info.produced_on_current_stream()
    return info


def seq_info(seq_lens, batch_size: int, device=None) -> SeqInfo:
    """Returns the (cached) SeqInfo for ``seq_lens``.

    A SeqInfo passes through unchanged.  Tensors are cached by identity and
    version counter, and the cache holds a reference to the tensor so its
    storage cannot be recycled under a stale entry; in-place edits through torch
    bump the version and miss the cache.  Tensors created inside
    ``torch.inference_mode()`` (the reference worker runs the whole forward there,
    energonai/worker.py:79) carry no version counter, so an edit could not be
    noticed: they are never cached and the prefix kernel runs on every call.
    A cached entry used on another stream than the one its kernels were launched
    on makes that stream wait for them first.
    """
    if isinstance(seq_lens, SeqInfo):
        if seq_lens.batch_size != batch_size:
            raise RuntimeError(f"SeqInfo was built for batch {seq_lens.batch_size}, call passes {batch_size}")
        seq_lens.order_current_stream()
        return seq_lens
    if not isinstance(seq_lens, torch.Tensor) or torch.is_inference(seq_lens):
        info = build_seq_info(seq_lens, batch_size, device)
        info.ephemeral = True
        return info
    key = (id(seq_lens), seq_lens._version, seq_lens.data_ptr(), batch_size, str(device))
    hit = _cache.get(key)
    if hit is not None and hit._source is seq_lens:
        _cache.move_to_end(key)
        hit.order_current_stream()
        return hit
    info = build_seq_info(seq_lens, batch_size, device)
    _cache[key] = info
    while len(_cache) > _CACHE_SIZE:
        _cache.popitem(last=False)
    return info


def clear_cache() -> None:
    _cache.clear()
