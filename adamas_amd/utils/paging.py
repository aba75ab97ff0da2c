"""Device-resident paging state for the Adamas decode path on MI355X.

What the reference keeps as Python lists that are turned into fresh device tensors on every forward
(adamas/utils/controller.py:82-131, adamas/utils/kv_cache.py:65-135) lives here permanently in HBM:

* `PagePool`      - the KV pages and the 2-bit code pages of ALL layers, addressed by one physical
                    page id, plus the free list.
* `PagedSequences`- for `batch` sequences: a fixed-stride int32 page table, its indptr and the int32
                    sequence lengths, all on the device and updated in place (only the entries that
                    change are written), so a decode step uploads a few bytes, not the whole table.

Token-level generalisation of the reference layout: codes are per token and share the KV page
table - token t of a sequence sits in physical page table[t // page_size], slot t % page_size, in
both pools.  (The reference gives the codes a second page list that is only consistent at page_size 1:
controller.py:30-39 with kv_cache.py:88 divides the capacity by page_size twice.)
"""
from __future__ import annotations

from operator import index
from typing import Iterable, List, Optional, Sequence

import torch

from .. import _lib

CODE_WORDS = 16  # uint16 words of packed 2-bit code per (token, head) at head_dim 128


class TensorLayout:
    """Layout tags of the reference (adamas/utils/utils.py:1-5): NHD pages are
    [2, page_size, heads, head_dim], HND pages [2, heads, page_size, head_dim].  The reference only
    instantiates NHD; the HIP kernels take either (NHD is the fast one for dense attention)."""
    NHD = 0
    HND = 1
    FORMAT2STR = {0: "NHD", 1: "HND"}


def _row_address(t: torch.Tensor, i: int) -> int:
    """t[i].data_ptr() without making the view, as a Python int whatever kind of integer i is."""
    try:
        i = index(i)
    except TypeError:   # (a slice or the like)
        return t[i].data_ptr()
    n = t.shape[0]
    if not -n <= i < n:
        raise IndexError(f"index {i} is out of bounds for dimension 0 with size {n}")
    return t.data_ptr() + (i + n if i < 0 else i) * t.stride(0) * t.element_size()


class PagePool:
    """Physical pages of every layer.

    kv    : [layers, pages, 2, page_size, heads, head_dim]  (0 = K, 1 = V), or
            [layers, pages, 2, heads, page_size, head_dim] with layout = TensorLayout.HND
    codes : [layers, pages, page_size, heads, 16] int16 (raw 2-bit code words), in both layouts
    `num_heads` counts key/value heads (fewer than the query heads with grouped-query attention).
    """

    def __init__(self, num_layers: int, num_heads: int, head_dim: int, page_size: int,
                 num_pages: int, dtype: torch.dtype, device, page_order: Optional[Iterable[int]] = None,
                 layout: int = TensorLayout.NHD):
        if num_pages <= 0 or page_size <= 0:
            raise ValueError("num_pages and page_size must be positive")
        self.page_size = page_size
        self.num_pages = num_pages
        if layout not in (TensorLayout.NHD, TensorLayout.HND):
            raise ValueError("layout must be TensorLayout.NHD or TensorLayout.HND")
        self.layout = layout
        page_shape = ((2, page_size, num_heads, head_dim) if layout == TensorLayout.NHD
                      else (2, num_heads, page_size, head_dim))
        self.kv = torch.empty((num_layers, num_pages) + page_shape, dtype=dtype, device=device)
        self.codes = torch.zeros((num_layers, num_pages, page_size, num_heads, head_dim // 8),
                                 dtype=torch.int16, device=device)
        order = list(range(num_pages)) if page_order is None else [int(p) for p in page_order]
        if sorted(order) != list(range(num_pages)):
            raise ValueError("page_order must be a permutation of range(num_pages)")
        self._free: List[int] = order[::-1]  # pop() hands pages out in `order`
        self._busy = set()

    def kv_address(self, layer: int) -> int:
        """Address of kv[layer] (1 us less than through a view of it)."""
        return _row_address(self.kv, layer)

    def codes_address(self, layer: int) -> int:
        """Address of codes[layer]."""
        return _row_address(self.codes, layer)

    @property
    def num_free_pages(self) -> int:
        return len(self._free)

    def take(self) -> int:
        if not self._free:
            # same exception type the reference raises on exhaustion (set.pop() in kv_cache.py:56-58)
            raise KeyError("page pool exhausted")
        p = self._free.pop()
        self._busy.add(p)
        return p

    def give_back(self, pages: Iterable[int]) -> None:
        for p in pages:
            if p not in self._busy:
                raise ValueError(f"page {p} is not in use")
            self._busy.remove(p)
            self._free.append(p)


class PagedSequences:
    """Page tables and lengths of `batch` sequences, mirrored on the device."""

    def __init__(self, pool: PagePool, batch: int, max_seq_len: int, device):
        self.pool = pool
        self.batch = batch
        self.max_pages = (max_seq_len + pool.page_size - 1) // pool.page_size
        self.max_seq_len = max_seq_len
        self.pages: List[List[int]] = [[] for _ in range(batch)]
        self.lengths: List[int] = [0] * batch
        self.device = device
        # fixed stride per sequence => the indptr never changes
        self._table_dev = torch.zeros(batch * self.max_pages, dtype=torch.int32, device=device)
        self.indptr_dev = (torch.arange(batch + 1, dtype=torch.int32) * self.max_pages).to(device)
        self._seq_lens_dev = torch.zeros(batch, dtype=torch.int32, device=device)
        # Lengths and page ids are written by a launch that the host does not wait for, while everything that reads them
        # is launched by this package's operators on the stream of that launch.  That is the default stream, and the
        # tables must have been allocated there: it cannot be captured, so the host can wait for what was written there
        # at any time (HIP refuses to wait for a stream that is being captured), and the tables' memory is not handed to
        # another before a write to it is done.  The first operator on another stream or in a graph (which is replayed
        # on whatever stream), and the first look from outside (a tensor or an address once handed out is used at any
        # time on any stream), wait for what is written and end that for good: from then on the host waits for every
        # write, and no stream can be too early.
        self._host_waits = not (self._table_dev.is_cuda and _lib.current_stream(self._table_dev.get_device()) == 0)
        self._writer: Optional[int] = None    # the default stream once it has a write that the host did not wait for

    @property
    def table_dev(self) -> torch.Tensor:
        """The page table [batch * max_pages] int32.  From the first look at it or at seq_lens_dev on, the host waits
        for every write, so that who holds them may read them on any stream, as soon as the call that grew a
        sequence has returned."""
        self._end_writes_without_waiting()
        return self._table_dev

    @property
    def seq_lens_dev(self) -> torch.Tensor:
        """The lengths [batch] int32 (see table_dev)."""
        self._end_writes_without_waiting()
        return self._seq_lens_dev

    @table_dev.setter
    def table_dev(self, table: torch.Tensor) -> None:
        self._end_writes_without_waiting()
        self._table_dev = table

    @seq_lens_dev.setter
    def seq_lens_dev(self, lengths: torch.Tensor) -> None:
        self._end_writes_without_waiting()
        self._seq_lens_dev = lengths

    def launch_addresses(self, stream: int):
        """(page table, indptr, lengths) on the device, for a launch on `stream` now; not to be kept."""
        if stream and not self._host_waits:   # (no capture is on the default stream)
            self._end_writes_without_waiting()
        return self._table_dev.data_ptr(), self.indptr_dev.data_ptr(), self._seq_lens_dev.data_ptr()

    def launch_table_address(self, stream: int, b: int = 0) -> int:
        """The page table of sequence b alone."""
        if stream and not self._host_waits:
            self._end_writes_without_waiting()
        return self._table_dev.data_ptr() + 4 * b * self.max_pages

    def launch_table(self) -> torch.Tensor:
        """table_dev for operators launched on the current stream now; not to be kept."""
        if not self._host_waits:
            self._note_use()
        return self._table_dev

    def _end_writes_without_waiting(self) -> None:
        if self._host_waits:
            return
        if self._writer is not None:
            _lib.wait_default_stream(self._table_dev.get_device())   # (also while another stream is captured)
            self._writer = None
        self._host_waits = True

    def _note_use(self) -> None:
        if _lib.current_stream(self._table_dev.get_device()) != 0:
            self._end_writes_without_waiting()

    def _write(self, dst: torch.Tensor, start: int, values: List[int]) -> None:
        """dst[start:] = values, without waiting for it where that is safe (see __init__): a decode loop that
        waits for the copy of one length after every token leaves the GPU idle while the host catches up
        (2000 + 24 tokens through three layers 11.47 -> 10.76 ms)."""
        n = len(values)
        if not self._host_waits:
            self._note_use()   # (ahead of any write from another stream)
        if self._host_waits or n > _lib.MAX_WORDS or dst.get_device() != torch.cuda.current_device():
            dst[start:start + n] = torch.tensor(values, dtype=torch.int32)
            return
        _lib.write_words(dst.data_ptr() + 4 * start, values, 0)
        self._writer = 0

    def __getstate__(self):   # (for a copy or another process)
        if self._writer is not None:
            _lib.wait_default_stream(self._table_dev.get_device())
        return dict(self.__dict__, _writer=None, _host_waits=True)

    def reserve(self, new_tokens: Sequence[int]) -> List[int]:
        """Grow sequence b by new_tokens[b] tokens; returns the number of new pages per sequence."""
        if len(new_tokens) != self.batch:
            raise ValueError("one token count per sequence expected")
        added = []
        ps = self.pool.page_size
        for b, n in enumerate(new_tokens):
            if n < 0:
                raise ValueError("negative token count")
            target = self.lengths[b] + n
            if target > self.max_seq_len:
                raise ValueError(f"sequence {b} would exceed max_seq_len {self.max_seq_len}")
            need = (target + ps - 1) // ps - len(self.pages[b])
            fresh = [self.pool.take() for _ in range(need)]
            if fresh:
                start = b * self.max_pages + len(self.pages[b])
                self._write(self._table_dev, start, fresh)
                self.pages[b].extend(fresh)
            self.lengths[b] = target
            added.append(need)
        self._write(self._seq_lens_dev, 0, self.lengths)
        return added

    def reserve_pages_ahead(self, extra_tokens: int) -> None:
        """Allocate (and publish in the device table) the pages the next `extra_tokens` tokens of
        every sequence will need, without changing any length: afterwards a sequence can grow by
        bumping its device-side length only, e.g. from inside a captured HIP graph."""
        ps = self.pool.page_size
        for b in range(self.batch):
            target = self.lengths[b] + extra_tokens
            if target > self.max_seq_len:
                raise ValueError(f"sequence {b} would exceed max_seq_len {self.max_seq_len}")
            need = (target + ps - 1) // ps - len(self.pages[b])
            if need > 0:
                fresh = [self.pool.take() for _ in range(need)]
                start = b * self.max_pages + len(self.pages[b])
                self._write(self._table_dev, start, fresh)
                self.pages[b].extend(fresh)

    def advance_on_device(self) -> None:
        """One more token for every sequence, on the device only (graph-capturable)."""
        if not self._host_waits:
            self._note_use()
        self._seq_lens_dev.add_(1)

    def note_advanced(self, n_tokens: int) -> None:
        """Bring the host-side lengths in line after `n_tokens` device-side advances."""
        for b in range(self.batch):
            self.lengths[b] += n_tokens
            if self.lengths[b] > len(self.pages[b]) * self.pool.page_size:
                raise RuntimeError("device-side advance ran past the reserved pages")

    def release(self) -> None:
        for b in range(self.batch):
            self.pool.give_back(self.pages[b])
            self.pages[b] = []
            self.lengths[b] = 0
        if not self._host_waits:
            self._note_use()
        self._seq_lens_dev.zero_()

    def table_ptr(self, b: int) -> int:
        """Device address of the first page-table entry of sequence b (see table_dev)."""
        return self.table_dev.data_ptr() + 4 * b * self.max_pages


class KvCache:
    """View of one sequence with the field names the reference's callers read
    (`iController.kv_cache.seqlen`, `.last_page_len`, `.indicies`, `.buf_layer`; kv_cache.py:98-120)."""

    def __init__(self, seqs: PagedSequences, b: int = 0, codes: bool = False):
        self._seqs, self._b, self._codes = seqs, b, codes

    @property
    def pool(self) -> PagePool:
        return self._seqs.pool

    @property
    def seqlen(self) -> int:
        return self._seqs.lengths[self._b]

    @property
    def last_page_len(self) -> int:
        return (self.seqlen - 1) % self._seqs.pool.page_size + 1

    @property
    def indicies(self) -> List[int]:  # (sic) spelling of the reference
        return self._seqs.pages[self._b]

    def buf_layer(self, layer_idx: int) -> torch.Tensor:
        buf = self._seqs.pool.codes if self._codes else self._seqs.pool.kv
        if not 0 <= layer_idx < buf.shape[0]:
            raise IndexError("layer index out of range")
        return buf[layer_idx]
