"""CPU-side checks: the C-ABI library loads and exports what include/adamas_hip.h declares, argument
validation returns the documented codes before anything is launched, and the host-side paging and
controller logic behaves like the reference's controller."""
import ctypes
import os
import re

import numpy as np
import pytest
import torch

import adamas_amd.utils as U
from adamas_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "adamas_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(adamas_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = _lib.load()
    names = _declared_symbols()
    assert len(names) >= 15
    for n in names:
        assert hasattr(lib, n), n
    assert set(names) == set(_lib.EXPORTED_SYMBOLS)
    assert lib.adamas_version() >= 100


def _declared_prototypes():
    """name -> list of parameter declarations, parsed from the header."""
    text = open(os.path.join(ROOT, "include", "adamas_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    protos = {}
    for m in re.finditer(r"\b(adamas_[a-z0-9_]+)\s*\(([^;{]*?)\)\s*;", text, flags=re.S):
        params = [p.strip() for p in m.group(2).replace("\n", " ").split(",")]
        protos[m.group(1)] = [] if params == ["void"] else params
    return protos


def test_ctypes_signatures_match_the_header():
    """Every prototype of the header against the ctypes table: same number of arguments, pointers
    bound as pointers, 64-bit integers as 64-bit, floats as floats."""
    import ctypes as C
    protos = _declared_prototypes()
    assert set(protos) == set(_lib.EXPORTED_SYMBOLS)
    for name, params in protos.items():
        _, argtypes = _lib._SIGNATURES[name]
        assert len(argtypes) == len(params), (name, len(argtypes), len(params))
        for decl, ct in zip(params, argtypes):
            if "*" in decl or "adamas_stream_t" in decl:
                assert ct in (C.c_void_p, C.c_char_p), (name, decl, ct)
            elif decl.startswith("float"):
                assert ct is C.c_float, (name, decl, ct)
            elif decl.startswith(("int64_t", "uint64_t", "size_t")):
                assert C.sizeof(ct) == 8, (name, decl, ct)
            else:
                assert decl.startswith(("uint32_t", "int32_t", "int ")), (name, decl)
                assert C.sizeof(ct) == 4, (name, decl, ct)


def test_argument_errors_are_reported_before_any_launch():
    lib = _lib.load()
    assert lib.adamas_hadamard(None, None, 0, 1.0, None) == 0                       # empty: no-op
    assert lib.adamas_hadamard(None, None, 4, 1.0, None) == -1                      # BADARG
    assert lib.adamas_hadamard(2, 2, 4, 1.0, None) == -4                            # ALIGN
    assert lib.adamas_pack_2bit(None, None, 3, None) == -1
    assert lib.adamas_append_decode(*([None] * 10), 1, 32, 32, 128, 16, 1.0, 0, None) == -1
    assert lib.adamas_append_prefill(16, 16, None, 4, 0, 16, 16, 16, 1, 32, 64, 16, 1.0, 0, None) == -2
    assert lib.adamas_append_prefill(16, 16, None, 40, 0, 16, 16, 16, 1, 32, 128, 16, 1.0, 0, None) == -1
    assert lib.adamas_estimate(16, 16, 16, 16, 16, 16, 8, 8, 0, 1, 0, 24, 16, 100, None) == -2    # no heads
    assert lib.adamas_estimate(16, 16, 16, 16, 16, 16, 8, 8, 0, 1, 32, 5, 16, 100, None) == -2    # 32 % kv heads
    assert lib.adamas_estimate(16, 16, 16, 16, 16, 16, 8, 8, 7, 1, 32, 32, 16, 100, None) == -1   # format
    assert lib.adamas_estimate(16, 16, 16, 16, 16, 16, 8, 8, 0, 1, 32, 8, 16, 1, None) == 0      # nothing to do
    assert lib.adamas_topk(None, 8, 8, None, 1, 0, None, 0, 1, 4, None, None, 4, 0, None, 0, None) == -1
    assert lib.adamas_topk(16, 8, 8, None, 1, 0, None, 0, 1, 4, 16, None, 2, 0, None, 0, None) == -1   # stride < k
    assert lib.adamas_topk(16, 40000, 40000, None, 1, 0, None, 0, 1, 4, 16, None, 4, 0, None, 0, None) == -3  # reduction levels need a workspace
    assert lib.adamas_topk_workspace_bytes(32, 131071, 255) >= 32 * 32 * 255 * 8
    # two-level integer path: 64 chunks x (128 candidates x 8 B + 512 B of histogram) per row
    assert lib.adamas_topk_workspace_bytes(32, 32767, 127) == 32 * 64 * (128 * 8 + 512)
    # k above 255: one row of 512 16-bit counts per chunk of 1024 keys
    assert lib.adamas_topk_workspace_bytes(32, 32767, 300) == 32 * 32 * 1024
    # short rows, k <= 255: 8 chunks x 128 candidates x 8 B per row (short candidate lists)
    assert lib.adamas_topk_workspace_bytes(32, 4096, 127) == 32 * 8 * 128 * 8
    assert lib.adamas_topk_workspace_bytes(32, 4096, 300) == 256       # one launch, no workspace
    assert lib.adamas_sparse_decode(16, 16, 16, 16, 16, None, 0, 0, 16, None, 0, 1, 32, 32, 64, 16, 0.1, 10, None) == -2
    # several splits without a workspace
    assert lib.adamas_sparse_decode(16, 16, 16, 16, 16, None, 0, 0, 16, None, 0, 1, 32, 8, 128, 16, 0.1, 5000, None) == -3
    assert lib.adamas_decode_step(*([16] * 7), 128, 16, None, None, 0, 1, 32, 32, 128, 16, 0.1, 100, 0, None) == -1
    assert lib.adamas_step_fused_supported(1, 32, 32768, 128) == 1
    assert lib.adamas_step_fused_supported(1, 32, 131072, 256) == 1       # 64 chunks of 2048 tokens
    assert lib.adamas_step_fused_supported(1, 32, 262144, 256) == 0       # too many candidate slots
    assert lib.adamas_step_fused_supported(1, 32, 4096, 1024) == 0        # budget beyond 256
    assert lib.adamas_step_fused_supported(1, 40, 32768, 128) == 1        # any multiple of 8 heads
    assert lib.adamas_step_fused_supported(1, 36, 32768, 128) == 0
    assert lib.adamas_step_candidates(16, 16, 16, 16, 16, 1024, 256, 1 << 30, 1, 32, 32, 16, 4096, 0, None) == -2
    assert lib.adamas_step_candidates(16, 16, 16, None, 16, 128, 256, 1 << 30, 1, 32, 32, 16, 4096, 0, None) == -1
    assert lib.adamas_step_attend(16, 16, 16, 16, 16, 16, 128, 16, None, None, 0, 1, 32, 32, 128, 16, 0.1, 4096, 0, None) == -1
    assert "workspace" in _lib.error_string(-3)
    with pytest.raises(RuntimeError):
        _lib.check(-2, "x")


def test_workspace_bytes_grows_with_sizes():
    lib = _lib.load()
    a = lib.adamas_workspace_bytes(1, 32, 4096, 64)
    b = lib.adamas_workspace_bytes(1, 32, 32768, 128)
    c = lib.adamas_workspace_bytes(16, 32, 32768, 128)
    assert 0 < a < b < c
    assert a % 256 == 0


def test_controller_workspace_covers_every_size_it_is_asked_for():
    """The size the library asks for is monotonic neither in the budget nor in the length: a
    controller that has served one size must still hand out enough bytes for the next, whatever
    the order (budget 300 then 256; 32832 tokens then 32769), and a sequence or a dense budget that
    grows token by token must not reallocate at every token."""
    lib = _lib.load()
    assert lib.adamas_workspace_bytes(1, 32, 32769, 128) > lib.adamas_workspace_bytes(1, 32, 32832, 128)
    c = _ctrl(max_seq_len=32832, num_layers=1)
    c.prepare_hadamard(32769)
    for budget in (32769, 128, 300, 256, 200, 128, 4096, 129):
        ws = c.workspace(budget)
        assert ws.numel() >= lib.adamas_workspace_bytes(1, 32, 32769, budget), budget
    seen = set()
    for _ in range(40):
        c.prepare_hadamard(1)
        n = c.max_len_now
        for budget in (n, 128):       # the dense layers, then the sparse ones, as a model alternates
            ws = c.workspace(budget)
            assert ws.numel() >= lib.adamas_workspace_bytes(1, 32, n, budget)
            seen.add(ws.data_ptr())
    assert len(seen) <= 2


def _ctrl(**kw):
    args = dict(num_layers=2, num_heads=32, head_dim=128, page_size=16, page_budget=64,
                max_seq_len=256, dtype=torch.float16, device="cpu")
    args.update(kw)
    return U.InferenceController(**args)


def test_controller_paging_and_budget_regime():
    c = _ctrl()
    assert not c.need_estimate()                      # before any begin_forward
    c.prepare_hadamard(40)                            # prefill of 40 tokens -> 3 pages
    assert c.kv_cache.seqlen == 40 and len(c.kv_cache.indicies) == 3
    assert c.kv_cache.last_page_len == 8 and c.hadamard_cache.seqlen == 40
    assert c.seq_lens.tolist() == [40]
    assert c.kv_indices_with_last[:3].tolist() == c.kv_cache.indicies
    c.begin_forward(40)
    c.end_forward()
    c.prepare_hadamard(1)
    c.begin_forward(1)
    assert c.inference_page_budget == 41 and not c.need_estimate()   # 41 tokens <= budget 64
    for _ in range(30):
        c.prepare_hadamard(1)
    c.begin_forward(1)
    assert c.inference_page_budget == 64 and c.need_estimate()
    assert c.topk_dindices_buffer.shape == (32, 63) and c.topk_dindices_buffer.dtype == torch.int32
    c.set_page_budget(1 << 20)                        # the two dense layers of the model
    c.begin_forward(1, updateTensor=False)
    assert not c.need_estimate()
    assert c.kv_indices_without_last is U.ALL_PAST_TOKENS
    c.clean_states()
    assert c.kv_cache.seqlen == 0 and c.pool.num_free_pages == 16


def test_controller_errors():
    with pytest.raises(RuntimeError):
        _ctrl(dtype=torch.float32)                    # fp16 (as the reference) and bf16 only
    with pytest.raises(RuntimeError):
        _ctrl(head_dim=64)
    with pytest.raises(RuntimeError):
        _ctrl(num_heads=12)
    c = _ctrl(max_seq_len=32)
    with pytest.raises(ValueError):
        c.prepare_hadamard(33)                        # beyond max_seq_len
    c.prepare_hadamard(1)
    with pytest.raises(AssertionError):
        c.begin_forward(1)                            # decode needs a past token
    with pytest.raises(ValueError):
        _ctrl(page_order=[0, 0, 1])


def test_pool_exhaustion_raises_keyerror_and_pages_are_reused():
    pool = U.PagePool(1, 32, 128, 16, 2, torch.float16, "cpu", page_order=[1, 0])
    assert pool.take() == 1 and pool.take() == 0
    with pytest.raises(KeyError):
        pool.take()
    pool.give_back([0])
    assert pool.take() == 0
    with pytest.raises(ValueError):
        pool.give_back([5])


def test_batched_sequences_fixed_stride_tables():
    c = _ctrl(batch_size=3, max_seq_len=64, page_order=list(range(11, -1, -1)))
    c.prepare_hadamard([5, 20, 64])
    assert c.seq_lens.tolist() == [5, 20, 64]
    assert c.kv_indptr_for_append.tolist() == [0, 4, 8, 12]
    assert [len(p) for p in c.seqs.pages] == [1, 2, 4]
    t = c.kv_indices_with_last.tolist()
    assert t[0] == 11 and t[4:6] == [10, 9] and t[8:12] == [8, 7, 6, 5]
    assert c.max_len_now == 64 and c.min_len_now == 5


def test_graph_decode_reserves_pages_ahead_and_tracks_lengths():
    """The HIP-graph decode loop: pages of the coming tokens are reserved up front, the lengths then
    advance on the device only, and the host catches up afterwards."""
    c = _ctrl(batch_size=2, max_seq_len=64)
    c.prepare_hadamard([10, 33])                       # 1 and 3 pages of 16 tokens
    free0 = c.pool.num_free_pages
    c.begin_graph_decode(20)                           # up to 30 and 53 tokens: 2 and 4 pages
    assert [len(p) for p in c.seqs.pages] == [2, 4]
    assert c.pool.num_free_pages == free0 - 2
    t = c.kv_indices_with_last.tolist()
    assert t[0:2] == c.seqs.pages[0] and t[4:8] == c.seqs.pages[1]
    assert c.max_len_now == 33 + 20                    # the bound the launches are sized with
    for _ in range(7):
        c.advance_on_device()
    assert c.seq_lens.tolist() == [17, 40]             # device lengths moved, host lengths did not
    assert c.seqs.lengths == [10, 33]
    c.end_graph_decode(7)
    assert c.seqs.lengths == [17, 40] and c.max_len_now == 40
    c.prepare_hadamard(1)                              # the eager path continues from there
    assert c.seq_lens.tolist() == [18, 41] and [len(p) for p in c.seqs.pages] == [2, 4]
    with pytest.raises(ValueError):
        c.begin_graph_decode(64)                       # beyond max_seq_len
    c.clean_states()
    assert c.pool.num_free_pages == 8 and c.seq_lens.tolist() == [0, 0]
    c.prepare_hadamard([3, 3])
    c.begin_graph_decode(4)
    with pytest.raises(RuntimeError):
        c.end_graph_decode(40)                         # more tokens than pages were reserved for


def test_ops_reject_cpu_tensors():
    c = _ctrl()
    c.prepare_hadamard(4)
    x = torch.zeros(4, 32, 128, dtype=torch.float16)
    with pytest.raises(RuntimeError):
        U.append_kvh(x, x, x, c, 0)
    with pytest.raises(RuntimeError):
        U.hadamard_transform(x)


def test_step_plan_covers_every_sequence_with_balanced_chunks():
    """The geometry the two-launch step derives from the sizes of a call (adamas_step_plan): the
    chunks tile the past tokens of the longest sequence in 16-token units, differ by at most one
    unit for a single sequence, fit the workgroup (at most four passes of 512 tokens) and the
    second launch (at most 64 chunks, 1024 candidate slots per head for one sequence, 2048 for a
    batch; a power of two of 8 .. 256 slots per chunk, never more than the budget needs)."""
    lens = sorted(set([2, 3, 17, 18, 33, 511, 512, 513, 514, 1000, 4096, 4097, 8192, 8193, 16384, 16385,
                       16400, 20000, 32767, 32768, 32769, 32784, 32785, 33024, 36864, 40000, 65536, 65537,
                       100000, 131056, 131072] + list(range(2, 140000, 3571))))
    for batch in (1, 2, 16):
        for heads in (32, 40, 64):
            for budget in (2, 16, 64, 128, 200, 256):
                for L in lens:
                    p = _lib.step_plan(batch, heads, L, budget)
                    where = (batch, heads, L, budget, p)
                    if not p["ok"]:
                        assert L - 1 > 64 * 2048 or (batch > 1 and L - 1 > 64 * 2048), where
                        continue
                    units = (L - 1 + 15) // 16
                    assert 1 <= p["chunks"] <= 64, where
                    assert p["heads"] in (4, 8) and heads % p["heads"] == 0, where
                    # the chunks cover all units: a single sequence is tiled exactly, a batch is
                    # covered by fixed-size chunks
                    total = p["chunks"] * p["units_q"] + p["units_r"]
                    if batch == 1 and p["units_r"] == 0 and p["units_q"] % 32 == 0 and p["chunks"] * p["units_q"] > units:
                        assert total - units < p["units_q"], where      # fixed 512-token chunks
                    elif batch == 1:
                        assert total == units or total - units < p["units_q"], where
                    else:
                        assert total >= units and p["units_r"] == 0, where
                    assert p["units_r"] < p["chunks"], where
                    longest = p["units_q"] + (1 if p["units_r"] else 0)
                    assert 1 <= p["passes"] <= 4 and longest <= 32 * p["passes"], where
                    assert longest > 32 * (p["passes"] - 1), where
                    assert p["partial"] == int(p["units_r"] != 0 or p["units_q"] % 32 != 0), where
                    kc = p["kc"]
                    assert kc in (8, 16, 32, 64, 128, 256), where
                    assert p["chunks"] * kc <= (1024 if batch == 1 else 2048) or kc == 8, where
                    # never more slots than the budget can use (rounded up to a power of two, at least 8)
                    need = 8
                    while need < budget - 1:
                        need *= 2
                    assert kc <= need, where
    # what the headline workloads get
    assert _lib.step_plan(1, 32, 32768, 128) == {"ok": 1, "heads": 8, "chunks": 64, "units_q": 32, "units_r": 0,
                                                 "passes": 1, "partial": 0, "kc": 16}
    p = _lib.step_plan(1, 32, 33024, 128)
    assert (p["chunks"], p["units_q"], p["units_r"], p["passes"], p["partial"]) == (64, 32, 16, 2, 1)
    assert _lib.step_plan(1, 32, 131072, 256)["passes"] == 4
    assert _lib.step_plan(16, 32, 32768, 128)["kc"] == 32
    assert _lib.step_plan(1, 32, 32768, 1024)["ok"] == 0       # budgets above 256 take the histogram path


def _prefill_plan_reference(n_new, past, heads, kv_heads):
    """The number of token ranges adamas_prefill_attention cuts the longest row block into, found with a
    search through all CUs of a head for every workgroup: slow, and plain to see."""
    group = heads // kv_heads
    rows = n_new * group
    blocks = -(-rows // 256)
    tiles = [(past + (min((b + 1) * 256, rows) - 1) // group) // 64 + 1 for b in range(blocks)]
    if blocks * kv_heads >= 1024:
        return 1
    slots = max(1, 256 // kv_heads)

    def cost(split):
        busy, moved = [0] * slots, 0.0
        for first in range(0, tiles[-1], split):
            for t in reversed(tiles):
                if t <= first:
                    break
                busy[busy.index(min(busy))] += min(t - first, split) + 2
                moved += 2.0 * 256 * 132 * 4 * kv_heads if t > split else 0.0
        return max(busy) + (3 + moved / 8.75e6 if split < tiles[-1] else 0.0)

    best, split = cost(tiles[-1]), tiles[-1]
    for per_slot in (1, 2, 3):
        lo = next((m for m in range(1, tiles[-1]) if sum(-(-t // m) for t in tiles) <= per_slot * slots), tiles[-1])
        if lo < tiles[-1] and cost(lo) < best:
            best, split = cost(lo), lo
    return -(-tiles[-1] // split)


@pytest.mark.parametrize("heads,kv_heads", [(32, 32), (32, 8), (32, 1), (24, 8), (512, 512)])
@pytest.mark.parametrize("n_new,past", [(1, 0), (64, 16000), (300, 900), (257, 63), (1000, 3000), (2000, 0),
                                        (300, 553), (500, 300)])    # (calls that may get workgroups of four waves)
def test_prefill_plan(heads, kv_heads, n_new, past):
    n_split = _prefill_plan_reference(n_new, past, heads, kv_heads)
    want = 0 if n_split == 1 else n_split * n_new * heads * 132 * 4
    assert _lib.load().adamas_prefill_workspace_bytes(n_new, past, heads, kv_heads) == want


@pytest.mark.parametrize("args", [(2000, 14003, 32, 1), (4000, 16000, 32, 1), (16000, 0, 16, 1)])
def test_prefill_plan_is_quick(args):
    """A few hundred workgroups are dealt out up to four times, in up to 0.5 units of time (a sum over
    10000 numbers in Python); a search through 256 CUs for each of them took 2.4 to 2.9."""
    import time
    lib = _lib.load()

    def best(call):
        times = []
        for _ in range(50):
            t = time.perf_counter()
            call()
            times.append(time.perf_counter() - t)
        return min(times)

    unit = best(lambda: sum(range(10000)))
    assert best(lambda: lib.adamas_prefill_workspace_bytes(*args)) < 1.2 * unit


def test_codes_cached_hint():
    """The controller's hint goes by what a token reads in all layers and sequences: codes, 32 bytes per token
    and key/value head, and here no selected rows."""
    from adamas_amd.utils.controller import CODES_CACHED_BYTES
    c = _ctrl(num_layers=3, batch_size=2)
    c.seqs.lengths[:] = [5, 7]
    edge = CODES_CACHED_BYTES // (3 * 2 * 32 * 32)
    c._len_bound = edge
    assert c.codes_hint == _lib.F_CODES_CACHED
    c._len_bound = edge + 1
    assert c.codes_hint == 0
    lib = _lib.load()    # a hint for the step and its two halves, not for the operators
    step = [16] * 7 + [8, 16, None, 256, 1 << 40, 1, 32, 32, 64, 16, 1.0, 100, 8]   # head_dim 64: refused later
    assert lib.adamas_decode_step_f(*step, _lib.F_CODES_CACHED, None) == -2
    assert lib.adamas_decode_step_f(*step, 2 * _lib.F_CODES_CACHED, None) == -1
    assert lib.adamas_sparse_decode_f(*[16] * 5, None, 0, 0, 16, None, 0, 1, 32, 32, 64, 16, 1.0, 100,
                                      _lib.F_CODES_CACHED, None) == -1


@pytest.mark.parametrize("kv_heads", [32, 8])
def test_codes_cached_hint_of_a_ragged_batch_with_a_budget(kv_heads):
    """Eager steps count the tokens that are there, and with them the selected K and V rows of every query head."""
    from adamas_amd.utils.controller import CODES_CACHED_BYTES
    layers, budget = 40, 100
    c = _ctrl(num_layers=layers, batch_size=3, num_kv_heads=kv_heads)
    rows = layers * 3 * budget * 32 * 2 * 256
    edge = (CODES_CACHED_BYTES - rows) // (layers * kv_heads * 32)     # tokens
    c.inference_page_budget = budget
    for tokens, want in ((edge, _lib.F_CODES_CACHED), (edge + 1, 0)):
        c.seqs.lengths[:] = [tokens - 900, 700, 200]
        assert c._len_bound is None and c.codes_hint == want
    c.inference_page_budget = None
    assert c.codes_hint == _lib.F_CODES_CACHED
    c.seqs.lengths[0] = CODES_CACHED_BYTES // (layers * kv_heads * 32) - 899
    assert c.codes_hint == 0


def test_current_stream_without_the_private_names(monkeypatch):
    """Falls back to the stream object where torch lacks them."""
    class Stream:
        cuda_stream = 77
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream")
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: Stream)
    assert _lib.current_stream() == 77


def test_hints_about_the_codes():
    """Either of them for the step, its halves and the layer step, not both; neither for the operators."""
    lib = _lib.load()
    cached, streamed = _lib.F_CODES_CACHED, _lib.F_CODES_STREAMED
    for hint, want in ((cached, -2), (streamed, -2), (cached | streamed, -1)):    # (head_dim 64, 4 heads: refused later)
        tail = (hint, None)
        assert lib.adamas_decode_step_f(*[16] * 7, 8, 16, None, 256, 1 << 40, 1, 32, 32, 64, 16, 1.0, 100, 8, *tail) == want
        assert lib.adamas_step_candidates_f(*[16] * 5, 8, 256, 1 << 40, 1, 4, 4, 16, 100, 8, *tail) == want
        assert lib.adamas_step_attend_f(*[16] * 6, 8, 16, None, 256, 1 << 40, 1, 32, 32, 64, 16, 1.0, 100, 8, *tail) == want
        assert lib.adamas_decode_layer_step(*[16] * 8, 8, 16, None, 256, 1 << 40, 1, 4, 4, 128, 16, 1.0, 100, 8, 1.0,
                                            *tail) == want
        assert lib.adamas_sparse_decode_f(*[16] * 5, None, 0, 0, 16, None, 0, 1, 32, 32, 64, 16, 1.0, 100, *tail) == -1
    c = _ctrl(num_layers=3)
    c._len_bound = 1 << 20
    assert c.codes_flags == streamed
    c._len_bound = 1
    assert c.codes_flags == cached


@pytest.mark.parametrize("length", [2, 4096, 140000])
def test_general_path_of_the_step_takes_the_codes_hint(length):
    """The step hands a budget of one token to the attention operator, which does not know the hint; without
    a device all that is left is the HIP runtime's error at the launch."""
    if torch.cuda.is_available():
        pytest.skip("would launch on addresses that are none")
    lib = _lib.load()
    need = lib.adamas_workspace_bytes(1, 32, length, 1)
    for flags in (0, _lib.F_CODES_CACHED):
        rc = lib.adamas_decode_step_f(*[256] * 7, 1, 256, None, 256, need, 1, 32, 32, 128, 16, 1.0, length,
                                      -(-length // 16), flags, None)
        assert rc > 0, (flags, rc)


def test_layer_addresses():
    """The addresses handed to the library are those of the layers' views, for the same indices."""
    c = _ctrl(num_layers=3)
    for layer in range(-3, 3):
        assert c.pool.kv_address(layer) == c.pool.kv[layer].data_ptr()
        assert c.pool.codes_address(layer) == c.pool.codes[layer].data_ptr()
    for layer in (1, -1):
        for kind in (np.int64, np.int32, np.uint8, torch.tensor, lambda i: torch.tensor(i, dtype=torch.int32)):
            if layer < 0 and kind is np.uint8:
                continue
            for address, views in ((c.pool.kv_address, c.pool.kv), (c.pool.codes_address, c.pool.codes)):
                got = address(kind(layer))
                ctypes.c_void_p.from_param(got)      # (as a call into the library does)
                assert got == views[layer].data_ptr()
    assert c.pool.kv_address(slice(1, 2)) == c.pool.kv[1].data_ptr()
    for layer in (-4, 3):
        with pytest.raises(IndexError):
            c.pool.kv_address(layer)
        with pytest.raises(IndexError):
            c.pool.codes_address(layer)


def test_write_words_arguments():
    lib = _lib.load()
    words = (_lib.c_int32 * 4)()
    assert lib.adamas_write_words(None, words, 4, None) == -1
    assert lib.adamas_write_words(16, None, 4, None) == -1
    assert lib.adamas_write_words(16, words, 0, None) == -1
    assert lib.adamas_write_words(16, words, _lib.MAX_WORDS + 1, None) == -1
    assert lib.adamas_write_words(18, words, 4, None) == -4


def test_a_call_that_the_native_host_side_leaves_costs_little():
    """Every operator asks the native function first, so one that declines (here: tensors on the CPU, neither h nor q,
    a controller that is none) must cost next to nothing: at most a few calls of an empty library function (0.9 of it
    measured; 15 where each decline was an exception)."""
    import time
    host, version = U._load_host(), _lib.load().adamas_version
    c = U.InferenceController(1, 8, 128, 16, 64, 64, torch.float16, "cpu")
    x = torch.zeros(1, 8, 128).half()
    declined = [lambda: host.hadamard(x, False, 1.0), lambda: host.hadamard(x, True, 1.0),
                lambda: host.append_decode(x, x, None, None, c, 0), lambda: host.append_decode(x, x, None, x, c, 0),
                lambda: host.estimate(x, c, 0), lambda: host.topk(x, c, None), lambda: host.sparse_attn(x, c, 0, None),
                lambda: host.step(x, x, c, 0), lambda: host.step(x, x, None, 0)]

    def best(call, n=2000):
        times = []
        for _ in range(20):
            t0 = time.perf_counter()
            for _ in range(n):
                call()
            times.append(time.perf_counter() - t0)
        return min(times)

    unit = best(version)
    for i, call in enumerate(declined):
        assert call() is None
        assert best(call) < 6 * unit, i


def test_tables_can_be_assigned():
    """As the plain attributes that they were: operators and later growth use the tensors given."""
    c = U.InferenceController(1, 32, 128, 16, 64, 64, torch.float16, "cpu")
    lengths, table = torch.zeros(1, dtype=torch.int32), torch.zeros(4, dtype=torch.int32)
    c.seqs.seq_lens_dev, c.seqs.table_dev = lengths, table
    c.prepare_hadamard(20)
    assert lengths.tolist() == [20] and table[:2].tolist() == c.seqs.pages[0]
    assert c.seq_lens is lengths and c.kv_indices_with_last is table
    assert c.seqs.launch_table_address(0) == table.data_ptr()
    assert c.seqs.launch_addresses(0) == (table.data_ptr(), c.seqs.indptr_dev.data_ptr(), lengths.data_ptr())


@pytest.mark.parametrize("missing", [True, False])
def test_operators_work_without_their_native_host_side(missing):
    """Without adamas_host.so, or with another torch than it was built for, a warning and the general way."""
    import subprocess
    import sys
    program = f"""
import warnings, torch
if {missing}:
    from adamas_amd import _lib
    _lib.HOST_PATH = _lib.HOST_PATH.with_name("absent.so")
else:
    torch.__version__ = "0.1"
import adamas_amd.utils as U
x = torch.zeros(1, 8, 128).half()
c = U.InferenceController(1, 8, 128, 16, 64, 64, torch.float16, "cpu")
calls = [lambda: U.hadamard_transform(x), lambda: U.append_kvh(x, x, None, c, 0, q=x),
         lambda: U.decode_estimate(x, c, 0), lambda: U.decode_topk(x, c), lambda: U.decode_sparse_attn(x, c, 0, None),
         lambda: U.decode_step(x, x, c, 0)]
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    for call in calls:
        try:
            call()
        except RuntimeError as e:
            print("CUDA" in str(e))
print(len(seen), {"'it is not built'" if missing else "'built for torch'"} in str(seen[0].message))
"""
    run = subprocess.run([sys.executable, "-c", program], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert run.stdout.split() == ["True"] * 6 + ["1", "True"], run.stdout + run.stderr
