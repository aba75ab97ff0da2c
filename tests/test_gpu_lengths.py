"""Lengths and page ids reach the device without the host waiting for them, and every reader finds them: on the
stream that wrote them, on others, in graphs that are replayed."""
import copy

import pytest
import torch

import adamas_amd.utils as U
from adamas_amd import _lib
from adamas_amd.decoder import DecoderConfig, LlamaShapedDecoder
from adamas_amd.utils.paging import PagedSequences, PagePool

pytestmark = pytest.mark.gpu


def _seqs(dev, batch, capacity, page=1):
    pool = PagePool(1, 8, 128, page, batch * -(-capacity // page), torch.float16, dev,
                    page_order=list(range(batch * -(-capacity // page)))[::-1])
    return PagedSequences(pool, batch, capacity, dev)


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, _lib.MAX_WORDS, _lib.MAX_WORDS + 1])
def test_pages_and_lengths_arrive(gpu_device, n):
    s = _seqs(gpu_device, 2, n + 3)
    s.reserve([n, 1])
    s.reserve([2, 0])
    assert not s._host_waits
    assert s.seq_lens_dev.tolist() == [n + 2, 1]
    table = s.table_dev.view(2, -1).tolist()
    assert table[0][:n + 2] == s.pages[0] and table[1][:1] == s.pages[1]
    assert not any(table[0][n + 2:]) and not any(table[1][1:])


def test_many_writes_behind_a_busy_stream_keep_their_order(gpu_device):
    s = _seqs(gpu_device, 1, 64)
    x = torch.randn(4096, 4096, device=gpu_device)
    seen = []
    for _ in range(20):
        x = x @ x * 1e-3      # the host is far ahead of the device
        s.reserve([1])
        seen.append(s._seq_lens_dev.clone())     # as an operator's launch reads them
    assert not s._host_waits
    assert torch.cat(seen).tolist() == list(range(1, 21))


def test_another_stream_waits(gpu_device):
    s = _seqs(gpu_device, 1, 64)
    x = torch.randn(8192, 8192, device=gpu_device)
    torch.cuda.synchronize()
    for _ in range(5):
        x = x @ x * 1e-4
    s.reserve([7])                                   # behind the products
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):                    # (no event between the streams)
        got = s.seq_lens_dev.clone()
        side.synchronize()
    assert got.tolist() == [7] and s._host_waits
    s.reserve([3])                                   # the host waits from now on
    with torch.cuda.stream(side):
        got = s.seq_lens_dev.clone()
    side.synchronize()
    assert got.tolist() == [10]


def test_a_captured_use_ends_writes_without_waiting(gpu_device):
    s = _seqs(gpu_device, 1, 64)
    s.reserve([2])
    out = torch.zeros(1, dtype=torch.int32, device=gpu_device)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out.copy_(s.seq_lens_dev)
    assert s._host_waits
    side = torch.cuda.Stream()
    for n in range(3, 8):
        s.reserve([1])
        with torch.cuda.stream(side):
            graph.replay()
        side.synchronize()
        assert out.item() == n


def test_eager_decoding_of_a_controller_on_one_stream(gpu_device):
    """Token by token with and without the wait: the same selections and outputs."""
    got = []
    for waits in (False, True):
        g = torch.Generator(device=gpu_device).manual_seed(1)
        c = U.InferenceController(1, 32, 128, 16, 64, 400, torch.float16, gpu_device)
        c.seqs._host_waits = waits
        k, v = (torch.randn(330, 32, 128, generator=g, device=gpu_device).half() for _ in range(2))
        c.prepare_hadamard(330)
        U.append_kvh(k, v, None, c, 0)
        out = []
        for _ in range(40):
            c.prepare_hadamard(1)
            c.begin_forward(1)
            q, k, v = (torch.randn(1, 32, 128, generator=g, device=gpu_device).half() for _ in range(3))
            out.append(U.decode_step(q, U.append_kvh(k, v, None, c, 0, q=q), c, 0))
        assert c.seqs._host_waits == waits
        got.append(torch.cat(out))
    assert torch.equal(*got)


def test_operators_see_to_other_streams_and_graphs(gpu_device):
    """The native host side leaves such calls to the getters of the tables."""
    c = U.InferenceController(1, 32, 128, 16, 64, 400, torch.float16, gpu_device)
    g = torch.Generator(device=gpu_device).manual_seed(2)
    k, v = (torch.randn(330, 32, 128, generator=g, device=gpu_device).half() for _ in range(2))
    q, kn, vn = (torch.randn(1, 32, 128, generator=g, device=gpu_device).half() for _ in range(3))
    want = []
    for use in ("same", "side", "graph"):
        c.clean_states()
        c.seqs._host_waits, c.seqs._writer = False, None
        c.prepare_hadamard(329)
        U.append_kvh(k[:329].contiguous(), v[:329].contiguous(), None, c, 0)
        c.prepare_hadamard(1)
        c.begin_forward(1)
        c.workspace(64)
        torch.cuda.synchronize()
        if use == "same":
            out = U.decode_step(q, U.append_kvh(kn, vn, None, c, 0, q=q), c, 0)
            assert not c.seqs._host_waits
        elif use == "side":
            side = torch.cuda.Stream()
            with torch.cuda.stream(side):
                out = U.decode_step(q, U.append_kvh(kn, vn, None, c, 0, q=q), c, 0)
            side.synchronize()
            assert c.seqs._host_waits
        else:
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                out = U.decode_step(q, U.append_kvh(kn, vn, None, c, 0, q=q), c, 0)
            assert c.seqs._host_waits
            graph.replay()
        want.append(out.clone())
    assert torch.equal(want[0], want[1]) and torch.equal(want[0], want[2])


@pytest.mark.parametrize("held", ["lengths", "table", "address"])
def test_what_has_been_handed_out_is_written_when_the_call_returns(gpu_device, held):
    """A tensor or an address taken once is right on any stream after every reserve."""
    c = U.InferenceController(1, 32, 128, 16, 64, 400, torch.float16, gpu_device, page_order=list(range(25))[::-1])
    c.prepare_hadamard(5)
    assert not c.seqs._host_waits
    if held == "lengths":
        view = c.seq_lens
    elif held == "table":
        view = c.kv_indices_with_last
    else:
        assert c.seqs.table_ptr(0) == c.seqs._table_dev.data_ptr()
        view = c.seqs._table_dev
    assert c.seqs._host_waits
    x = torch.randn(8192, 8192, device=gpu_device)
    torch.cuda.synchronize()
    for _ in range(5):
        x = x @ x * 1e-4
    c.prepare_hadamard(30)                           # behind the products
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):                    # (no event between the streams)
        got = view.clone()
        side.synchronize()
    assert got[:3].tolist() == ([35] if held == "lengths" else [24, 23, 22])


def test_a_request_waits_for_no_write(gpu_device):
    """Prompt and eager steps of a decoder take nothing that would make the host wait."""
    cfg = DecoderConfig(num_layers=2, hidden=256, num_heads=8, intermediate=512, vocab=64, dense_layers=1)
    model = LlamaShapedDecoder(cfg, gpu_device)
    model.init_cache(16, 128, 32)
    ids = torch.arange(60, device=gpu_device)
    for _ in range(2):
        model.clear()
        model.prefill(ids[:50])
        for i in range(50, 60):
            model.decode_step_eager(ids[i:i + 1])
    assert not model.ctrl.seqs._host_waits
    assert model.ctrl.seq_lens.tolist() == [60]


@pytest.mark.parametrize("default", [True, False])
def test_a_capture_waits_for_what_is_still_to_be_written(gpu_device, default):
    """Written on the default stream and captured on another one, without the synchronization that torch.cuda.graph
    begins with; or all on one other stream, where the host waits for every write.  Replayed on a third stream."""
    writer = torch.cuda.default_stream() if default else torch.cuda.Stream()
    other, third = torch.cuda.Stream(), torch.cuda.Stream()
    x = torch.randn(8192, 8192, device=gpu_device)
    lens, pages = (torch.zeros(1, dtype=torch.int32, device=gpu_device) for _ in range(2))
    torch.cuda.synchronize()
    with torch.cuda.stream(writer):
        s = _seqs(gpu_device, 1, 64)
        x = x @ x * 1e-4
        torch.cuda.synchronize()
        for _ in range(5):
            x = x @ x * 1e-4
        s.reserve([7])                               # behind the products
        assert s._host_waits != default
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(other if default else writer):
        graph.capture_begin()
        s.launch_addresses(_lib.current_stream())    # as an operator asks for them
        lens.copy_(s._seq_lens_dev)
        pages.copy_(s._table_dev[:1])
        graph.capture_end()
    assert s._host_waits and s._writer is None
    for _ in range(2):
        with torch.cuda.stream(third):
            graph.replay()
        third.synchronize()
        assert lens.tolist() == [7] and pages.tolist() == [63]
        with torch.cuda.stream(third):
            lens.zero_()
            pages.zero_()


def test_a_copy_waits_for_its_own_writes(gpu_device):
    s = _seqs(gpu_device, 1, 64)
    s.reserve([7])
    t = copy.deepcopy(s)
    assert t._host_waits and not s._host_waits
    t.reserve([1])
    assert t.seq_lens_dev.tolist() == [8] and s.seq_lens_dev.tolist() == [7]


@pytest.mark.parametrize("pages", [1, _lib.MAX_WORDS, _lib.MAX_WORDS + 1])
def test_a_write_from_another_stream_comes_behind_those_before(gpu_device, pages):
    """Whatever its size, and so by whatever way it goes."""
    s = _seqs(gpu_device, 1, pages + 8)
    x = torch.randn(8192, 8192, device=gpu_device)
    x = x @ x * 1e-4
    torch.cuda.synchronize()
    for _ in range(5):
        x = x @ x * 1e-4
    s.reserve([7])                                   # behind the products
    event = torch.cuda.Event()
    event.record()
    with torch.cuda.stream(torch.cuda.Stream()):
        assert not event.query()
        s.reserve_pages_ahead(pages)
        assert event.query() and s._host_waits and s._writer is None
    assert s.table_dev.tolist() == s.pages[0] + [0] * (s.max_pages - 7 - pages) and s.seq_lens_dev.tolist() == [7]
