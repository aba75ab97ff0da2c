"""The decode step against the stand-alone operators on the same caches (estimate, top-k, attention),
selections equal, outputs within the rounding of the format: at budgets above 256 where its chunks of
distances change size (512, 1024 and 2048 tokens), and with grouped queries where one lane of the
estimator serves four query heads (whole and partial passes, wide and narrow workgroups)."""
import pytest
import torch

import adamas_amd.utils as U

pytestmark = pytest.mark.gpu


def _controller(dev, lens, budget, page, kv_heads, dtype, layout, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    ctrl = U.InferenceController(1, 32, 128, page, budget, max(lens), dtype, dev, batch_size=len(lens),
                                 num_kv_heads=kv_heads, layout=layout, hadamard_scale=U.RAW_SCALE)
    ctrl.pool.kv.copy_(torch.randn(ctrl.pool.kv.shape, generator=g, device=dev))
    ctrl.pool.codes.copy_(torch.randint(-32768, 32768, ctrl.pool.codes.shape, generator=g, device=dev))
    ctrl.prepare_hadamard(lens)
    ctrl.begin_forward(1)
    q, k, v = (torch.randn(len(lens), h, 128, generator=g, device=dev).to(dtype) for h in (32, kv_heads, kv_heads))
    return ctrl, q, U.append_kvh(k, v, None, ctrl, 0, q=q)


@pytest.mark.parametrize("lens,budget,page,kv_heads,dtype,layout", [
    ([32769], 300, 16, 32, torch.float16, 0),       # the last length with chunks of 512
    ([32770], 300, 16, 8, torch.bfloat16, 1),       # the first with 1024
    ([65537], 1000, 1, 8, torch.float16, 0),
    ([65538], 4000, 16, 32, torch.float16, 0),      # the first with 2048
    ([131073], 2000, 32, 8, torch.bfloat16, 0),     # the longest
    ([300, 40000, 2049, 1025, 70001], 257, 16, 8, torch.float16, 0),
    ([1100, 513, 514, 300, 1026, 2], 512, 16, 4, torch.float16, 1),
])
def test_step_large_budget_chunk_sizes(gpu_device, lens, budget, page, kv_heads, dtype, layout):
    _check(gpu_device, lens, budget, page, kv_heads, dtype, layout)


@pytest.mark.parametrize("lens,budget,page,kv_heads,dtype,layout", [
    ([32768], 128, 16, 8, torch.float16, 0),        # one whole pass
    ([33000], 128, 16, 8, torch.bfloat16, 1),       # a second pass of a few units
    ([48017], 256, 1, 8, torch.float16, 0),
    ([100001], 200, 16, 4, torch.float16, 0),
    ([9000, 17, 600, 513, 2], 100, 16, 8, torch.float16, 0),
    ([40000, 3000], 256, 32, 4, torch.bfloat16, 0),
])
def test_step_grouped_queries_share_a_lane(gpu_device, lens, budget, page, kv_heads, dtype, layout):
    _check(gpu_device, lens, budget, page, kv_heads, dtype, layout)


@pytest.mark.parametrize("length,budget", [(40000, 128), (33000, 256), (5000, 64)])
def test_layer_step_grouped_queries(gpu_device, length, budget):
    """From the fused projection: codes made in the estimator, four heads to a lane."""
    ctrl, q, _ = _controller(gpu_device, [length], budget, 16, 8, torch.float16, 0, length)
    g = torch.Generator(device=gpu_device).manual_seed(length)
    qkv = torch.randn(1, 48, 128, generator=g, device=gpu_device).half()
    ang = torch.rand(length, 64, generator=g, device=gpu_device) * 6
    cos, sin = ang.cos(), ang.sin()
    q2, code = U.rope_append_decode(qkv, cos, sin, ctrl, 0)
    want, sel = U.decode_step(q2, code, ctrl, 0, return_indices=True)
    sel = sel.clone()
    o, sel2 = U.decode_layer_step(qkv, cos, sin, ctrl, 0, return_indices=True)
    assert torch.equal(sel, sel2)
    assert bool(((o.float() - want.float()).abs() <= 2.0 ** -10 * want.float().abs() + 1e-5).all())


def _check(gpu_device, lens, budget, page, kv_heads, dtype, layout):
    ctrl, q, q_code = _controller(gpu_device, lens, budget, page, kv_heads, dtype, layout, lens[0] + budget)
    o, sel = U.decode_step(q, q_code, ctrl, 0, return_indices=True)
    sel = sel.clone()
    assert torch.equal(o, U.decode_step(q, q_code, ctrl, 0))
    U.decode_topk(U.decode_estimate(q_code, ctrl, 0), ctrl)
    want = ctrl.topk_dindices_buffer
    assert torch.equal(sel.sort(dim=1).values, want.sort(dim=1).values)
    o2 = U.decode_sparse_attn(q, ctrl, 0, want)
    # the same rows in another order of summation: fp32 sums, one rounding to 16 bits each
    ulp = 2.0 ** (-10 if dtype == torch.float16 else -7)
    assert bool(((o.float() - o2.float()).abs() <= ulp * o2.float().abs() + 1e-5).all())


@pytest.mark.parametrize("heads,length,page", [(8, 33000, 16), (8, 70001, 1), (16, 40000, 16), (32, 32768, 32)])
def test_step_reads_codes_through_and_past_the_caches(gpu_device, heads, length, page, monkeypatch):
    """The hint about cached codes changes no bit: both instances of the wide estimator (fewer workgroups than
    CUs) and the one that ignores the hint, from the projection and from query codes; selection against the
    stand-alone operators."""
    from adamas_amd.utils import controller as C
    dev = gpu_device
    g = torch.Generator(device=dev).manual_seed(length)
    ctrl = U.InferenceController(1, heads, 128, page, 128, length, torch.float16, dev)
    ctrl.pool.kv.copy_(torch.randn(ctrl.pool.kv.shape, generator=g, device=dev))
    ctrl.pool.codes.copy_(torch.randint(-32768, 32768, ctrl.pool.codes.shape, generator=g, device=dev))
    ctrl.prepare_hadamard(length)
    ctrl.begin_forward(1)
    qkv = torch.randn(1, 3 * heads, 128, generator=g, device=dev).half()
    angle = torch.rand(length, 64, generator=g, device=dev)
    q, k, v = (x.contiguous() for x in qkv.chunk(3, dim=1))
    q_code = U.append_kvh(k, v, None, ctrl, 0, q=q)
    got = []
    for limit in (0, 1 << 40):
        monkeypatch.setattr(C, "CODES_CACHED_BYTES", limit)
        o, sel = U.decode_step(q, q_code, ctrl, 0, return_indices=True)
        got.append((o, sel.clone()))
        o, sel = U.decode_layer_step(qkv, angle.cos(), angle.sin(), ctrl, 0, return_indices=True)
        got.append((o, sel.clone()))
        U.append_kvh(k, v, None, ctrl, 0, q=q)     # (the layer step rotated the new token's row)
    assert torch.equal(got[0][0], got[2][0]) and torch.equal(got[0][1], got[2][1])
    assert torch.equal(got[1][0], got[3][0]) and torch.equal(got[1][1], got[3][1])
    U.decode_topk(U.decode_estimate(q_code, ctrl, 0), ctrl)
    want = ctrl.topk_dindices_buffer.sort(dim=1).values
    assert torch.equal(got[0][1].sort(dim=1).values, want)


@pytest.mark.parametrize("lens,budget,page", [
    ([700, 5000, 1, 513, 2049], 100, 16),     # selection, narrow workgroups of a batch
    ([9000], 64, 1),                          # selection, narrow workgroups of one sequence
    ([700, 5000, 1, 513, 2049], 600, 16),     # histograms
    ([16385], 300, 32),
])
def test_step_of_narrow_workgroups_reads_codes_through_and_past_the_caches(gpu_device, lens, budget, page, monkeypatch):
    """Both instances give the same bits, and the selection of the stand-alone operators."""
    from adamas_amd.utils import controller as C
    dev = gpu_device
    g = torch.Generator(device=dev).manual_seed(sum(lens))
    n = len(lens)
    ctrl = U.InferenceController(1, 32, 128, page, budget, max(lens) + 1, torch.float16, dev, batch_size=n)
    ctrl.pool.kv.copy_(torch.randn(ctrl.pool.kv.shape, generator=g, device=dev))
    ctrl.pool.codes.copy_(torch.randint(-32768, 32768, ctrl.pool.codes.shape, generator=g, device=dev))
    ctrl.prepare_hadamard(lens)
    ctrl.prepare_hadamard(1)
    ctrl.begin_forward(1)
    q, k, v = (torch.randn(n, 32, 128, generator=g, device=dev).half() for _ in range(3))
    q_code = U.append_kvh(k, v, None, ctrl, 0, q=q)
    got = []
    for limit in (0, 1 << 40):
        monkeypatch.setattr(C, "CODES_CACHED_BYTES", limit)
        o, sel = U.decode_step(q, q_code, ctrl, 0, return_indices=True)
        got.append((o, sel.clone()))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    U.decode_topk(U.decode_estimate(q_code, ctrl, 0), ctrl)
    assert torch.equal(got[0][1].sort(dim=1).values, ctrl.topk_dindices_buffer.sort(dim=1).values)


@pytest.mark.parametrize("lens,budget,cached,unknown", [
    ([4096], 64, False, False), ([700, 5000, 513], 100, False, False),    # selection, narrow workgroups
    ([32768], 128, True, True),                                           # wide ones on the whole chip
    ([4096], 600, False, False), ([700, 5000, 513], 600, False, False),   # histograms
    ([19000] + [600] * 15, 100, False, True),                             # 16 * 19000 tokens: 311 MB of codes at most
])
def test_step_reads_codes_past_the_caches_when_told_so(gpu_device, lens, budget, cached, unknown):
    """The last template argument of the estimator that is launched, for each hint and for none."""
    from torch.profiler import ProfilerActivity, profile
    from adamas_amd import _lib
    c, q, q_code = _controller(gpu_device, lens, budget, 16, 32, torch.float16, 0, 7)
    o, ws = torch.empty_like(q), c.workspace(budget)

    def launched(flags):
        with profile(activities=[ProfilerActivity.CUDA]) as p:
            rc = _lib.load().adamas_decode_step_f(
                q.data_ptr(), q_code.data_ptr(), c.pool.kv.data_ptr(), c.pool.codes.data_ptr(),
                c.seqs.table_dev.data_ptr(), c.seqs.indptr_dev.data_ptr(), c.seqs.seq_lens_dev.data_ptr(), budget,
                o.data_ptr(), None, ws.data_ptr(), ws.numel(), len(lens), 32, 32, 128, 16, 128 ** -0.5, max(lens),
                c.seqs.max_pages, flags, _lib.current_stream())
            assert rc == 0
            torch.cuda.synchronize()
        name = next(e.name for e in p.events() if "estimate_select_kernel" in e.name)
        return {"true": True, "false": False}[name.split("<")[1].split(">")[0].split(", ")[-1]]

    assert launched(_lib.F_CODES_STREAMED)
    assert launched(_lib.F_CODES_CACHED) == cached
    assert launched(0) == unknown


@pytest.mark.parametrize("lens,budget,kv_heads", [
    ([4096], 1, 32), ([3000, 700], 1, 8),     # nothing is selected
    ([140000], 300, 32), ([140000], 1000, 8), # longer than the histograms go
])
def test_step_on_the_general_path_takes_the_codes_hint(gpu_device, lens, budget, kv_heads, monkeypatch):
    from adamas_amd.utils import controller as C
    ctrl, q, q_code = _controller(gpu_device, lens, budget, 16, kv_heads, torch.float16, 0, 5)
    got = []
    for limit in (0, 1 << 40):
        monkeypatch.setattr(C, "CODES_CACHED_BYTES", limit)
        assert bool(ctrl.codes_hint) == bool(limit)
        got.append(U.decode_step(q, q_code, ctrl, 0))
    assert torch.equal(*got) and bool(got[0].any())


@pytest.mark.parametrize("longest,kv_heads,layout", [(3072, 32, 0), (3074, 8, 1), (4097, 32, 0)])
def test_step_of_more_slabs_than_run_at_once(gpu_device, longest, kv_heads, layout):
    """512 (sequence, head) pairs: slabs of 1024 tokens up to 3073, of 2048 beyond."""
    lens = [longest] + [2 + (613 * i) % (longest - 2) for i in range(15)]
    _check(gpu_device, lens, 600, 16, kv_heads, torch.float16, layout)


@pytest.mark.parametrize("lens,budget,page,kv_heads,dtype,layout", [
    ([10241], 1024, 16, 32, torch.float16, 0),          # ten slabs of 1024: the last with 256 threads on each
    ([10242], 1024, 16, 8, torch.bfloat16, 1),          # the first of 2048 with 512
    ([10242], 9000, 1, 32, torch.float16, 0),           # nearly every token
    ([24577], 512, 16, 8, torch.float16, 0),            # slabs of 4096, the last with one token
    ([65537], 2000, 16, 8, torch.float16, 0),           # 512 workgroups: the last with 512 threads
    ([65538], 2000, 16, 8, torch.float16, 1),           # the first with 256 again
    ([16000, 900, 2, 4098], 300, 16, 4, torch.bfloat16, 0),
])
def test_step_of_workgroups_of_512(gpu_device, lens, budget, page, kv_heads, dtype, layout):
    _check(gpu_device, lens, budget, page, kv_heads, dtype, layout)


@pytest.mark.parametrize("lens,budget,kv_heads", [
    ([131073], 2000, 8),             # a wave's rows hold 32768 tokens, all in one bin
    ([65537], 2000, 32),             # the same for the eight waves of the wide workgroup
    ([4097, 900, 33000], 300, 16),
])
def test_step_of_equal_distances_takes_the_first_tokens(gpu_device, lens, budget, kv_heads):
    ctrl, q, q_code = _controller(gpu_device, lens, budget, 16, kv_heads, torch.float16, 0, 3)
    ctrl.pool.codes.fill_(0x1b1b)
    _, sel = U.decode_step(q, q_code, ctrl, 0, return_indices=True)
    pos = torch.arange(budget - 1, device=gpu_device, dtype=torch.int32)
    for b, n in enumerate(lens):
        rows = sel[32 * b:32 * (b + 1)].sort(dim=1).values
        assert torch.equal(rows, pos.expand(32, -1)), b
    o, _ = U.decode_step(q, q_code, ctrl, 0, return_indices=True)
    assert torch.equal(o, U.decode_step(q, q_code, ctrl, 0))
    o2 = U.decode_sparse_attn(q, ctrl, 0, sel.contiguous())
    assert bool(((o.float() - o2.float()).abs() <= 2.0 ** -10 * o2.float().abs() + 1e-5).all())


@pytest.mark.parametrize("kv_heads", [1, 2, 16])
def test_step_in_the_order_of_key_value_heads(gpu_device, kv_heads):
    """The workgroups of the heads that share a key/value head lie together."""
    _check(gpu_device, [5000, 700], 400, 16, kv_heads, torch.float16, 0)


@pytest.mark.parametrize("lens,budget,page,kv_heads,layout", [
    ([70001, 1030, 2], 128, 16, 32, 0),     # narrow workgroups, four passes, the last one ragged
    ([33000, 600], 64, 1, 32, 1),           # two passes
    ([66000, 65537], 200, 16, 8, 0),        # four heads to a lane
])
def test_step_of_several_passes_counts_as_it_goes(gpu_device, lens, budget, page, kv_heads, layout):
    _check(gpu_device, lens, budget, page, kv_heads, torch.float16, layout)
