"""Dense decode attention of ragged batches, whose tokens the kernels share out as one list: lengths at
the edges of its units, parts that cross into the next sequence, more than 64 sequences (the second
round of the prefix sum), a sequence without tokens, both merges of the parts; against float64."""
import math

import pytest
import torch

import adamas_amd.utils as U
from adamas_amd import _lib

pytestmark = pytest.mark.gpu

LONG = [9001, 128, 1, 33, 4097, 127, 129, 0]
MANY = [1 + (37 * i) % 230 for i in range(70)]
TWO = [30000, 31]                                # few sequences: the parts get a merge launch


@pytest.mark.parametrize("lens,kv_heads,page,dtype,layout", [
    (LONG, 32, 16, torch.float16, 0),
    (LONG, 8, 16, torch.bfloat16, 0),
    (LONG, 16, 1, torch.float16, 1),
    (LONG, 4, 32, torch.float16, 0),
    (MANY, 32, 16, torch.bfloat16, 1),
    (MANY, 8, 16, torch.float16, 0),
    (TWO, 32, 16, torch.float16, 0),
    (TWO, 8, 16, torch.float16, 1),
])
def test_dense_attention_of_ragged_batches(gpu_device, lens, kv_heads, page, dtype, layout):
    dev = gpu_device
    g = torch.Generator(device=dev).manual_seed(len(lens) + kv_heads)
    ctrl = U.InferenceController(1, 32, 128, page, 1 << 20, max(lens), dtype, dev, batch_size=len(lens),
                                 num_kv_heads=kv_heads, layout=layout)
    ctrl.pool.kv.copy_(torch.randn(ctrl.pool.kv.shape, generator=g, device=dev))
    ctrl.prepare_hadamard(lens)
    ctrl.begin_forward(1) if min(lens) > 1 else setattr(ctrl, "inference_page_budget", max(lens))
    q = torch.randn(len(lens), 32, 128, generator=g, device=dev).to(dtype)
    o = U.decode_sparse_attn(q, ctrl, 0, U.ALL_PAST_TOKENS)
    assert torch.equal(o, U.decode_sparse_attn(q, ctrl, 0, U.ALL_PAST_TOKENS))
    u = 2.0 ** (-11 if dtype == torch.float16 else -8)   # half an ulp of 11 or 8 significant bits
    for b, n in enumerate(lens):
        if n == 0:
            assert not o[b].any()
            continue
        kv = ctrl.pool.kv[0][torch.tensor(ctrl.seqs.pages[b], device=dev)]
        kv = (kv if layout == 0 else kv.transpose(2, 3)).transpose(0, 1).reshape(2, -1, kv_heads, 128)
        k, v = (x[:n].repeat_interleave(32 // kv_heads, dim=1).transpose(0, 1).double() for x in kv)
        w = torch.softmax((k @ q[b].double()[:, :, None])[..., 0] / math.sqrt(128), dim=-1)
        ref, mag = (w[:, None] @ v)[:, 0], (w[:, None] @ v.abs())[:, 0]
        # the result rounded to 16 bits, the rest fp32 with scores below 2^7; weights on the matrix cores
        # are two 16-bit values, so their rounding (2^-16 in bf16) is in the second term, and what is
        # left of an fp16 weight may be denormal: 2^-25 absolute against a sum of weights of at least 1
        bound = u * ref.abs() + 2.0 ** -14 * mag + 2.0 ** -25 * v.abs().sum(1)
        assert bool(((o[b].double() - ref).abs() <= bound).all()), (b, n)


@pytest.mark.parametrize("lens,kv_heads,page,dtype,layout", [
    ([1408], 32, 16, torch.float16, 0),               # two rows in flight, the last split full
    ([1409], 8, 1, torch.bfloat16, 1),                # and with one row
    ([2048], 8, 1, torch.bfloat16, 1),                # the last length of them
    ([2049], 32, 16, torch.float16, 0),               # four
    ([1000, 1, 999, 641], 8, 16, torch.float16, 0),   # four sequences whose workgroups just run at once
    ([1025, 1, 999, 641], 8, 16, torch.float16, 0),   # and no longer
    ([512, 500, 129, 3, 257, 511, 64, 65], 4, 16, torch.bfloat16, 0),
    ([513, 500, 129, 3, 257, 511, 64, 65], 16, 32, torch.float16, 1),
    ([256] * 8, 32, 16, torch.float16, 0),
    ([250, 193] * 8, 32, 16, torch.bfloat16, 0),      # more than run at once: four rows in flight
])
def test_dense_attention_at_the_edges_of_the_row_kernel(gpu_device, lens, kv_heads, page, dtype, layout):
    test_dense_attention_of_ragged_batches(gpu_device, lens, kv_heads, page, dtype, layout)


@pytest.mark.parametrize("n,dtype,as_list", [
    (1409, torch.float16, False), (2048, torch.float16, False), (2000, torch.bfloat16, False),
    (1500, torch.bfloat16, True), (2048, torch.float16, True)])
def test_splits_of_one_sequence_are_of_128_rows(gpu_device, n, dtype, as_list):
    """Rows 0 and 1 cancel inside their split; row 128 is far too small to survive beside either of them
    and only counts because it is added up in another split."""
    dev = gpu_device
    big, small = (65504., 0.75 * 2.0 ** -9) if dtype == torch.float16 else (2.0 ** 60, 1.)
    ctrl = U.InferenceController(1, 32, 128, 16, 1 << 20, n, dtype, dev)
    ctrl.pool.kv.zero_()
    ctrl.prepare_hadamard(n)
    ctrl.begin_forward(1)
    for pos, value in ((0, big), (1, -big), (128, small)):
        ctrl.pool.kv[0][ctrl.seqs.pages[0][pos // 16], 1, pos % 16] = value
    sel = U.ALL_PAST_TOKENS
    if as_list:     # (the current token is the last row)
        sel = torch.arange(n - 1, device=dev, dtype=torch.int32).expand(32, -1).contiguous()
    o = U.decode_sparse_attn(torch.zeros(1, 32, 128, dtype=dtype, device=dev), ctrl, 0, sel)
    # every weight is 1 / n; one rounding to 16 bits (half an ulp of 8 bits, or of fp16's denormals)
    assert bool(((o.double() - small / n).abs() <= 2.0 ** -8 * small / n + 2.0 ** -25).all()), float(o.float().max())


@pytest.mark.parametrize("lens,kv_heads,dtype", [
    ([2000, 1777], 8, torch.float16), ([2000, 1777], 4, torch.float16), ([1900] * 4, 16, torch.float16),
    ([2000, 1777], 8, torch.bfloat16), ([9000], 8, torch.float16)])
def test_dense_attention_of_many_small_weights(gpu_device, lens, kv_heads, dtype):
    """One key outweighs each of the others by 2^20.35, but its value is zero: the output is the sum of the
    small weights, which are below the smallest normal number of fp16."""
    dev = gpu_device
    ctrl = U.InferenceController(1, 32, 128, 16, 1 << 20, max(lens), dtype, dev, batch_size=len(lens),
                                 num_kv_heads=kv_heads)
    ctrl.prepare_hadamard(lens)
    q = torch.zeros(len(lens), 32, 128, device=dev, dtype=dtype)
    q[:, :, 0] = 8.0
    for b, n in enumerate(lens):
        k = torch.zeros(n, kv_heads, 128, device=dev, dtype=dtype)
        k[n // 3, :, 0] = 20.35 / math.log2(math.e) * math.sqrt(128) / 8.0
        v = torch.ones_like(k)
        v[n // 3] = 0
        U.append_kvh(k, v, None, ctrl, 0, seq_idx=b)
    top = 8.0 * float(torch.tensor(20.35 / math.log2(math.e) * math.sqrt(128) / 8.0).to(dtype)) / math.sqrt(128)
    ctrl.begin_forward(1)
    o = U.decode_sparse_attn(q, ctrl, 0, U.ALL_PAST_TOKENS).double()
    for b, n in enumerate(lens):
        rest = (n - 1) * math.exp(-top)
        ref = rest / (1.0 + rest)
        # 2^-16 of a weight's rounding in bf16 (2^-22 in fp16), fp32 scores of about 2^4 (2^-19 in the
        # exponent), fp32 sums: below 2^-14; the result rounded once (fp16: normal above 2^-14)
        bound = (2.0 ** -14 + 2.0 ** (-11 if dtype == torch.float16 else -8)) * ref
        assert float((o[b] - ref).abs().max()) <= bound, (b, n)


SHORT = [1500, 1333, 40, 1201]


def _short_batch(dev, kv_heads, dtype):
    ctrl = U.InferenceController(1, 32, 128, 16, 1 << 20, max(SHORT), dtype, dev, batch_size=len(SHORT),
                                 num_kv_heads=kv_heads)
    ctrl.prepare_hadamard(SHORT)
    q = torch.zeros(len(SHORT), 32, 128, device=dev, dtype=dtype)
    k = torch.zeros(max(SHORT), kv_heads, 128, device=dev, dtype=dtype)
    g = torch.Generator(device=dev).manual_seed(kv_heads)
    v = [torch.randn(n, kv_heads, 128, generator=g, device=dev).to(dtype) for n in SHORT]
    return ctrl, q, k, v


@pytest.mark.parametrize("kv_heads", [32, 16, 8, 4])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_dense_attention_with_every_score_at_minus_infinity(gpu_device, kv_heads, dtype):
    """No token has a weight: zeros, whatever the slots past the end of a tile hold."""
    ctrl, q, k, v = _short_batch(gpu_device, kv_heads, dtype)
    q[:, :, 3] = 1.0
    k[:, :, 3] = -math.inf
    for b, n in enumerate(SHORT):
        U.append_kvh(k[:n].contiguous(), v[b], None, ctrl, 0, seq_idx=b)
    ctrl.begin_forward(1)
    assert not U.decode_sparse_attn(q, ctrl, 0, U.ALL_PAST_TOKENS).any()


@pytest.mark.parametrize("kv_heads", [32, 16, 8, 4])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_dense_attention_of_infinite_values(gpu_device, kv_heads, dtype):
    """Equal weights (exact in 16 bits: nothing is left over); an infinite channel of the value of one token,
    the last one among them, is infinite in the sum, with its sign, and no other channel sees it."""
    ctrl, q, k, v = _short_batch(gpu_device, kv_heads, dtype)
    for b, n in enumerate(SHORT):
        v[b][n // 2, :, 5] = math.inf
        v[b][n - 1, :, 70] = -math.inf
        U.append_kvh(k[:n].contiguous(), v[b], None, ctrl, 0, seq_idx=b)
    ctrl.begin_forward(1)
    o = U.decode_sparse_attn(q, ctrl, 0, U.ALL_PAST_TOKENS)
    want = torch.zeros_like(o)
    want[:, :, 5], want[:, :, 70] = math.inf, -math.inf
    assert not o.isnan().any() and torch.equal(torch.where(o.isinf(), o, 0), want)


@pytest.mark.parametrize("kv_heads,flags", [(32, 0), (8, 0), (8, _lib.F_NO_MFMA)])
def test_dense_attention_that_needs_no_workspace_takes_any(gpu_device, kv_heads, flags):
    """70 sequences of up to 500 tokens keep every CU busy without a split: a workspace that is missing, too
    small or misaligned is not used and refuses nothing.  One sequence is split and wants a whole one."""
    dev = gpu_device
    lens = [500 - 7 * i for i in range(70)]
    ctrl = U.InferenceController(1, 32, 128, 16, 1 << 20, max(lens), torch.float16, dev, batch_size=len(lens),
                                 num_kv_heads=kv_heads)
    g = torch.Generator(device=dev).manual_seed(1)
    ctrl.pool.kv.copy_(torch.randn(ctrl.pool.kv.shape, generator=g, device=dev))
    ctrl.prepare_hadamard(lens)
    ctrl.begin_forward(1)
    q = torch.randn(len(lens), 32, 128, generator=g, device=dev).half()
    want = U.decode_sparse_attn(q, ctrl, 0, U.ALL_PAST_TOKENS)
    ws = ctrl.workspace(1)
    need = _lib.load().adamas_workspace_bytes(len(lens), 32, 1, 1)

    def call(pointer, size, batch=len(lens), longest=max(lens)):
        o = torch.empty_like(q)
        rc = _lib.load().adamas_sparse_decode_f(
            q.data_ptr(), ctrl.pool.kv[0].data_ptr(), ctrl.seqs.table_dev.data_ptr(),
            ctrl.seqs.indptr_dev.data_ptr(), ctrl.seqs.seq_lens_dev.data_ptr(), None, 0, 0, o.data_ptr(), pointer,
            size, batch, 32, kv_heads, 128, 16, 1.0 / math.sqrt(128), longest, flags, _lib.current_stream())
        return rc, o

    assert ws.numel() >= need + 16
    for pointer, size in ((None, 0), (ws.data_ptr(), 16), (ws.data_ptr() + 16, need)):
        rc, o = call(pointer, size)
        assert rc == 0
        torch.testing.assert_close(o, want, rtol=2e-3, atol=2e-3)   # fp16 results of sums in another order
    # (the length bound may exceed the lengths: equal parts of the bound, most of them empty)
    assert call(None, 0, batch=1, longest=8000)[0] == -3
    assert call(ws.data_ptr(), 16, batch=1, longest=8000)[0] == -3
    assert call(ws.data_ptr() + 16, need, batch=1, longest=8000)[0] == -4


@pytest.mark.parametrize("heads,kv_heads,lens,dtype,layout", [
    (8, 8, [60000, 1], torch.float16, 0),          # one head group: its parts fill every slot for partials
    (8, 2, [60000, 1, 1], torch.bfloat16, 1),
    (16, 16, [60000, 1], torch.bfloat16, 0),       # two head groups
    (16, 4, [60000, 1, 1], torch.float16, 0),
    (8, 1, [40000, 300], torch.float16, 0),
    (32, 2, [9001, 128, 1, 4097], torch.float16, 0),   # rows that several workgroups read
    (24, 8, [9001, 128, 1, 4097], torch.bfloat16, 1),  # a group that is no power of two
    (40, 8, [5000], torch.float16, 0),
    (32, 1, [3000], torch.bfloat16, 0),
    (32, 16, [2600], torch.float16, 0),            # equal parts, two query heads per key/value head
    (32, 16, [7001], torch.bfloat16, 1),
    # batches of short sequences on both sides of the rule for the row kernel
    (32, 8, [48 - i for i in range(26)], torch.float16, 0),
    (32, 8, [48 - i for i in range(27)], torch.float16, 1),
    (32, 2, [100 - i for i in range(26)], torch.bfloat16, 0),
    (24, 8, [128 - i for i in range(14)], torch.float16, 0),
    (8, 4, [129 - i for i in range(128)], torch.float16, 0),
    (8, 2, [300, 1, 299, 7] * 9, torch.bfloat16, 1),
    (8, 8, [1300, 1200] * 16, torch.float16, 0),
    (32, 32, [129, 3, 128, 64] * 10, torch.float16, 0),
])
def test_dense_attention_of_other_head_counts(gpu_device, heads, kv_heads, lens, dtype, layout):
    dev = gpu_device
    g = torch.Generator(device=dev).manual_seed(heads + kv_heads)
    ctrl = U.InferenceController(1, heads, 128, 16, 1 << 20, max(lens), dtype, dev, batch_size=len(lens),
                                 num_kv_heads=kv_heads, layout=layout)
    ctrl.pool.kv.copy_(torch.randn(ctrl.pool.kv.shape, generator=g, device=dev))
    ctrl.prepare_hadamard(lens)
    ctrl.inference_page_budget = max(lens)
    q = torch.randn(len(lens), heads, 128, generator=g, device=dev).to(dtype)
    o = U.decode_sparse_attn(q, ctrl, 0, U.ALL_PAST_TOKENS)
    assert torch.equal(o, U.decode_sparse_attn(q, ctrl, 0, U.ALL_PAST_TOKENS))
    u = 2.0 ** (-11 if dtype == torch.float16 else -8)
    for b, n in enumerate(lens):
        kv = ctrl.pool.kv[0][torch.tensor(ctrl.seqs.pages[b], device=dev)]
        kv = (kv if layout == 0 else kv.transpose(2, 3)).transpose(0, 1).reshape(2, -1, kv_heads, 128)[:, :n]
        for h in range(heads):
            k, v = (x[:, h // (heads // kv_heads)].double() for x in kv)
            w = torch.softmax(k @ q[b, h].double() / math.sqrt(128), dim=-1)
            ref, mag = w @ v, w @ v.abs()
            # as above: the result rounded to 16 bits, weights of at least 16 significant bits, fp32 sums
            assert bool(((o[b, h].double() - ref).abs() <= u * ref.abs() + 2.0 ** -14 * mag).all()), (b, h)
