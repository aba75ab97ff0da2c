"""prefill_forward on the matrix cores at the edges of its tiles: rows of a workgroup (256 stacked query
rows, 32 per wave), tokens of a tile (64), token ranges that are merged, scores that keep growing (the
running maximum has to move), against float64."""
import math

import pytest
import torch

import adamas_amd.utils as U
from adamas_amd import _lib

pytestmark = pytest.mark.gpu


def _cache(dev, n, past, kv_heads, page, dtype, layout, growing, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    length = n + past
    pages = -(-length // page)
    order = torch.randperm(pages, generator=torch.Generator().manual_seed(seed)).tolist()
    ctrl = U.InferenceController(1, 32, 128, page, 64, length, dtype, dev, page_order=order,
                                 num_kv_heads=kv_heads, layout=layout)
    k = torch.randn(length, kv_heads, 128, generator=g, device=dev)
    q = torch.randn(n, 32, 128, generator=g, device=dev)
    if growing:   # every tile beats the maximum of the ones before it
        k = k * 0.1 + torch.arange(length, device=dev)[:, None, None] / length * 8.0
        q = q * 0.1 + 1.0
    k, q = k.to(dtype), q.to(dtype)
    v = torch.randn(length, kv_heads, 128, generator=g, device=dev).to(dtype)
    ctrl.prepare_hadamard(length)
    U.append_kvh(k, v, None, ctrl, 0) if length > 1 else U.append_kvh(k, v, k.clone(), ctrl, 0)
    return ctrl, q, k, v


def _reference(q, k, v, past, scale=1 / math.sqrt(128)):
    """(attention, sum of weights * |v|) in float64."""
    n, hq, _ = q.shape
    group = hq // k.shape[1]
    out = torch.empty(n, hq, 128, dtype=torch.float64, device=q.device)
    mag = torch.empty_like(out)
    hidden = torch.arange(k.shape[0], device=q.device)[None] > (past + torch.arange(n, device=q.device))[:, None]
    for h in range(hq):
        s = q[:, h].double() @ k[:, h // group].double().T * scale
        w = s.masked_fill(hidden, -math.inf).softmax(-1)
        vh = v[:, h // group].double()
        out[:, h], mag[:, h] = w @ vh, w @ vh.abs()
    return out, mag


@pytest.mark.parametrize("n,past,kv_heads,page,dtype,layout,growing", [
    (1, 0, 32, 16, torch.float16, 0, False),
    (1, 63, 32, 16, torch.bfloat16, 0, False),
    (31, 64, 32, 1, torch.float16, 1, False),
    (64, 65, 8, 16, torch.float16, 0, True),       # exactly one workgroup of stacked rows
    (65, 0, 8, 32, torch.bfloat16, 1, False),      # one query token more
    (255, 1, 32, 16, torch.float16, 0, True),
    (257, 127, 32, 12, torch.bfloat16, 0, False),  # a page size that is no power of two
    (96, 2000, 4, 16, torch.float16, 0, True),     # token ranges, merged
    (20, 5003, 8, 16, torch.bfloat16, 1, False),
    (300, 900, 32, 16, torch.float16, 0, False),
])
def test_prefill_attention_edges(gpu_device, n, past, kv_heads, page, dtype, layout, growing):
    ctrl, q, k, v = _cache(gpu_device, n, past, kv_heads, page, dtype, layout, growing, 11 * n + past)
    split = _lib.load().adamas_prefill_workspace_bytes(n, past, 32, kv_heads) > 0
    assert split == (past >= 900), "the token ranges are tested where they are meant to be"
    o = U.prefill_forward(q, ctrl, 0)
    ref, mag = _reference(q, k, v, past)
    # every weight is rounded to 16 bits (u = 2^-11 with the 11 significant
    # bits of fp16, 2^-8 with the 8 of bf16; 2^-25 absolute where fp16 turns
    # denormal, weights taken relative to a maximum of at least 1), the result once more; scores and
    # sums are fp32: scores of up to 2^7 leave 2^-16 in the exponent
    u = 2.0 ** (-11 if dtype == torch.float16 else -8)
    bound = u * (mag + ref.abs()) + 2.0 ** -14 * mag + 2.0 ** -25 * v.double().abs().sum(0).max()
    err = (o.double() - ref).abs()
    assert bool((err <= bound).all()), f"error {float((err - bound).max()):.3e} above the bound"


@pytest.mark.parametrize("n,past,kv_heads,page,dtype,layout", [
    (130, 70, 32, 8, torch.float16, 0),       # the smallest page with one address for a wave's eight rows
    (130, 70, 8, 4, torch.bfloat16, 1),       # the largest power of two below it
    (100, 301, 8, 24, torch.float16, 0),      # a multiple of eight that is no power of two
    (65, 190, 32, 128, torch.bfloat16, 1),    # a page of two tiles, the second tile not begun
    (128, 300, 32, 16, torch.float16, 0),     # 128 stacked rows: the last call of eight waves
    (129, 300, 32, 16, torch.bfloat16, 1),    # four waves, one row in the second workgroup
    (50, 2510, 8, 16, torch.float16, 0),      # 2560 tokens: the longest call of four waves
    (50, 2511, 8, 16, torch.bfloat16, 0),     # eight
    (4230, 0, 8, 16, torch.float16, 0),       # 67 tiles: the page ids a wave keeps are looked up again
    (4230, 0, 8, 1, torch.bfloat16, 0),
])
def test_prefill_attention_page_sizes(gpu_device, n, past, kv_heads, page, dtype, layout):
    ctrl, q, k, v = _cache(gpu_device, n, past, kv_heads, page, dtype, layout, False, n + page)
    if n > 4096:
        assert _lib.load().adamas_prefill_workspace_bytes(n, past, 32, kv_heads) == 0, "one range of all tiles"
    ref, mag = _reference(q, k, v, past)
    # as at the edges above
    u = 2.0 ** (-11 if dtype == torch.float16 else -8)
    bound = u * (mag + ref.abs()) + 2.0 ** -14 * mag + 2.0 ** -25 * v.double().abs().sum(0).max()
    assert bool(((U.prefill_forward(q, ctrl, 0).double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("kv_heads,page,dtype,layout", [
    (32, 1 << 19, torch.float16, 0),          # K and V of a page exactly 2^32 bytes apart
    (32, (1 << 19) + 1, torch.float16, 0),    # and a little more, addresses made in every lane
    (8, 1 << 21, torch.bfloat16, 1),
    (8, (1 << 21) - 1, torch.float16, 0),     # a little less
])
def test_prefill_attention_of_a_whole_context_in_one_page(gpu_device, kv_heads, page, dtype, layout):
    n, past = 70, 200
    ctrl, q, k, v = _cache(gpu_device, n, past, kv_heads, page, dtype, layout, False, kv_heads)
    ref, mag = _reference(q, k, v, past)
    # as at the edges above
    u = 2.0 ** (-11 if dtype == torch.float16 else -8)
    bound = u * (mag + ref.abs()) + 2.0 ** -14 * mag + 2.0 ** -25 * v.double().abs().sum(0).max()
    assert bool(((U.prefill_forward(q, ctrl, 0).double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("n,past,kv_heads,dtype", [
    (1200, 0, 32, torch.float16), (850, 0, 8, torch.bfloat16),      # token ranges
    (200, 1200, 32, torch.float16), (64, 1000, 8, torch.float16),
    (700, 0, 32, torch.float16), (2000, 553, 8, torch.bfloat16),    # one range of all tiles
])
def test_prefill_attention_of_both_workgroups_is_the_same(gpu_device, n, past, kv_heads, dtype):
    """Pages of 16 slots get workgroups of four waves, pages of 4 those of eight."""
    ctrl, q, k, v = _cache(gpu_device, n, past, kv_heads, 16, dtype, 0, False, n)
    other = U.InferenceController(1, 32, 128, 4, 64, n + past, dtype, gpu_device, num_kv_heads=kv_heads)
    other.prepare_hadamard(n + past)
    U.append_kvh(k, v, None, other, 0)
    assert torch.equal(U.prefill_forward(q, ctrl, 0), U.prefill_forward(q, other, 0))


def test_prefill_attention_of_a_misaligned_view(gpu_device):
    ctrl, q, k, v = _cache(gpu_device, 40, 0, 32, 16, torch.float16, 0, False, 3)
    flat = torch.empty(q.numel() + 1, dtype=q.dtype, device=gpu_device)
    flat[1:] = q.reshape(-1)
    assert torch.equal(U.prefill_forward(flat[1:].view(q.shape), ctrl, 0), U.prefill_forward(q, ctrl, 0))


def _rms(x):
    return float(x.double().pow(2).mean().sqrt())


@pytest.mark.parametrize("n,past,kv_heads,dtype,sharpness", [
    (300, 900, 8, torch.float16, 1.0),     # grouped heads behind a cache, token ranges merged
    (300, 900, 8, torch.bfloat16, 1.0),
    (1200, 300, 4, torch.bfloat16, 3.0),
    (777, 0, 32, torch.float16, 3.0),      # one weight near 1, the maximum found late
    (777, 0, 8, torch.bfloat16, 3.0),
    (400, 1100, 32, torch.bfloat16, 1.0),
])
def test_prefill_attention_error_is_that_of_its_roundings(gpu_device, n, past, kv_heads, dtype, sharpness):
    """rms error against float64.  Grouped heads behind a cache: the rounding of the output and nothing
    else (weights of 22 or 16 significant bits add less than 1e-4 of it).  The other calls: the weights
    are rounded to 16 bits too, relative to the largest.  More than 10^6 values: the rms of two
    realisations of the same roundings differs by about 0.1 %, 2 % are allowed."""
    ctrl, q, k, v = _cache(gpu_device, n, past, kv_heads, 16, dtype, 0, False, n + past)
    q = (q * sharpness).to(dtype)
    ref, _ = _reference(q, k, v, past)
    best = ref
    if past == 0 or kv_heads == 32:
        best = torch.empty_like(ref)
        hidden = (torch.arange(n + past, device=gpu_device)[None] >
                  (past + torch.arange(n, device=gpu_device))[:, None])
        for h in range(32):
            kh, vh = (x[:, h // (32 // kv_heads)].double() for x in (k, v))
            s = (q[:, h].double() @ kh.T / math.sqrt(128)).masked_fill(hidden, -math.inf)
            w = torch.exp(s - s.amax(-1, keepdim=True))
            best[:, h] = (w.to(dtype).double() @ vh) / w.sum(-1, keepdim=True)
    err = _rms(U.prefill_forward(q, ctrl, 0).double() - ref)
    assert err <= 1.02 * _rms(best.to(dtype).double() - ref)


@pytest.mark.parametrize("n,past,kv_heads,dtype", [
    (70, 0, 32, torch.float16), (200, 41, 8, torch.bfloat16), (200, 41, 8, torch.float16),
    (90, 5000, 8, torch.float16), (90, 5000, 32, torch.bfloat16)])
def test_prefill_attention_of_infinite_values(gpu_device, n, past, kv_heads, dtype):
    """Equal weights; an infinite channel of a value is infinite, with its sign, for the query tokens that see
    it, does not reach the tiles of tokens before it, and no other channel sees it.  (For the queries of its
    own tile that do not see it, zero times an infinity is NaN, as in any product with a masked matrix.)"""
    ctrl, q, k, v = _cache(gpu_device, n, past, kv_heads, 16, dtype, 0, False, n)
    mid, last = past + n // 2, past + n - 1
    v[mid, :, 5] = math.inf
    v[last, :, 70] = -math.inf
    ctrl.clean_states()
    ctrl.prepare_hadamard(past + n)
    U.append_kvh(k, v, None, ctrl, 0)
    o = U.prefill_forward(torch.zeros_like(q), ctrl, 0)
    assert bool((o[n // 2:, :, 5] == math.inf).all()) and bool((o[n - 1, :, 70] == -math.inf).all())
    rest = torch.ones(128, dtype=torch.bool, device=gpu_device)
    rest[[5, 70]] = False
    assert bool(o[:, :, rest].isfinite().all())
    # queries whose last 256-row block of stacked rows ends before the tile of the token
    blocks = (max(0, (mid // 64 * 64) - past) * 32 // kv_heads) // 256
    assert bool(o[:blocks * 256 * kv_heads // 32, :, 5].isfinite().all())


@pytest.mark.parametrize("scale", [-0.11, 0.0, -0.0, 1e-30])
@pytest.mark.parametrize("n,past,kv_heads,dtype", [(90, 0, 32, torch.float16), (130, 77, 8, torch.bfloat16)])
def test_prefill_attention_of_any_scale(gpu_device, n, past, kv_heads, dtype, scale):
    """No scale lets a query see a later token or loses the maximum.  Bound as in the test of the edges."""
    ctrl, q, k, v = _cache(gpu_device, n, past, kv_heads, 16, dtype, 0, False, 5)
    lib = _lib.load()
    o = torch.empty_like(q)
    need = lib.adamas_prefill_workspace_bytes(n, past, 32, kv_heads)
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device=gpu_device)
    rc = lib.adamas_prefill_attention(q.data_ptr(), ctrl.kv_cache.buf_layer(0).data_ptr(), ctrl.seqs.table_ptr(0),
                                      o.data_ptr(), ws.data_ptr(), need, n, past, 32, kv_heads, 128, 16, scale,
                                      ctrl.kv_flags, _lib.current_stream())
    assert rc == 0
    ref, mag = _reference(q, k, v, past, scale)
    u = 2.0 ** (-11 if dtype == torch.float16 else -8)
    bound = u * (mag + ref.abs()) + 2.0 ** -14 * mag + 2.0 ** -25 * v.double().abs().sum(0).max()
    assert bool(((o.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("n,past,kv_heads,layout", [(40, 0, 32, 0), (33, 70, 8, 1)])
def test_prefill_attention_carries_gradients_and_transforms(gpu_device, n, past, kv_heads, layout):
    """Gradients of q against float64 autograd, forward mode against the same, vmap against single calls."""
    ctrl, q, k, v = _cache(gpu_device, n, past, kv_heads, 16, torch.float16, layout, False, 7)
    g = torch.Generator(device=gpu_device).manual_seed(8)
    w = torch.randn(q.shape, generator=g, device=gpu_device)

    def reference(x):
        group = 32 // kv_heads
        kk, vv = (t.double().repeat_interleave(group, dim=1).transpose(0, 1) for t in (k, v))
        hidden = (torch.arange(n + past, device=gpu_device)[None] >
                  past + torch.arange(n, device=gpu_device)[:, None])
        s = x.transpose(0, 1) @ kk.transpose(1, 2) / math.sqrt(128)
        return (s.masked_fill(hidden, -math.inf).softmax(-1) @ vv).transpose(0, 1)

    plain = U.prefill_forward(q, ctrl, 0)
    x = q.clone().requires_grad_()
    o = U.prefill_forward(x, ctrl, 0)
    torch.testing.assert_close(o, plain, rtol=2e-3, atol=2e-3)     # both rounded to fp16
    o.backward(w.half())
    x64 = q.double().requires_grad_()
    reference(x64).backward(w.half().double())
    # fp32 all the way, the gradient rounded to fp16 (2^-11)
    torch.testing.assert_close(x.grad.double(), x64.grad, rtol=1e-3, atol=1e-4)
    with torch.no_grad():
        assert U.prefill_forward(x, ctrl, 0).grad_fn is None and torch.equal(U.prefill_forward(x, ctrl, 0), plain)
    _, tangent = torch.func.jvp(lambda t: U.prefill_forward(t, ctrl, 0), (q,), (w.half(),))
    _, want = torch.func.jvp(reference, (q.double(),), (w.half().double(),))
    torch.testing.assert_close(tangent.double(), want, rtol=1e-3, atol=1e-4)
    both = torch.func.vmap(lambda t: U.prefill_forward(t, ctrl, 0))(torch.stack([q, -q]))
    torch.testing.assert_close(both[0], plain, rtol=2e-3, atol=2e-3)
    torch.testing.assert_close(both[1], U.prefill_forward(-q, ctrl, 0), rtol=2e-3, atol=2e-3)


def test_prefill_attention_launches_on_the_device_of_its_tensors(gpu_device, monkeypatch):
    ctrl, q, _, _ = _cache(gpu_device, 40, 0, 32, 16, torch.float16, 0, False, 3)
    entered = []
    enter = torch.cuda.device.__enter__
    monkeypatch.setattr(torch.cuda.device, "__enter__", lambda self: (entered.append(self.idx), enter(self))[1])
    U.prefill_forward(q, ctrl, 0)
    assert entered == []
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: q.device.index + 1)   # (another one than q's)
    U.prefill_forward(q, ctrl, 0)
    assert entered == [q.device.index]


@pytest.mark.parametrize("heads,kv_heads,n,past,dtype,page", [
    (24, 8, 200, 0, torch.float16, 16),      # groups of 3: the heads of a query cross from one 256-row block to the next
    (24, 8, 86, 2000, torch.bfloat16, 16),   # the same, token ranges merged
    (40, 8, 257, 63, torch.bfloat16, 12),    # groups of 5
    (40, 8, 52, 5000, torch.float16, 16),
    (32, 1, 70, 0, torch.float16, 16),       # one key/value head
    (32, 1, 33, 3000, torch.bfloat16, 16),
    (8, 1, 300, 100, torch.float16, 1),
])
def test_prefill_attention_of_other_groups(gpu_device, heads, kv_heads, n, past, dtype, page):
    dev = gpu_device
    g = torch.Generator(device=dev).manual_seed(heads + n)
    length = n + past
    ctrl = U.InferenceController(1, heads, 128, page, 64, length, dtype, dev, num_kv_heads=kv_heads)
    k, v = (torch.randn(length, kv_heads, 128, generator=g, device=dev).to(dtype) for _ in range(2))
    q = torch.randn(n, heads, 128, generator=g, device=dev).to(dtype)
    ctrl.prepare_hadamard(length)
    U.append_kvh(k, v, None, ctrl, 0)
    split = _lib.load().adamas_prefill_workspace_bytes(n, past, heads, kv_heads) > 0
    assert split or past < 2000, "the token ranges are tested where they are meant to be"
    ref, mag = _reference(q, k, v, past)
    # as at the edges above
    u = 2.0 ** (-11 if dtype == torch.float16 else -8)
    bound = u * (mag + ref.abs()) + 2.0 ** -14 * mag + 2.0 ** -25 * v.double().abs().sum(0).max()
    assert bool(((U.prefill_forward(q, ctrl, 0).double() - ref).abs() <= bound).all())
