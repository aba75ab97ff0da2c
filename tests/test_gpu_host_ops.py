"""The operators of a decode token by way of the native host function and by the general way: the same tensors,
and every call that the native function does not serve goes the general way, errors included."""
import numpy as np
import pytest
import torch

import adamas_amd.utils as U

pytestmark = pytest.mark.gpu


class _Nothing:
    """Serves no call."""
    def __getattr__(self, name):
        return lambda *args: None


class _Counting:
    def __init__(self, host):
        self.host, self.served = host, []

    def __getattr__(self, name):
        def call(*args):
            out = getattr(self.host, name)(*args)
            self.served.append(out is not None)
            return out
        return call


def _controller(dev, lens, budget, kv_heads, dtype, layout=0, layers=2):
    c = U.InferenceController(layers, 32, 128, 16, budget, max(lens) + 8, dtype, dev, batch_size=len(lens),
                              num_kv_heads=kv_heads, layout=layout)
    g = torch.Generator(device=dev).manual_seed(5)
    c.pool.kv.copy_(torch.randn(c.pool.kv.shape, generator=g, device=dev))
    c.pool.codes.copy_(torch.randint(-32768, 32768, c.pool.codes.shape, generator=g, device=dev))
    c.prepare_hadamard(lens)
    c.begin_forward(1)
    rows = [torch.randn(len(lens), h, 128, generator=g, device=dev).to(dtype) for h in (32, kv_heads, kv_heads)]
    return c, rows


def _token(c, q, k, v, layer):
    x = torch.cat((q, k)) if q.shape == k.shape else torch.cat((q.view(-1, 128), k.view(-1, 128)))
    h = U.hadamard_transform(x, scale=c.hadamard_scale)
    code = U.append_kvh(k, v, h, c, layer)
    code_q = U.append_kvh(k, v, None, c, layer, q=q)
    est = U.decode_estimate(code, c, layer)
    U.decode_topk(est, c)
    sel, val = c.topk_dindices_buffer.clone(), c.topk_dout_buffer.clone()
    out = [h, code, code_q, est, sel, val, U.decode_sparse_attn(q, c, layer, sel),
           U.decode_sparse_attn(q, c, layer, c.kv_indices_without_last), U.decode_sparse_attn(q, c, layer, None),
           U.decode_step(q, code, c, layer)]
    U.decode_topk(est.clone(), c, False)
    out += [c.topk_dindices_buffer.clone(), c.pool.kv.clone(), c.pool.codes.clone()]
    if est.dim() == 3:      # nothing is written past the end of a shorter sequence
        for b, n in enumerate(c.seqs.lengths):
            est[b, :, n - 1:] = 0
        c._estimate_version = c._estimate_buf._version
    assert est._base is c._estimate_buf and c._estimate_version == c._estimate_buf._version
    return out


@pytest.mark.parametrize("lens,budget,kv_heads,dtype,layout,layer", [
    ([700], 64, 32, torch.float16, 0, 0),
    ([700], 300, 8, torch.bfloat16, 1, -1),
    ([400, 37, 900], 128, 8, torch.float16, 0, 1),
    ([130, 3], 400, 32, torch.bfloat16, 0, 1),      # the budget holds the longest sequence
])
def test_native_and_general_way_agree(gpu_device, monkeypatch, lens, budget, kv_heads, dtype, layout, layer):
    got = []
    for host in (_Nothing(), _Counting(U._load_host())):
        monkeypatch.setattr(U, "_host", host)
        c, (q, k, v) = _controller(gpu_device, lens, budget, kv_heads, dtype, layout)
        for t in (q, k, v):
            t.requires_grad_()      # (results carry no gradient either way)
        c.workspace(c.inference_page_budget)
        c.topk_workspace(max(lens) - 1, c.inference_page_budget - 1)
        got.append(_token(c, q.detach(), k, v, layer))
    # a batch that ends up longer than its budget serves every call; all of them are served here
    assert host.served and all(host.served)
    for a, b in zip(*got):
        assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)
        assert not a.requires_grad and not b.requires_grad


def test_calls_that_go_the_general_way(gpu_device, monkeypatch):
    dev = gpu_device
    host = _Counting(U._load_host())
    monkeypatch.setattr(U, "_host", host)
    c, (q, k, v) = _controller(dev, [700], 64, 32, torch.float16)

    def general(call):
        host.served.clear()
        out = call()
        assert host.served == [False]
        return out

    code = U.append_kvh(k, v, None, c, 0, q=q)
    general(lambda: U.decode_step(q, code, c, 0))                      # the workspace is made there
    want = U.decode_step(q, code, c, 1)
    assert host.served == [False, True]

    class Sub(torch.Tensor):
        pass

    for index in (np.int64(1), torch.tensor(1)):
        assert torch.equal(general(lambda: U.decode_step(q, code, c, index)), want)
    assert torch.equal(general(lambda: U.decode_step(q.as_subclass(Sub), code, c, 1)), want)

    class Other(U.InferenceController):
        max_len_now = property(lambda self: 700)
    c.__class__ = Other
    assert torch.equal(general(lambda: U.decode_step(q, code, c, 1)), want)
    c.__class__ = U.InferenceController

    x = torch.randn(4, 128, device=dev).half()
    y = U.hadamard_transform(x)
    host.served.clear()
    assert U.hadamard_transform(x, True) is x and torch.equal(x, y) and host.served == [True]
    assert torch.equal(general(lambda: U.hadamard_transform(x, scale=1)), U.hadamard_transform(x, scale=1.0))
    est = U.decode_estimate(code, c, 0)
    est.mul_(1)                                                        # edited: arbitrary keys from now on
    U.decode_topk(est, c)

    for call, what in ((lambda: U.decode_step(q.cpu(), code, c, 0), "must be a CUDA"),
                       (lambda: U.decode_step(q.float(), code, c, 0), "must have dtype"),
                       (lambda: U.decode_step(torch.cat((q, q), 2)[:, :, :128], code, c, 0), "must be contiguous"),
                       (lambda: U.decode_step(q[:, :8].contiguous(), code, c, 0), r"q must be \[B, H, D\]"),
                       (lambda: U.decode_step(torch.cat((q, q)), code, c, 0), r"q must be \[B, H, D\]"),
                       (lambda: U.decode_step(q, code[:, :8].contiguous(), c, 0), "packed query code"),
                       (lambda: U.decode_step(q, code.long(), c, 0), "packed query code"),
                       (lambda: U.decode_step(q[:, :8].contiguous(), code, c, 0, return_indices=True), "q must be"),
                       (lambda: U.append_kvh(k, v[:, :8].contiguous(), None, c, 0, q=q), "same shape"),
                       (lambda: U.append_kvh(k, v, None, c, 0, q=q[:, :8].contiguous()), "q must be"),
                       (lambda: U.decode_estimate(code.long(), c, 0), "packed query code"),
                       (lambda: U.decode_topk(est[:, :10], c), "fewer candidates"),
                       (lambda: U.decode_topk(est.float(), c), "float16"),
                       (lambda: U.decode_sparse_attn(q, c, 0, c.topk_dindices_buffer.long()), "must have dtype"),
                       (lambda: U.hadamard_transform(x[:, :64].contiguous()), "last dimension")):
        with pytest.raises(RuntimeError, match=what):
            call()
    with pytest.raises(IndexError):
        U.decode_step(q, code, c, 2)
    assert torch.equal(general(lambda: U.decode_step(q.view(8, 4, 128), code, c, 1)).view_as(want), want)
    batched = torch.func.vmap(lambda t: t * 1)(q)
    assert torch.equal(U.decode_step(batched, code, c, 1), want)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda t: U.decode_step(t, code, c, 1))(q[None])


def test_results_of_the_library_are_errors_with_its_text(gpu_device):
    c, (q, k, v) = _controller(gpu_device, [700], 64, 32, torch.float16)
    code = U.append_kvh(k, v, None, c, 0, q=q)
    U.decode_step(q, code, c, 0)
    odd = torch.empty(32 * 128 + 1, device=gpu_device, dtype=torch.float16)[1:].view(1, 32, 128)
    with pytest.raises(RuntimeError, match="adamas_decode_step failed with error code -4"):
        U.decode_step(odd, code, c, 0)


@pytest.mark.parametrize("op", ["hadamard", "hadamard in place", "append", "estimate", "topk", "sparse_attn", "step"])
def test_on_the_current_stream(gpu_device, monkeypatch, op):
    """The native function launches behind what its stream holds: on a side stream the input gets its values behind
    matrix products that outlast the call, and nothing waits in between."""
    c, (q, k, v) = _controller(gpu_device, [700], 64, 32, torch.float16)
    code = U.append_kvh(k, v, None, c, 0, q=q)
    est = U.decode_estimate(code, c, 0)
    U.decode_topk(est, c)
    sel = c.topk_dindices_buffer.clone()
    U.decode_step(q, code, c, 0)
    assert c.seq_lens.tolist() == [700]     # (looked at: the lengths are there for every stream)

    def topk(x):
        U.decode_topk(x, c, True)
        return c.topk_dindices_buffer.clone()

    value, call = {"hadamard": (q, U.hadamard_transform),
                   "hadamard in place": (q, lambda x: U.hadamard_transform(x, True)),
                   "append": (q, lambda x: U.append_kvh(k, v, None, c, 0, q=x)),
                   "estimate": (code, lambda x: U.decode_estimate(x, c, 0)),
                   "topk": (est, topk),
                   "sparse_attn": (q, lambda x: U.decode_sparse_attn(x, c, 0, sel)),
                   "step": (q, lambda x: U.decode_step(x, code, c, 0))}[op]
    want = call(value.clone())
    early = call(torch.zeros_like(value)).clone()
    assert not torch.equal(early, want)     # what a launch ahead of the values would give
    want, x = want.clone(), torch.zeros_like(value)
    a = torch.randn(8192, 8192, device=gpu_device)
    a @ a
    host = _Counting(U._load_host())
    monkeypatch.setattr(U, "_host", host)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        for _ in range(6):
            a = a @ a * 1e-4
        busy = torch.cuda.Event()
        busy.record()
        x.copy_(value)
        got = call(x)
        assert not busy.query()             # (the products are still running: nobody has waited)
        got = got.clone()
    side.synchronize()
    assert host.served == [True]
    assert torch.equal(got, want)
