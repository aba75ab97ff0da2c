"""GPU parity tests of the two operators the reference's attention module calls around the decode
path: apply_rope_in_place (adamas/utils/__init__.py:26-53, reference test adamas/tests/test_rope.py)
and prefill_forward (adamas/utils/__init__.py:159-201, reference test
adamas/tests/test_prefill_attention.py), and of the module's whole call order, prefill then decode,
through the operator API only (adamas/models/Adamas.py:112-201).

Bars: rotary embedding within one fp16 (bf16) rounding step of the oracle's float64 result plus the
error of an fp32 sine of an fp32 angle: |got - want| <= 1e-3 + |want| * 2**-9 for fp16 (2**-7 for
bf16), far inside the reference test's 5e-3 + 5e-3 |want|.  Attention outputs within 2e-3 max-abs.
"""
import itertools

import numpy as np
import pytest
import torch

import adamas_amd.utils as U
from oracle import adamas_oracle as O
from tests import helpers as T

pytestmark = pytest.mark.gpu
ATTN_TOL_ABS = 2e-3


def _rope_close(got: torch.Tensor, want: np.ndarray) -> bool:
    rel = 2.0 ** -7 if got.dtype == torch.bfloat16 else 2.0 ** -9
    return bool((np.abs(T.np16(got).astype(np.float64) - want) <= 1e-3 + np.abs(want) * rel).all())


# the grid of the reference's test (adamas/tests/test_rope.py:33), thinned to its corners and middle
@pytest.mark.parametrize("past_kv_len, seq_len",
                         list(itertools.product([13, 244, 1110], [2, 31, 251])) + [(0, 1), (32767, 1)])
def test_apply_rope_in_place_reference_grid(gpu_device, past_kv_len, seq_len):
    g = torch.Generator().manual_seed(past_kv_len * 1000 + seq_len)
    q = torch.randn(seq_len, 32, 128, generator=g).half()
    k = torch.randn(seq_len, 32, 128, generator=g).half()
    qd, kd = q.to(gpu_device), k.to(gpu_device)
    assert U.apply_rope_in_place(qd, kd, past_kv_len) is None   # in place, like the reference
    assert _rope_close(qd, O.rope(T.np16(q), past_kv_len))
    assert _rope_close(kd, O.rope(T.np16(k), past_kv_len))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("heads, kv_heads", [(32, 8), (5, 5), (40, 40)])
def test_apply_rope_in_place_heads_scale_theta(gpu_device, dtype, heads, kv_heads):
    g = torch.Generator().manual_seed(heads)
    q = torch.randn(70, heads, 128, generator=g).to(dtype)
    k = torch.randn(70, kv_heads, 128, generator=g).to(dtype)
    qd, kd = q.to(gpu_device), k.to(gpu_device)
    U.apply_rope_in_place(qd, kd, 9000, rope_scale=2.0, rope_theta=5e5)
    assert _rope_close(qd, O.rope(T.np16(q), 9000, 2.0, 5e5))
    assert _rope_close(kd, O.rope(T.np16(k), 9000, 2.0, 5e5))


def test_apply_rope_in_place_long_prefill_matches_table_kernel(gpu_device):
    """32768 rows at once (more rows than grid rows) against the oracle on samples, and against the
    table-driven rotary kernel of the decoder on every element."""
    n = 70000
    g = torch.Generator().manual_seed(5)
    qkv = torch.randn(n, 3, 2, 128, generator=g).half().to(gpu_device)
    q, k = qkv[:, 0].contiguous(), qkv[:, 1].contiguous()
    q0, k0 = q.clone(), k.clone()
    U.apply_rope_in_place(q, k, 17)
    for r in (0, 1, 65534, 65535, 65536, n - 1):
        assert _rope_close(q[r:r + 1], O.rope(T.np16(q0[r:r + 1]), 17 + r))
        assert _rope_close(k[r:r + 1], O.rope(T.np16(k0[r:r + 1]), 17 + r))
    ang = (torch.arange(n + 17, dtype=torch.float32)[:, None] *
           torch.from_numpy(O.rope_freqs())[None, :])
    q2, k2, _ = U.rope_split(qkv, ang.cos().to(gpu_device), ang.sin().to(gpu_device), start_pos=17)
    assert (q.float() - q2.float()).abs().max().item() <= 4e-3   # one rounding step at |x| < 8
    assert (k.float() - k2.float()).abs().max().item() <= 4e-3


def test_apply_rope_in_place_rejects_bad_arguments(gpu_device):
    q = torch.zeros(4, 32, 128, dtype=torch.float16, device=gpu_device)
    with pytest.raises(RuntimeError):
        U.apply_rope_in_place(q, torch.zeros(3, 32, 128, dtype=torch.float16, device=gpu_device), 0)
    with pytest.raises(RuntimeError):
        U.apply_rope_in_place(q, q.float(), 0)
    with pytest.raises(RuntimeError):
        U.apply_rope_in_place(q.float(), q.float(), 0)
    with pytest.raises(RuntimeError):
        U.apply_rope_in_place(q, q[:, :, :64], 0)
    with pytest.raises(RuntimeError):
        U.apply_rope_in_place(q.cpu(), q.cpu(), 0)
    with pytest.raises(RuntimeError):
        U.apply_rope_in_place(q, q.clone(), -1)
    with pytest.raises(RuntimeError):
        U.apply_rope_in_place(q, q.clone(), 0, rope_scale=0.0)
    U.apply_rope_in_place(q[:0], q[:0].clone(), 0)   # no rows: nothing to do


@pytest.mark.parametrize("layout", [U.TensorLayout.NHD, U.TensorLayout.HND])
@pytest.mark.parametrize("heads, kv_heads, page_size, n_first, n_second",
                         [(32, 32, 16, 333, 0), (32, 4, 16, 200, 77), (32, 32, 1, 50, 50),
                          (64, 16, 32, 5000, 300)])
def test_prefill_forward_causal(gpu_device, layout, heads, kv_heads, page_size, n_first, n_second):
    """Fresh prompt (q covers the whole sequence), then a second piece whose queries also see the
    first one; shuffled pages."""
    g = torch.Generator().manual_seed(n_first + heads)
    total = n_first + n_second
    q = torch.randn(total, heads, 128, generator=g).half()
    k = torch.randn(total, kv_heads, 128, generator=g).half()
    v = torch.randn(total, kv_heads, 128, generator=g).half()
    ctrl = T.make_controller(gpu_device, total + 40, 64, page_size, shuffle_seed=3, num_heads=heads,
                             num_kv_heads=kv_heads, layout=layout)
    done = 0
    for n in (n_first, n_second):
        if n == 0:
            continue
        T.fill_sequence(ctrl, k[done:done + n].to(gpu_device), v[done:done + n].to(gpu_device))
        done += n
        o = U.prefill_forward(q[done - n:done].to(gpu_device).contiguous(), ctrl, 0)
        assert o.shape == (n, heads, 128) and o.dtype == torch.float16
        rows = np.unique(np.concatenate((np.arange(min(n, 8)), np.arange(max(0, n - 8), n),
                                         np.random.default_rng(n).integers(0, n, 16))))
        kk, vv = T.np16(k[:done]), T.np16(v[:done])
        for r in rows:   # row r of this piece is token done - n + r of the sequence
            upto = done - n + r + 1
            want = O.causal_attention(T.np16(q[done - n + r:done - n + r + 1]), kk[:upto], vv[:upto])
            assert np.abs(T.np16(o[r:r + 1]).astype(np.float64) - want).max() <= ATTN_TOL_ABS, r


def test_prefill_forward_rejects_bad_arguments(gpu_device):
    ctrl = T.make_controller(gpu_device, 64, 16, 16, num_heads=32)
    k = torch.zeros(10, 32, 128, dtype=torch.float16, device=gpu_device)
    T.fill_sequence(ctrl, k, k)
    with pytest.raises(RuntimeError):
        U.prefill_forward(torch.zeros(11, 32, 128, dtype=torch.float16, device=gpu_device), ctrl, 0)
    with pytest.raises(RuntimeError):
        U.prefill_forward(torch.zeros(10, 64, 128, dtype=torch.float16, device=gpu_device), ctrl, 0)
    with pytest.raises(RuntimeError):
        U.prefill_forward(torch.zeros(10, 32, 128, dtype=torch.float32, device=gpu_device), ctrl, 0)
    ctrl2 = T.make_controller(gpu_device, 64, 16, 16, num_heads=32, batch_size=2)
    with pytest.raises(RuntimeError):
        U.prefill_forward(k, ctrl2, 0)


def _module_forward(x_q, x_k, x_v, ctrl, layer, scale):
    """The call order of the reference's attention module between its projections
    (adamas/models/Adamas.py:112-201), with this package's operators under the reference's names.
    x_q, x_k, x_v [q_len, H, 128] are the projected states before the rotary embedding."""
    q_len = x_q.shape[0]
    U.apply_rope_in_place(x_q, x_k, ctrl.kv_cache.seqlen - q_len)
    if q_len > 1:
        h = U.hadamard_transform(x_k, inplace=False, scale=scale)
        U.append_kvh(x_k, x_v, h, ctrl, layer)
        return U.prefill_forward(x_q, ctrl, layer)
    h = torch.cat((x_q, x_k), dim=0)
    U.hadamard_transform(h, inplace=True, scale=scale)
    q_code = U.append_kvh(x_k, x_v, h, ctrl, layer)
    if not ctrl.need_estimate():
        return U.decode_sparse_attn(x_q, ctrl, layer, ctrl.kv_indices_without_last)
    est = U.decode_estimate(q_code, ctrl, layer)
    U.decode_topk(est, ctrl)
    return U.decode_sparse_attn(x_q, ctrl, layer, ctrl.topk_dindices_buffer)


@pytest.mark.parametrize("budget", [48, 1 << 20])
def test_module_call_order_prefill_then_decode(gpu_device, budget):
    """Prompt of 300 tokens, then 4 decode steps, driven exactly as the reference's module and model
    drive the operators (prepare_hadamard / begin_forward / end_forward as in llama.py:420-486);
    every output against the oracle on the rotated states."""
    g = torch.Generator().manual_seed(budget % 97)
    heads, prompt, steps = 32, 300, 4
    total = prompt + steps
    xq = torch.randn(total, heads, 128, generator=g).half()
    xk = torch.randn(total, heads, 128, generator=g).half()
    xv = torch.randn(total, heads, 128, generator=g).half()
    # the oracle's view: states rotated at their positions, rounded to fp16 as the cache holds them
    rq = O.rope(T.np16(xq), 0).astype(np.float16).astype(np.float32)
    rk = O.rope(T.np16(xk), 0).astype(np.float16).astype(np.float32)
    vv = T.np16(xv)
    ctrl = T.make_controller(gpu_device, total + 16, budget, 16, shuffle_seed=11)
    ctrl.set_page_budget(budget)

    def run(lo, hi):
        n = hi - lo
        ctrl.prepare_hadamard(n)
        ctrl.begin_forward(n)
        out = _module_forward(xq[lo:hi].to(gpu_device), xk[lo:hi].to(gpu_device),
                              xv[lo:hi].to(gpu_device), ctrl, 0, 1.0)
        ctrl.end_forward()
        return out

    o = run(0, prompt)
    kc, _, _ = T.read_logical_cache(ctrl)
    # the cache holds the kernel's rotated keys: within one fp16 step of the oracle's
    assert np.abs(kc.astype(np.float64) - rk[:prompt]).max() <= 8e-3
    for r in (0, 1, 150, prompt - 1):
        want = O.causal_attention(rq[r:r + 1], kc[:r + 1], vv[:r + 1])
        assert np.abs(T.np16(o[r:r + 1]).astype(np.float64) - want).max() <= 3e-3, r
    for t in range(prompt, total):
        o = run(t, t + 1)
        kc, vc, _ = T.read_logical_cache(ctrl)
        # the selection depends on the exact fp16 states the kernels produced: take the rotated
        # query from the same kernel and the keys from the cache, and check the oracle's step on them
        qg = xq[t:t + 1].to(gpu_device)
        U.apply_rope_in_place(qg, xk[t:t + 1].to(gpu_device), t)
        qd = T.np16(qg)[0]
        assert np.abs(qd.astype(np.float64) - rq[t]).max() <= 8e-3
        step = O.decode_step(qd, kc, vc, min(budget, t + 1))
        assert np.abs(T.np16(o[0]).astype(np.float64) - step["out"]).max() <= ATTN_TOL_ABS, t


def test_operators_launch_on_the_current_stream(gpu_device):
    from adamas_amd import _lib
    side = torch.cuda.Stream(gpu_device)
    for stream in (torch.cuda.current_stream(), side):
        with torch.cuda.stream(stream):
            assert _lib.current_stream() == torch.cuda.current_stream().cuda_stream == stream.cuda_stream
