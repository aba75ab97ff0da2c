"""Attention over lists of positions and over all positions, against float64 torch: row counts around the sizes of a
split and of the workgroups, page sizes that are no power of two, odd head groups, unused entries, values that are
infinite where nothing looks."""
import pytest
import torch

import adamas_amd.utils as U

pytestmark = pytest.mark.gpu


def _setup(dev, lens, page, heads, kv_heads, dtype, layout):
    g = torch.Generator(device=dev).manual_seed(sum(lens) + page)
    c = U.InferenceController(1, heads, 128, page, 64, max(lens) + 1, dtype, dev, batch_size=len(lens),
                              num_kv_heads=kv_heads, layout=layout,
                              page_order=torch.randperm(-(-(max(lens) + 1) // page) * len(lens)).tolist())
    c.pool.kv.zero_()
    c.prepare_hadamard(lens)
    kv = []
    for b, n in enumerate(lens):
        k, v = (torch.randn(n, kv_heads, 128, generator=g, device=dev).to(dtype) for _ in range(2))
        kv.append([k, v])
    c.begin_forward(1)
    q = torch.randn(len(lens), heads, 128, generator=g, device=dev).to(dtype)
    return c, q, kv, g


def _append(c, kv):
    for b, (k, v) in enumerate(kv):
        U.append_kvh(k, v, None, c, 0, seq_idx=b)


def _want(q, k, v, pos):
    """q [H, 128], pos [H, n] (-1 = unused, the newest token is added) -> [H, 128] in float64."""
    heads, kv_heads = q.shape[0], k.shape[1]
    kv_of = torch.arange(heads, device=q.device) // (heads // kv_heads)
    pos = torch.cat((pos, torch.full_like(pos[:, :1], k.shape[0] - 1)), 1).long()
    unused = (pos < 0) | (pos >= k.shape[0])
    at = pos.clamp(0, k.shape[0] - 1)
    kk, vv = k[at, kv_of[:, None]].double(), v[at, kv_of[:, None]].double()
    s = (kk * q.double()[:, None]).sum(-1) / 128 ** 0.5
    w = s.masked_fill(unused, -torch.inf).softmax(-1)
    return (w[..., None] * vv.masked_fill(unused[..., None], 0)).sum(1)


@pytest.mark.parametrize("lens,rows,page,heads,kv_heads,dtype,layout", [
    ([700], 1, 16, 32, 32, torch.float16, 0),
    ([700], 63, 1, 32, 8, torch.float16, 0), ([700], 64, 24, 32, 32, torch.bfloat16, 1),
    ([700], 127, 16, 24, 8, torch.float16, 0), ([700], 128, 16, 40, 8, torch.float16, 1),
    ([700], 511, 5, 32, 4, torch.bfloat16, 0), ([700], 512, 32, 32, 32, torch.float16, 0),
    ([2500], 2047, 16, 32, 8, torch.float16, 0), ([2500], 2048, 16, 8, 8, torch.float16, 0),
    ([5000], 4100, 48, 32, 32, torch.float16, 0),
    ([300, 90, 2], 100, 16, 32, 8, torch.float16, 0), ([260] * 20, 200, 7, 32, 32, torch.bfloat16, 0),
])
def test_lists_of_positions(gpu_device, lens, rows, page, heads, kv_heads, dtype, layout):
    c, q, kv, g = _setup(gpu_device, lens, page, heads, kv_heads, dtype, layout)
    sel = torch.full((len(lens) * heads, rows), -1, dtype=torch.int32, device=gpu_device)
    for r in range(sel.shape[0]):
        n = lens[r // heads] - 1
        if n < 1:
            continue
        some = torch.randperm(n, generator=g, device=gpu_device)[:rows].int()
        at = torch.randperm(rows, generator=g, device=gpu_device)[:some.numel()]
        sel[r, at] = some
        sel[r, torch.rand(rows, generator=g, device=gpu_device) < 0.1] = -1      # unused in the middle too
        sel[r, rows // 2] = 1 << 30 if r % 2 else -7                             # outside the sequence
    # the first token of every sequence is what a clamped position reads: infinite and attended by nobody
    sel[sel == 0] = -1
    for b, n in enumerate(lens):
        if n > 1:
            kv[b][1][0] = torch.inf
    _append(c, kv)
    got = U.decode_sparse_attn(q, c, 0, sel)
    ulp = 2.0 ** (-10 if dtype == torch.float16 else -7)
    for b in range(len(lens)):
        want = _want(q[b], *kv[b], sel.view(len(lens), heads, rows)[b])
        # one rounding of the result, and fp32 sums of up to 4101 terms of size 1
        assert bool(((got[b].double() - want).abs() <= ulp * want.abs() + 2e-5).all()), b


@pytest.mark.parametrize("rows,used,batch,kv_heads", [
    (63, 5, 3, 32), (127, 1, 4, 8), (128, 33, 4, 32), (511, 40, 8, 32), (512, 0, 20, 8), (999, 65, 3, 32),
    (999, 130, 20, 8), (2047, 257, 8, 32), (2500, 3, 2, 8),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_lists_mostly_unused(gpu_device, rows, used, batch, kv_heads, dtype):
    """Whole tiles without an entry, for lists of every kind of workgroup: the first sequence's list is full, the others
    have `used` entries, in front or (every other sequence) at the end."""
    lens = [2600] + [max(used, 1) + 2] * (batch - 1)
    c, q, kv, g = _setup(gpu_device, lens, 16, 32, kv_heads, dtype, 0)
    sel = torch.full((batch, 32, rows), -1, dtype=torch.int32, device=gpu_device)
    for b, n in enumerate(lens):
        kv[b][1][0] = torch.inf      # (what a clamped position reads, attended by nobody)
        m = rows if b == 0 else used
        for h in range(32):
            some = torch.randperm(n - 2, generator=g, device=gpu_device)[:m].int() + 1
            sel[b, h, (slice(0, m) if b % 2 == 0 else slice(rows - m, rows))] = some
    _append(c, kv)
    got = U.decode_sparse_attn(q, c, 0, sel.view(batch * 32, rows))
    ulp = 2.0 ** (-10 if dtype == torch.float16 else -7)
    for b in range(batch):
        want = _want(q[b], *kv[b], sel[b])
        # one rounding of the result, and fp32 sums of up to 2501 terms of size 1
        assert bool(((got[b].double() - want).abs() <= ulp * want.abs() + 2e-5).all()), b


@pytest.mark.parametrize("lens,page,heads,kv_heads", [
    ([64], 16, 32, 32), ([129], 5, 32, 8), ([1000], 24, 32, 32), ([1409], 16, 24, 8), ([4096], 48, 32, 32),
    ([150, 250, 3], 16, 32, 32), ([600, 1000], 7, 32, 8),
])
def test_all_positions(gpu_device, lens, page, heads, kv_heads):
    c, q, kv, _ = _setup(gpu_device, lens, page, heads, kv_heads, torch.float16, 0)
    _append(c, kv)
    got = U.decode_sparse_attn(q, c, 0, None)
    for b, n in enumerate(lens):
        pos = torch.arange(n - 1, device=gpu_device).expand(heads, n - 1)
        want = _want(q[b], *kv[b], pos)
        assert bool(((got[b].double() - want).abs() <= 2.0 ** -10 * want.abs() + 2e-5).all()), b
