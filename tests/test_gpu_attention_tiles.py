"""GPU parity of the paged-attention kernel at the edges of its 32-token steps
and partitions: contexts one token around a step, a block and a partition,
every head size at group sizes that leave matrix columns empty, slots past the
context holding NaN and infinities, padded query and output rows.

Bar, elementwise against the float64 oracle: 2^-11 |o| for the fp16 rounding
and 2^-17 max|v| for the fp32 logits (|logit| up to about 16, so exp's argument
is off by at most 2^-19 or so relative to p), the two-part p (2^-22) and the
fp32 sums.
"""
from __future__ import annotations

import sys

import numpy as np
import pytest
import torch

from hip_extends import _lib
from oracle import attention as A

pytestmark = pytest.mark.gpu


def say(msg: str) -> None:
    print(f"[case] {msg}", flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("ctxs,heads,kvh,hs,bs,alibi,pad", [
    ([1, 31, 32, 33, 15, 16, 17, 63, 65], 6, 2, 128, 16, False, 0),
    ([1, 31, 32, 33, 64, 65, 96, 127, 129], 10, 2, 128, 32, True, 0),
    ([4095, 4097, 1], 7, 1, 64, 16, False, 0),        # long partitions, 7 heads per kv head
    ([2049, 255, 2300], 8, 1, 80, 32, False, 8),
    ([300, 1030], 15, 3, 96, 16, True, 24),           # padded query rows
    ([500, 40, 129], 8, 2, 112, 16, False, 8),
    ([700, 33], 6, 2, 256, 32, False, 0),
    ([129, 1000], 3, 1, 256, 16, True, 40),
    ([130] * 70, 16, 8, 64, 32, False, 0),            # more pairs than CUs
    ([130, 1, 33, 600], 8, 8, 64, 32, False, 0),      # one head per kv head, partitioned
    ([1024, 17, 600, 1000, 31], 40, 40, 80, 16, True, 8),   # and one 16-wave workgroup each
    ([1500] * 20, 64, 8, 128, 16, False, 0),          # one 8-wave workgroup per pair
])
def test_paged_attention_edges(hip_device, ctxs, heads, kvh, hs, bs, alibi, pad):
    say(f"attention edges ctxs={ctxs[:9]} heads={heads}/{kvh} hs={hs} bs={bs} alibi={alibi} pad={pad}")
    rng = np.random.default_rng(hs + len(ctxs))
    n, per = len(ctxs), (max(ctxs) + bs - 1) // bs
    tables = rng.permutation(n * per).astype(np.int32).reshape(n, per)
    kc = (rng.standard_normal((n * per, kvh, hs // 8, bs, 8)) * 1.5).astype(np.float16)
    vc = rng.standard_normal((n * per, kvh, hs, bs)).astype(np.float16)
    q = rng.standard_normal((n, heads, hs)).astype(np.float16)
    slopes = (2.0 ** -np.arange(1, heads + 1) * 0.5).astype(np.float32) if alibi else None
    scale = hs ** -0.5
    ref = A.paged_attention(q, kc, vc, tables, np.array(ctxs), scale, slopes)
    bad = np.array([np.nan, np.inf, -np.inf, 65504], np.float16)
    for s, c in enumerate(ctxs):  # the rest of the last block, and the blocks after it
        for t in range(c, min(per * bs, c + 70)):
            kc[tables[s, t // bs], :, :, t % bs, :] = bad[t % 4]
            vc[tables[s, t // bs], :, :, t % bs] = bad[(t + 1) % 4]
    kd, vd = torch.from_numpy(kc).to(hip_device), torch.from_numpy(vc).to(hip_device)
    ptrs = [torch.tensor([t[i].data_ptr() for i in range(n * per)], dtype=torch.int64, device=hip_device)
            for t in (kd, vd)]
    row = heads * hs
    qd = torch.zeros(n, row + pad, dtype=torch.float16, device=hip_device)
    qd[:, :row] = torch.from_numpy(q.reshape(n, row)).to(hip_device)
    out = torch.full((n, row + pad), 7.0, dtype=torch.float16, device=hip_device)
    tab, lens = torch.from_numpy(tables).to(hip_device), torch.tensor(ctxs, dtype=torch.int32, device=hip_device)
    sl = None if slopes is None else torch.from_numpy(slopes).to(hip_device)
    nbytes = _lib.paged_attention_workspace_size(n, heads, kvh, hs, bs, max(ctxs))
    ws = torch.empty(max(16, nbytes), dtype=torch.uint8, device=hip_device)
    outs = []
    for _ in range(2):
        _lib.call("dw4_paged_attention", n, heads, kvh, hs, bs, qd.data_ptr(), qd.stride(0), out.data_ptr(),
                  out.stride(0), ptrs[0].data_ptr(), ptrs[1].data_ptr(), hs * bs, float(scale),
                  tab.data_ptr(), per, lens.data_ptr(), max(ctxs), None if sl is None else sl.data_ptr(),
                  ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        outs.append(out.clone())
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    got = out.cpu().numpy()
    assert pad == 0 or (got[:, row:] == 7.0).all()
    err = np.abs(got[:, :row].reshape(ref.shape).astype(np.float64) - ref)
    vmax = 6.0  # of the N(0, 1) values
    assert np.all(err <= 2.0 ** -11 * np.abs(ref) + 2.0 ** -17 * vmax), float(err.max())


def test_infinite_value_stays_infinite(hip_device):
    """An infinite cached value (an overflowed projection) makes its dim
    infinite in every head whose softmax gives the token any weight, however
    small, and leaves the other dims as they are."""
    say("attention with infinite values")
    heads, kvh, hs, bs, ctx = 8, 2, 128, 16, 300
    rng = np.random.default_rng(5)
    per = (ctx + bs - 1) // bs
    tables = np.arange(per, dtype=np.int32).reshape(1, per)
    kc = rng.standard_normal((per, kvh, hs // 8, bs, 8)).astype(np.float16)
    vc = rng.standard_normal((per, kvh, hs, bs)).astype(np.float16)
    vc[17 // bs, 0, 3, 17 % bs] = np.inf
    vc[299 // bs, 1, 90, 299 % bs] = -np.inf
    q = rng.standard_normal((1, heads, hs)).astype(np.float16)
    q[0, 1] *= 3   # logits to about +-35, weights down to e^-60
    q[0, 6] *= 2
    ref = A.paged_attention(q, kc, vc, tables, np.array([ctx]), 0.3, None)
    kd, vd = torch.from_numpy(kc).to(hip_device), torch.from_numpy(vc).to(hip_device)
    ptrs = [torch.tensor([t[i].data_ptr() for i in range(per)], dtype=torch.int64, device=hip_device)
            for t in (kd, vd)]
    qd, out = torch.from_numpy(q).to(hip_device), torch.empty(1, heads, hs, dtype=torch.float16, device=hip_device)
    tab, lens = torch.from_numpy(tables).to(hip_device), torch.tensor([ctx], dtype=torch.int32, device=hip_device)
    nbytes = _lib.paged_attention_workspace_size(1, heads, kvh, hs, bs, ctx)
    ws = torch.empty(max(16, nbytes), dtype=torch.uint8, device=hip_device)
    _lib.call("dw4_paged_attention", 1, heads, kvh, hs, bs, qd.data_ptr(), heads * hs, out.data_ptr(), heads * hs,
              ptrs[0].data_ptr(), ptrs[1].data_ptr(), hs * bs, 0.3, tab.data_ptr(), per, lens.data_ptr(), ctx,
              None, ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
    got = out.cpu().numpy().astype(np.float64)
    inf = ~np.isfinite(ref)
    assert inf.sum() == 8 and (got[inf] == ref[inf]).all()
    # fp32 sums of 128 products to 35: logits off by 2^-16 at most, outputs by twice that of max|v|
    err = np.abs(got[~inf] - ref[~inf])
    assert np.all(err <= 2.0 ** -11 * np.abs(ref[~inf]) + 2.0 ** -15 * 6), float(err.max())


@pytest.mark.parametrize("heads,kvh,hs,bs", [(16, 2, 128, 16), (8, 2, 64, 32), (6, 2, 256, 16)])
def test_probabilities_keep_their_bits(hip_device, heads, kvh, hs, bs):
    """Two tokens, each with a one in a dim of its own: the partition's fp32
    sums are then the two probabilities themselves, 1 and p, and its sum of
    them is 1 + p rounded once, to the bit.  (Two fp16 parts of p, 21 bits
    cut downwards, miss the sum in one case of five.)"""
    say(f"probabilities heads={heads}/{kvh} hs={hs} bs={bs}")
    n, ctx_max = 30, 600
    rng = np.random.default_rng(hs)
    kc = np.zeros((n, kvh, hs // 8, bs, 8), np.float16)
    kc[:, :, :, 1, :] = rng.standard_normal((n, kvh, hs // 8, 8))
    vc = np.zeros((n, kvh, hs, bs), np.float16)
    vc[:, :, 0, 0] = vc[:, :, 1, 1] = 1
    q = rng.standard_normal((n, heads, hs)).astype(np.float16)
    tables = np.zeros((n, (ctx_max + bs - 1) // bs), np.int32)
    tables[:, 0] = np.arange(n)
    dev = lambda a: torch.from_numpy(a).to(hip_device)  # noqa: E731
    kd, vd, qd, tab = dev(kc), dev(vc), dev(q), dev(tables)
    ptrs = [torch.tensor([t[i].data_ptr() for i in range(n)], dtype=torch.int64, device=hip_device)
            for t in (kd, vd)]
    lens = torch.full((n,), 2, dtype=torch.int32, device=hip_device)
    out = torch.empty(n, heads, hs, dtype=torch.float16, device=hip_device)
    nbytes = _lib.paged_attention_workspace_size(n, heads, kvh, hs, bs, ctx_max)
    ws = torch.full((nbytes // 4,), float("nan"), device=hip_device)
    _lib.call("dw4_paged_attention", n, heads, kvh, hs, bs, qd.data_ptr(), heads * hs, out.data_ptr(), heads * hs,
              ptrs[0].data_ptr(), ptrs[1].data_ptr(), hs * bs, hs ** -0.5, tab.data_ptr(), tables.shape[1],
              lens.data_ptr(), ctx_max, None, ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
    # partial results: (max, sum) of every partition, then the outputs, of which
    # only the first partition (the others hold no token) writes any
    parts = (int((~torch.isnan(ws)).sum()) // (n * heads) - hs) // 2
    assert parts > 1
    rows = n * heads * parts
    ml = ws[:2 * rows].view(n, heads, parts, 2)[:, :, 0].cpu().numpy()
    o = ws[2 * rows:rows * (2 + hs)].view(n, heads, parts, hs)[:, :, 0, :2].cpu().numpy()
    assert (o.max(axis=2) == 1).all() and (o.min(axis=2) > 0).all()
    assert np.array_equal(o[..., 0] + o[..., 1], ml[..., 1])


@pytest.mark.parametrize("heads,kvh,hs,bs,most,calls", [
    (32, 8, 128, 32, (32, 3072), [(1, 2048), (9, 1025), (32, 128)]),
    (16, 4, 64, 16, (24, 4000), [(3, 600), (1, 2049), (1, 2048)]),
    (8, 2, 256, 16, (5, 9000), [(4, 9000), (5, 2048), (1, 4097)])])
def test_one_workspace_serves_smaller_calls(hip_device, heads, kvh, hs, bs, most, calls):
    """A workspace of the size for the most sequences and the longest context
    (which run as one workgroup per pair, without one) takes every call of
    fewer or shorter ones."""
    ws = torch.empty(max(16, _lib.paged_attention_workspace_size(most[0], heads, kvh, hs, bs, most[1])),
                     dtype=torch.uint8, device=hip_device)
    rng = np.random.default_rng(hs)
    for n, ctx in calls:
        say(f"attention {n} x {ctx} in the workspace of {most}")
        per = (ctx + bs - 1) // bs
        tables = rng.permutation(n * per).astype(np.int32).reshape(n, per)
        kc = rng.standard_normal((n * per, kvh, hs // 8, bs, 8)).astype(np.float16)
        vc = rng.standard_normal((n * per, kvh, hs, bs)).astype(np.float16)
        q = rng.standard_normal((n, heads, hs)).astype(np.float16)
        ctxs = rng.integers(1, ctx + 1, n)
        ctxs[0] = ctx
        ref = A.paged_attention(q, kc, vc, tables, ctxs, hs ** -0.5, None)
        kd, vd, qd, tab = (torch.from_numpy(a).to(hip_device) for a in (kc, vc, q, tables))
        ptrs = [torch.tensor([t[i].data_ptr() for i in range(n * per)], dtype=torch.int64, device=hip_device)
                for t in (kd, vd)]
        lens = torch.from_numpy(ctxs.astype(np.int32)).to(hip_device)
        out = torch.empty(n, heads, hs, dtype=torch.float16, device=hip_device)
        _lib.call("dw4_paged_attention", n, heads, kvh, hs, bs, qd.data_ptr(), heads * hs, out.data_ptr(),
                  heads * hs, ptrs[0].data_ptr(), ptrs[1].data_ptr(), hs * bs, hs ** -0.5, tab.data_ptr(), per,
                  lens.data_ptr(), ctx, None, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
        err = np.abs(out.cpu().numpy().astype(np.float64) - ref)
        assert np.all(err <= 2.0 ** -11 * np.abs(ref) + 2.0 ** -17 * 6), float(err.max())
