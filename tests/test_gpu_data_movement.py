"""GPU parity of the tiled data-movement kernels at the edges of their tiles:
cache writes and restores (runs that start inside an 8-token cell, several
runs in one tile, scattered slots, padding, head sizes with a partial and a
second slab, rows and blocks that are not 16-byte aligned) and the dequantiser
(partial strip groups, strided and unaligned outputs, act-order).  Everything
here is bit-exact.  Every case prints its name before touching the GPU.
"""
from __future__ import annotations

import sys

import numpy as np
import pytest
import torch

from gptq_synth import make_layer
from hip_extends import _lib
from hip_extends.w4a16 import CacheV2, Q4MatrixV2, TuningParams
from oracle import attention as A
from oracle import gptq

pytestmark = pytest.mark.gpu


def say(msg: str) -> None:
    print(f"[case] {msg}", flush=True)
    sys.stdout.flush()


def _runs(bs, start, counts):
    """Slots of runs of consecutive tokens, each run in blocks of its own."""
    out, blk = [], 0
    for i, c in enumerate(counts):
        s0 = blk * bs + (start if i == 0 else (3 * i) % 8)
        out += list(range(s0, s0 + c))
        blk = (s0 + c) // bs + 1
    return np.array(out, np.int64)


SLOTS = {
    "run from a cell": lambda bs: _runs(bs, 0, [70]),
    "run inside a cell": lambda bs: _runs(bs, 5, [67]),
    "several runs": lambda bs: _runs(bs, 2, [9, 31, 8, 1, 17]),
    "one token": lambda bs: np.array([bs + 3], np.int64),
    "padding": lambda bs: np.where(np.arange(40) % 9 == 4, -1, np.arange(40)).astype(np.int64),
    "padding first": lambda bs: np.concatenate([[-1, -1], np.arange(8, 30)]).astype(np.int64),
    "scattered": lambda bs: np.random.default_rng(bs).permutation(6 * bs)[:45].astype(np.int64),
}


@pytest.mark.parametrize("slots", SLOTS, ids=lambda s: s.replace(" ", "-"))
@pytest.mark.parametrize("bs,kvh,hs,row_pad,block_pad", [
    # narrow rows of few tokens, and rows 2-byte aligned: the element-wise kernel
    (16, 4, 128, 0, 0), (32, 3, 64, 8, 0), (32, 2, 256, 0, 0), (16, 2, 40, 0, 0),
    (16, 2, 128, 3, 0), (32, 2, 128, 0, 1), (16, 32, 128, 3, 0),
    # the tiles
    (16, 32, 128, 0, 0), (32, 64, 64, 8, 0), (32, 16, 256, 0, 0), (16, 104, 40, 0, 0),
    (32, 32, 128, 0, 1),  # blocks 2-byte aligned: no 16-byte units on the cache side
])
def test_cache_tile_edges(hip_device, slots, bs, kvh, hs, row_pad, block_pad):
    say(f"cache tile {slots} bs={bs} heads={kvh} hs={hs} pads={row_pad},{block_pad}")
    sl = SLOTS[slots](bs)
    n, blocks, per = len(sl), int(sl.max()) // bs + 1, kvh * hs * bs
    rng = np.random.default_rng(n)
    key, val = (rng.standard_normal((n, kvh, hs)).astype(np.float16) for _ in range(2))
    kc, vc = A.empty_cache(blocks, kvh, hs, bs, fill=0.0)
    A.reshape_and_cache(key, val, kc, vc, sl)
    kbuf, vbuf = (torch.zeros(blocks * (per + block_pad), dtype=torch.float16, device=hip_device)
                  for _ in range(2))
    ptrs = [torch.tensor([b.data_ptr() + 2 * (i * (per + block_pad) + block_pad) for i in range(blocks)],
                         dtype=torch.int64, device=hip_device) for b in (kbuf, vbuf)]
    rows = [torch.zeros(n, kvh * hs + row_pad, dtype=torch.float16, device=hip_device) for _ in range(4)]
    for r, a in zip(rows, (key, val)):
        r[:, :kvh * hs] = torch.from_numpy(a.reshape(n, -1)).to(hip_device)
    sd = torch.from_numpy(sl).to(hip_device)
    stream = torch.cuda.current_stream().cuda_stream
    _lib.call("dw4_reshape_and_cache", n, kvh, hs, bs, rows[0].data_ptr(), rows[0].stride(0),
              rows[1].data_ptr(), rows[1].stride(0), ptrs[0].data_ptr(), ptrs[1].data_ptr(), hs * bs,
              sd.data_ptr(), stream)
    _lib.call("dw4_restore_from_cache", n, kvh, hs, bs, rows[2].data_ptr(), rows[2].stride(0),
              rows[3].data_ptr(), rows[3].stride(0), ptrs[0].data_ptr(), ptrs[1].data_ptr(), hs * bs,
              sd.data_ptr(), stream)
    torch.cuda.synchronize()
    for buf, ref in ((kbuf, kc), (vbuf, vc)):
        got = buf.cpu().numpy().reshape(blocks, per + block_pad)[:, block_pad:]
        assert np.array_equal(got.view(np.uint16), ref.reshape(blocks, per).view(np.uint16))
    for r, a in zip(rows[2:], (key, val)):
        want = np.where((sl >= 0)[:, None], a.reshape(n, -1), np.float16(0))
        got = r.cpu().numpy()
        assert np.array_equal(got[:, :kvh * hs].view(np.uint16), want.view(np.uint16))
        assert not got[:, kvh * hs:].any()  # the padding between rows is not written


@pytest.mark.parametrize("k,n,g,act,pad", [
    (128, 16, 128, False, 0), (384, 144, 32, False, 0), (256, 400, 64, True, 8),
    (512, 272, 128, False, 3), (640, 128, 640, True, 1)])
@pytest.mark.parametrize("bf16", [False, True], ids=["fp16", "bf16"])
def test_dequant_tile_edges(hip_device, k, n, g, act, pad, bf16):
    say(f"dequant {k}x{n} g={g} act={act} pad={pad} bf16={bf16}")
    lay = make_layer(k, n, g, seed=n + k, act_order=act)
    a = lay.numpy()
    ref = (gptq.dequantize_bf16 if bf16 else gptq.dequantize)(
        a["qweight"], a["qzeros"], a["scales"], a["g_idx"]).view(np.uint16)
    cache = CacheV2(hip_device)
    d = lay.to(hip_device)
    q4 = Q4MatrixV2(d.qweight, d.qzeros, d.scales, k, n, d.g_idx if act else None, act, TuningParams(),
                    cache)
    w = torch.full((k, n + pad), -1, dtype=torch.int16, device=hip_device)
    _lib.call("dw4_dequant_bf16" if bf16 else "dw4_dequant", k, n, g, q4.qweight.data_ptr(),
              q4.qzeros.data_ptr(), q4.scales.data_ptr(), q4.perm.data_ptr() if q4.use_act else None,
              w.data_ptr(), w.stride(0), torch.cuda.current_stream().cuda_stream)
    got = w.cpu().numpy().view(np.uint16)
    assert np.array_equal(got[:, :n], ref)
    assert (got[:, n:] == 0xFFFF).all()  # the padding between rows is not written


@pytest.mark.parametrize("n,kvh,hs,bs", [(383, 8, 128, 16), (384, 8, 128, 16), (448, 8, 64, 32), (500, 2, 80, 32),
                                         (761, 32, 64, 16), (762, 32, 64, 16)])
def test_cache_rules(hip_device, n, kvh, hs, bs):
    """Both sides of the lines between the element-wise copy and the tiles
    (narrow rows of few tokens) and between their 512 and 256 threads (up to
    768 workgroups), in runs that begin inside a cell."""
    say(f"cache {n} x {kvh} x {hs} bs={bs}")
    sl = _runs(bs, 3, [n // 3, n // 2, n - n // 3 - n // 2])
    blocks, per = int(sl.max()) // bs + 1, kvh * hs * bs
    rng = np.random.default_rng(n)
    key, val = (rng.standard_normal((n, kvh, hs)).astype(np.float16) for _ in range(2))
    kc, vc = A.empty_cache(blocks, kvh, hs, bs, fill=0.0)
    A.reshape_and_cache(key, val, kc, vc, sl)
    bufs = [torch.zeros(blocks * per, dtype=torch.float16, device=hip_device) for _ in range(2)]
    ptrs = [torch.arange(blocks, dtype=torch.int64, device=hip_device) * (2 * per) + b.data_ptr() for b in bufs]
    rows = [torch.from_numpy(a.reshape(n, -1)).to(hip_device) for a in (key, val)]
    back = [torch.zeros_like(r) for r in rows]
    sd, stream = torch.from_numpy(sl).to(hip_device), torch.cuda.current_stream().cuda_stream
    for name, r in (("dw4_reshape_and_cache", rows), ("dw4_restore_from_cache", back)):
        _lib.call(name, n, kvh, hs, bs, r[0].data_ptr(), r[0].stride(0), r[1].data_ptr(), r[1].stride(0),
                  ptrs[0].data_ptr(), ptrs[1].data_ptr(), hs * bs, sd.data_ptr(), stream)
    for buf, ref in zip(bufs, (kc, vc)):
        assert np.array_equal(buf.cpu().numpy().view(np.uint16), ref.reshape(-1).view(np.uint16))
    assert all(torch.equal(a, b) for a, b in zip(rows, back))
