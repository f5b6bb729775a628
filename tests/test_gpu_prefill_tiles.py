"""GPU parity of the prefill kernels' tiles at their edges: every tile of the
K-sliced and the LDS-streamed kernel (a case names its plan on 256 CUs, and
the test asserts it) with partial row and column tiles, fewer chunks than
waves, K splits, every group size form, act-order with and without room for the
gathered rows, fp16 and bf16 activations, strided and unaligned rows, and the
grouped launch.

Bar, elementwise against the float64 product of x and s * (q - z): with u the
unit roundoff of the output type (2^-11 fp16, 2^-8 bf16; half-ulp rounding is
at most u/2 relative, bf16 weights are rounded to bf16, fp16 ones to fp16),
  |y - ref| <= u/2 |x|.|W| + 2^-23 sqrt(K) |x|.|W| + u |ref| + u |bias|,
the weight roundings, the fp32 sums (K terms, random signs) and the output
roundings (product, then bias).
"""
from __future__ import annotations

import sys

import numpy as np
import pytest
import torch

from gptq_synth import make_layer
from hip_extends import _lib
from hip_extends.w4a16 import CacheV2, Q4MatrixV2, TuningParams, gemm_group
from oracle import gptq

pytestmark = pytest.mark.gpu


def say(msg: str) -> None:
    print(f"[case] {msg}", flush=True)
    sys.stdout.flush()


def _build(k, n, g, act, dev, m, seed=0):
    lay = make_layer(k, n, g, seed=k + n + g + seed, act_order=act)
    d = lay.to(dev)
    cache = CacheV2(dev)
    q4 = Q4MatrixV2(d.qweight, d.qzeros, d.scales, k, n, d.g_idx if act else None, act,
                    TuningParams(MAX_M=m), cache)
    cache.init_cache()
    a = lay.numpy()
    q = gptq.unpack_qweight(a["qweight"]).astype(np.float64)
    z = gptq.unpack_qzeros(a["qzeros"]).astype(np.float64)
    gi = a["g_idx"].astype(np.int64)
    w = a["scales"].astype(np.float64)[gi] * (q - (z + 1.0)[gi])
    return q4, w


def _x(m, k, dtype, seed):
    return torch.randn(m, k, generator=torch.Generator().manual_seed(seed)).to(dtype)


def _check(y, x, w, bias, what):
    u = 2.0 ** -11 if y.dtype == torch.float16 else 2.0 ** -8
    xd = x.double().numpy()
    ref, mag = xd @ w, np.abs(xd) @ np.abs(w)
    b = np.zeros(w.shape[1]) if bias is None else bias.double().numpy()
    bound = (u / 2 + 2.0 ** -23 * w.shape[0] ** 0.5) * mag + u * np.abs(ref) + u * np.abs(b)
    err = np.abs(y.double().cpu().numpy() - ref - b)
    assert np.all(np.isfinite(err)) and np.all(err <= bound), \
        f"{what}: worst error / bound {np.nanmax(err / bound):.3f}"


# the plan on 256 CUs: K-sliced or LDS-streamed, tile, K splits
CASES = [
    # m, k, n, group, act, plan
    (33, 256, 80, 128, False, "K 64x32/1"),      # two chunks for eight waves
    (64, 640, 400, 32, False, "K 64x32/1"),      # 25 strips (the last column tile half full)
    (97, 5120, 1040, 128, False, "K 64x32/3"),
    (65, 640, 4112, 64, False, "K 32x64/1"),     # five chunks
    (65, 4096, 1040, 4096, False, "K 64x32/2"),  # one group
    (33, 1024, 8208, 32, False, "K 64x64/1"),
    (97, 1024, 4112, 256, True, "K 64x64/1"),
    (130, 5120, 1040, 256, True, "K 64x32/2"),
    (97, 256, 4112, 128, False, "L 32x128/1"),
    (130, 384, 8208, 64, False, "L 64x128/1"),
    (97, 4096, 8208, 128, False, "L 64x256/3"),
    (300, 256, 8208, 32, True, "L 32x128/1"),
    (700, 1024, 8208, 128, False, "L 128x256/1"),
    (600, 256, 8208, 128, False, "L 96x256/1"),
    (385, 512, 8208, 64, False, "L 64x256/1"),   # one row in the last tile
    (1300, 384, 4112, 32, False, "L 96x256/1"),
    (500, 7552, 8192, 128, False, "L 128x128/1"),
    (520, 13824, 2064, 64, True, "L 96x256/4"),
]


@pytest.mark.parametrize("m,k,n,g,act,plan", CASES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
def test_prefill_tiles(hip_device, m, k, n, g, act, plan, dtype):
    q4, w = _build(k, n, g, act, hip_device, m)
    x = _x(m, k, dtype, m)
    xd = x.to(hip_device)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(1)) * 0.5).to(dtype)
    perm = q4.perm.data_ptr() if q4.use_act else None
    room = _lib.workspace_size(m, k, n, g, act)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    # dense rows and a full workspace; strided x and unaligned y; splits 1, 3
    for pad_x, pad_y, split in ((0, 0, 0), (8, 3, 1), (0, 8, 3)):
        if dtype == torch.bfloat16 and split == 3:
            continue  # no split argument
        say(f"prefill tiles {k}x{n} g={g} act={act} M={m} {dtype} pads={pad_x},{pad_y} split={split}")
        xs = torch.zeros(m, k + pad_x, dtype=dtype, device=hip_device)
        xs[:, :k] = xd
        y = torch.full((m, n + pad_y), float("nan"), dtype=dtype, device=hip_device)
        planes = 16384 + 4 * m * n * 4 + 512 + 2 * m * k
        ws = torch.zeros(max(16, room, planes if split else 0), dtype=torch.uint8, device=hip_device)
        if split == 0:
            p = _lib.prefill_plan(m, k, n, g, act, ws.numel())
            assert f"{'RLK'[p.kernel]} {p.tile_rows}x{p.tile_cols}/{p.splits}" == plan
        args = (m, k, n, g, xs.data_ptr(), xs.stride(0), q4.qweight.data_ptr(), q4.qzeros.data_ptr(),
                q4.scales.data_ptr(), perm, bias.to(hip_device).data_ptr(), y.data_ptr(), y.stride(0),
                ws.data_ptr(), ws.numel(), stream)
        if dtype == torch.float16:
            st = lib.dw4_gemm_path(_lib.DW4_PATH_PREFILL, split, *args)
        else:
            st = lib.dw4_gemm_bf16_prefill(*args)
        assert st == _lib.DW4_OK, _lib.strerror(st)
        torch.cuda.synchronize()
        _check(y[:, :n], x, w, bias, f"M={m} split={split}")
        assert bool(torch.isnan(y[:, n:]).all())  # nothing outside the columns
        assert not ws[:16384].any() or room == 0 and not split  # the counter head stays zero


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
def test_act_order_without_room(hip_device, dtype):
    """fp16: the kernels that gather per workgroup; bf16: refused before any
    launch, and matmul takes the dense route."""
    m, k, n = 100, 512, 400
    q4, w = _build(k, n, 64, True, hip_device, m)
    x = _x(m, k, dtype, 3)
    xd = x.to(hip_device)
    y = torch.full((m, n), 7.0, dtype=dtype, device=hip_device)
    args = (m, k, n, 64, xd.data_ptr(), k, q4.qweight.data_ptr(), q4.qzeros.data_ptr(),
            q4.scales.data_ptr(), q4.perm.data_ptr(), None, y.data_ptr(), n, None, 0,
            torch.cuda.current_stream().cuda_stream)
    say(f"act-order without room {dtype}")
    if dtype == torch.float16:
        assert _lib.load().dw4_gemm(*args) == _lib.DW4_OK
    else:
        assert _lib.load().dw4_gemm_bf16_prefill(*args) == _lib.DW4_ERR_WORKSPACE
        torch.cuda.synchronize()
        assert bool((y == 7.0).all())
        q4.cache._workspace = torch.zeros(16, dtype=torch.uint8, device=hip_device)
        q4.matmul(xd, output=y)
    torch.cuda.synchronize()
    _check(y, x, w, None, "no room")


@pytest.mark.parametrize("m,k,n,count,g", [
    (40, 1024, 4112, 3, 128), (100, 4096, 2064, 2, 64), (300, 512, 4112, 3, 32), (700, 256, 4096, 2, 128)])
def test_grouped_prefill(hip_device, m, k, n, count, g):
    """Matrices sharing x, in one launch or one after another by the model."""
    say(f"grouped prefill {count} x {k}x{n} g={g} M={m}")
    mats = [_build(k, n, g, False, hip_device, m, seed=i) for i in range(count)]
    x = _x(m, k, torch.float16, 9)
    ys = gemm_group(x.to(hip_device), [q4 for q4, _ in mats])
    torch.cuda.synchronize()
    for (_, w), y in zip(mats, ys):
        _check(y, x, w, None, "grouped")


def test_wide_row_stride_keeps_the_64_bit_kernel(hip_device):
    """Rows of x more than 2^22 elements apart: the register-fed kernel."""
    m, k, n = 40, 256, 400
    q4, w = _build(k, n, 128, False, hip_device, m)
    x = _x(m, k, torch.float16, 4)
    say("wide row stride")
    store = torch.empty((m - 1) * ((1 << 22) + 8) + k, dtype=torch.float16, device=hip_device)
    xs = store.as_strided((m, k), ((1 << 22) + 8, 1))
    xs.copy_(x.to(hip_device))
    y = q4.matmul(xs, path=_lib.DW4_PATH_PREFILL)
    torch.cuda.synchronize()
    _check(y, x, w, None, "wide stride")


def test_bf16_rows_keep_dense_semantics(hip_device):
    # above the decode rows: a given weight buffer is filled, and a recorded
    # input gets its gradient (dy W^T; bf16 operands, so 2^-8 of each product)
    lay = make_layer(512, 256, 128, seed=91).to(hip_device)
    cache = CacheV2(hip_device)
    q4 = Q4MatrixV2(lay.qweight, lay.qzeros, lay.scales, 512, 256, None, False, TuningParams(MAX_M=256), cache)
    cache.init_cache()
    w = q4.get_bfloat16_weights_matrix_v2().float()
    x = torch.randn(100, 512, device=hip_device).to(torch.bfloat16)
    buf = torch.zeros(512 * 256, dtype=torch.float16, device=hip_device)
    say("bf16 100 rows with a weight buffer, then recorded")
    q4.matmul(x, temp_weight=buf)
    assert torch.equal(buf.view(torch.bfloat16).view(512, 256).float(), w)
    tracked = x.clone().requires_grad_(True)
    dx, = torch.autograd.grad(q4.matmul(tracked).float().sum(), tracked)
    ref = w.sum(dim=1).expand(100, 512)
    assert ((dx.float() - ref).abs() <= 2.0 ** -8 * w.abs().sum(dim=1)).all()


@pytest.mark.parametrize("m,k,n,g,act", [(100, 512, 400, 128, True), (300, 384, 4112, 64, False),
                                         (700, 512, 1040, 32, False)])
def test_bf16_prefill_takes_the_dequantised_weight(hip_device, m, k, n, g, act):
    """The packed bf16 product is over the very weight of the dense route,
    bf16(fp16(s (q - z))): against its float64 product only half an ulp of
    the output and the fp32 sums are left (K terms of random sign, rounded at
    2^-24 of a partial sum each; twice that).  A weight rounded once, an ulp
    off in one value of thirty, moves one output in fifteen past this."""
    q4, _ = _build(k, n, g, act, hip_device, m)
    w = q4.get_bfloat16_weights_matrix_v2().double().cpu().numpy()
    x = _x(m, k, torch.bfloat16, m + 1)
    say(f"bf16 prefill over the dequantised weight {k}x{n} g={g} act={act} M={m}")
    y = q4.matmul(x.to(hip_device)).double().cpu().numpy()
    xd = x.double().numpy()
    ref = xd @ w
    half_ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ref), np.abs(y)))) - 8)
    sums = 2.0 ** -23 * k ** 0.5 * np.sqrt((xd ** 2) @ (w ** 2))
    bad = np.abs(y - ref) > half_ulp + sums
    assert not bad.any(), f"{bad.mean():.4f} of the outputs"


@pytest.mark.parametrize("scale", [float("inf"), 30000.0])
def test_bf16_prefill_overflowing_scales(hip_device, scale):
    """An infinite scale, and one whose weights overflow fp16: infinities and
    NaN where the dense product over the dequantised weight has them."""
    lay = make_layer(256, 80, 128, seed=93, symmetric=True)
    scales = lay.scales.clone()
    scales[1, 5] = scale
    qweight = lay.qweight | -0x66666667  # 0x99999999: codes above the zero of 8, weights > 0
    cache = CacheV2(hip_device)
    q4 = Q4MatrixV2(*(t.to(hip_device) for t in (qweight, lay.qzeros, scales)), 256, 80, None, False,
                    TuningParams(MAX_M=128), cache)
    cache.init_cache()
    say(f"bf16 prefill with a scale of {scale}")
    x = _x(100, 256, torch.bfloat16, 5).to(hip_device)
    x[::2] = x[::2].abs()  # infinite in every other row, inf - inf in the rest
    y, ref = q4.matmul(x).float(), q4.matmul(x, must_blas=True).float()
    assert torch.isposinf(ref[::2, 5]).all() and torch.isnan(ref[1::2, 5]).all()
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    assert torch.equal(torch.isposinf(y), torch.isposinf(ref))
