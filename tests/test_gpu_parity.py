"""GPU parity of the HIP W4A16 path against the pinned CPU oracle.

Bars: dequantised fp16 weights bit-exact; GEMM outputs within
max|y - y_ref| <= 2e-2 * ||y_ref row||_inf of a wide-accumulated reference.
Every case prints its name before touching the GPU.
"""
from __future__ import annotations

import ctypes
import functools
import sys

import numpy as np
import pytest
import torch

from gptq_synth import make_layer, make_x
from hip_extends import _lib
from hip_extends.w4a16 import CacheV2, Q4MatrixV2, TuningParams, gemm_group
from oracle import gptq

pytestmark = pytest.mark.gpu

TOL = 2e-2  # max-abs error <= 2e-2 * ||row||_inf


def say(msg: str) -> None:
    print(f"[case] {msg}", flush=True)
    sys.stdout.flush()


def build(layer, dev, max_m=4096):
    lay = layer.to(dev)
    cache = CacheV2(dev)
    q4 = Q4MatrixV2(lay.qweight, lay.qzeros, lay.scales, lay.in_features, lay.out_features,
                    lay.g_idx if lay.act_order else None, lay.act_order,
                    TuningParams(MAX_M=max_m), cache)
    cache.init_cache()
    return q4


@functools.lru_cache(maxsize=8)
def oracle_w(k, n, g, seed, sym, act):
    lay = make_layer(k, n, g, seed=seed, symmetric=sym, act_order=act)
    a = lay.numpy()
    return lay, gptq.dequantize(a["qweight"], a["qzeros"], a["scales"], a["g_idx"])


def check_tol(y_gpu: torch.Tensor, y_ref: np.ndarray, what: str) -> float:
    y = y_gpu.float().cpu().numpy()
    assert np.all(np.isfinite(y)), what
    ok, worst = gptq.within_tolerance(y, y_ref, TOL)
    assert ok, f"{what}: worst error ratio {worst:.4f} > 1"
    return worst


# ---------------------------------------------------------------------------
# bit-exact dequantisation
# ---------------------------------------------------------------------------
def test_golden_dequant_bit_exact(hip_device):
    data = np.load("tests/golden/gptq_small.npz")
    names = sorted({k.split("/")[0] for k in data.files})
    for name in names:
        say(f"golden dequant {name}")
        k, n, g, sym, act, m = data[f"{name}/meta"].tolist()
        cache = CacheV2(hip_device)
        q4 = Q4MatrixV2(torch.from_numpy(data[f"{name}/qweight"]).to(hip_device),
                        torch.from_numpy(data[f"{name}/qzeros"]).to(hip_device),
                        torch.from_numpy(data[f"{name}/scales"]).to(hip_device), k, n,
                        torch.from_numpy(data[f"{name}/g_idx"]).to(hip_device) if act else None,
                        bool(act), TuningParams(), cache)
        cache.init_cache()
        w = q4.get_float16_weights_matrix_v2().cpu().numpy().view(np.uint16)
        assert np.array_equal(w, data[f"{name}/w"]), name


def test_dequant_exhaustive_kat(hip_device):
    """All 16 q x 16 stored zeros x 65,536 fp16 scale patterns, bit for bit."""
    say("exhaustive dequant KAT K=512 N=65536 g=32")
    K, N, G = 512, 65536, 16
    q = np.zeros((K, N), dtype=np.uint8)
    for z in range(16):
        for qq in range(16):
            q[z * 32 + 2 * qq: z * 32 + 2 * qq + 2, :] = qq
    zeros = np.repeat(np.arange(16, dtype=np.uint8)[:, None], N, axis=1)
    srow = np.arange(65536, dtype=np.uint32).astype(np.uint16)
    scales = np.repeat(srow[None, :], G, axis=0).view(np.float16)
    qweight, qzeros = gptq.pack_qweight(q), gptq.pack_qzeros(zeros)
    g_idx = (np.arange(K) // 32).astype(np.int32)
    with np.errstate(all="ignore"):
        ref = gptq.dequantize(qweight, qzeros, scales, g_idx)
    cache = CacheV2(hip_device)
    q4 = Q4MatrixV2(torch.from_numpy(qweight).to(hip_device), torch.from_numpy(qzeros).to(hip_device),
                    torch.from_numpy(scales).to(hip_device), K, N, None, False, TuningParams(), cache)
    w = q4.get_float16_weights_matrix_v2().cpu().numpy()
    same = (w.view(np.uint16) == ref.view(np.uint16)) | (np.isnan(w) & np.isnan(ref))
    assert same.all(), np.argwhere(~same)[:5]


# ---------------------------------------------------------------------------
# GEMM parity
# ---------------------------------------------------------------------------
def test_golden_gemm(hip_device):
    data = np.load("tests/golden/gptq_small.npz")
    names = sorted({k.split("/")[0] for k in data.files})
    for name in names:
        k, n, g, sym, act, m = data[f"{name}/meta"].tolist()
        cache = CacheV2(hip_device)
        q4 = Q4MatrixV2(torch.from_numpy(data[f"{name}/qweight"]).to(hip_device),
                        torch.from_numpy(data[f"{name}/qzeros"]).to(hip_device),
                        torch.from_numpy(data[f"{name}/scales"]).to(hip_device), k, n,
                        torch.from_numpy(data[f"{name}/g_idx"]).to(hip_device) if act else None,
                        bool(act), TuningParams(), cache)
        cache.init_cache()
        x = torch.from_numpy(data[f"{name}/x"]).to(hip_device)
        bias = data[f"{name}/bias"] if f"{name}/bias" in data.files else None
        bt = torch.from_numpy(bias).to(hip_device) if bias is not None else None
        # reference value (wide accumulation) for the tolerance check
        w = data[f"{name}/w"].view(np.float16)
        y_ref = gptq.gemm_ref(data[f"{name}/x"], w)
        if bias is not None:
            y_ref = y_ref + bias.astype(np.float64)[None, :]
        paths = [_lib.DW4_PATH_AUTO, _lib.DW4_PATH_PREFILL]
        if m <= 64:
            paths.append(_lib.DW4_PATH_DECODE)
        for path in paths:
            say(f"golden gemm {name} path={path}")
            y = q4.matmul(x, bias=bt, path=path)
            torch.cuda.synchronize()
            check_tol(y, y_ref, f"{name} path {path}")
            fix = data[f"{name}/y"].view(np.float16).astype(np.float64)
            assert np.max(np.abs(y.float().cpu().numpy() - fix)) <= \
                np.max(np.abs(fix)) * 4e-3 + 1e-3, name


SHAPES_7B = [(4096, 4096), (4096, 11008), (11008, 4096)]


@pytest.mark.parametrize("kn", SHAPES_7B, ids=lambda kn: f"{kn[0]}x{kn[1]}")
def test_decode_7b_shapes(hip_device, kn):
    k, n = kn
    lay, w = oracle_w(k, n, 128, 1000 + SHAPES_7B.index(kn), False, False)
    q4 = build(lay, hip_device)
    for m in (1, 2, 4, 8, 16, 20, 32, 33, 48, 64):
        say(f"decode 7B {k}x{n} M={m}")
        x = make_x(m, k, seed=m)
        y = q4.matmul(x.to(hip_device), path=_lib.DW4_PATH_DECODE)
        torch.cuda.synchronize()
        check_tol(y, gptq.gemm_ref(x.numpy(), w), f"decode {k}x{n} M={m}")


@pytest.mark.parametrize("k,n,m,g", [(11008, 4096, 16, 128), (11008, 4096, 40, 128),
                                     (4096, 4096, 64, 128), (4096, 11008, 24, 128),
                                     (2048, 8208, 16, 64), (8192, 2064, 24, 32),
                                     (8192, 2064, 33, 128)],
                         ids=["11008x4096_M16", "11008x4096_M40", "4096x4096_M64",
                              "4096x11008_M24", "2048x8208_M16_g64", "8192x2064_M24_g32",
                              "8192x2064_M33"])
def test_decode_wide_and_split_plans(hip_device, k, n, m, g):
    """The register-fed decode kernel with four strips per workgroup and K
    split over workgroups (fp32 planes summed in split order), with a
    partial last strip group (N / 16 not a multiple of 4) and groups of 32 /
    64: within tolerance of the oracle, deterministic, and -- given no
    workspace -- the unsplit plan, also within tolerance."""
    lay, w = oracle_w(k, n, g, 7000 + m, False, False)
    q4 = build(lay, hip_device)
    lib = _lib.load()
    x = make_x(m, k, seed=m + 31)
    xd = x.to(hip_device)
    ref = gptq.gemm_ref(x.numpy(), w)
    outs = []
    for size in (_lib.workspace_size(m, k, n, g, False),) * 2 + (0,):
        say(f"decode wide/split {k}x{n} M={m} g={g} workspace={size}")
        ws = torch.zeros(max(16, size), dtype=torch.uint8, device=hip_device)
        y = torch.empty(m, n, dtype=torch.float16, device=hip_device)
        st = lib.dw4_gemm_path(_lib.DW4_PATH_DECODE, 0, m, k, n, g, xd.data_ptr(), k,
                               q4.qweight.data_ptr(), q4.qzeros.data_ptr(), q4.scales.data_ptr(),
                               None, None, y.data_ptr(), n, ws.data_ptr(), size,
                               torch.cuda.current_stream().cuda_stream)
        assert st == _lib.DW4_OK, _lib.strerror(st)
        torch.cuda.synchronize()
        assert not ws[:4096 * 4].any()
        check_tol(y, ref, f"decode {k}x{n} M={m} g={g} workspace {size}")
        outs.append(y.cpu())
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


@pytest.mark.parametrize("kn", SHAPES_7B, ids=lambda kn: f"{kn[0]}x{kn[1]}")
def test_prefill_7b_shapes(hip_device, kn):
    k, n = kn
    lay, w = oracle_w(k, n, 128, 1000 + SHAPES_7B.index(kn), False, False)
    q4 = build(lay, hip_device)
    for m in (16, 64, 100, 256):
        say(f"prefill 7B {k}x{n} M={m}")
        x = make_x(m, k, seed=m + 7)
        y = q4.matmul(x.to(hip_device), path=_lib.DW4_PATH_PREFILL)
        torch.cuda.synchronize()
        check_tol(y, gptq.gemm_ref(x.numpy(), w), f"prefill {k}x{n} M={m}")


def test_symmetric_c1(hip_device):
    lay, w = oracle_w(4096, 4096, 128, 0, True, False)
    q4 = build(lay, hip_device)
    say("symmetric (all zeros 8) 4096x4096 M=1")
    x = make_x(1, 4096, seed=0)
    y = q4.matmul(x.to(hip_device))
    torch.cuda.synchronize()
    check_tol(y, gptq.gemm_ref(x.numpy(), w), "symmetric")


@pytest.mark.parametrize("kn", [(5120, 5120), (13824, 5120), (5120, 13824)],
                         ids=lambda kn: f"{kn[0]}x{kn[1]}")
def test_act_order_13b(hip_device, kn):
    k, n = kn
    lay, w = oracle_w(k, n, 128, 2000 + k + n, False, True)
    q4 = build(lay, hip_device)
    assert q4.use_act
    for m in (1, 8, 24, 64):
        for path in (_lib.DW4_PATH_DECODE, _lib.DW4_PATH_PREFILL):
            say(f"act-order 13B {k}x{n} M={m} path={path}")
            x = make_x(m, k, seed=m + 11)
            y = q4.matmul(x.to(hip_device), path=path)
            torch.cuda.synchronize()
            check_tol(y, gptq.gemm_ref(x.numpy(), w), f"act {k}x{n} M={m} path {path}")


@pytest.mark.parametrize("kn", [(5120, 5120), (13824, 5120), (5120, 13824), (16384, 1024),
                                (16512, 1024)],
                         ids=lambda kn: f"{kn[0]}x{kn[1]}")
def test_act_order_m1_lds_gather(hip_device, kn):
    """Act-order at M=1: the staged decode kernel copies x into LDS and
    gathers its units from there by perm (K <= 16384; 16512 takes the gather
    launch instead).  The same plan through dw4_gemm_group (one item) gathers
    per workgroup from global memory: the staged values and the sums are the
    same, so the outputs are bit-identical, and both are within the oracle's
    tolerance.  No workspace is needed for the LDS gather."""
    k, n = kn
    lay, w = oracle_w(k, n, 128, 3100 + k + n, False, True)
    q4 = build(lay, hip_device)
    lib = _lib.load()
    x = make_x(1, k, seed=k + n)
    xd = x.to(hip_device)
    ref = gptq.gemm_ref(x.numpy(), w)
    say(f"act-order M=1 LDS gather {k}x{n}")
    y = q4.matmul(xd, path=_lib.DW4_PATH_DECODE)
    torch.cuda.synchronize()
    check_tol(y, ref, f"act M=1 {k}x{n}")
    say(f"act-order M=1 {k}x{n}: no workspace")
    y0 = torch.empty(1, n, dtype=torch.float16, device=hip_device)
    st = lib.dw4_gemm_path(_lib.DW4_PATH_DECODE, 0, 1, k, n, 128, xd.data_ptr(), k,
                           q4.qweight.data_ptr(), q4.qzeros.data_ptr(), q4.scales.data_ptr(),
                           q4.perm.data_ptr(), None, y0.data_ptr(), n, None, 0,
                           torch.cuda.current_stream().cuda_stream)
    assert st == _lib.DW4_OK, _lib.strerror(st)
    say(f"act-order M=1 {k}x{n}: grouped launch, per-workgroup gather")
    (yg,) = gemm_group(xd, [q4])
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), yg.view(torch.int16)), f"{k}x{n}"
    assert torch.equal(y0.view(torch.int16), yg.view(torch.int16)), f"{k}x{n} no workspace"


def test_act_order_gather_first_matches_in_kernel_gather(hip_device):
    """Act-order calls gather x into the packed row order in the workspace
    when it has room, else the kernels gather per workgroup.  The second
    route gets room for the decode plan's split-K planes but none for the
    gathered rows, so both routes run the same plan.
    Where that is the same kernel (decode; prefill tiles below 256 columns)
    they feed the same values to the same sums and the outputs are
    bit-identical.
    At M=300 the gathered rows go to the K-sliced 64 x 64 tile kernel, whose
    waves each sum every eighth chunk and add up at the end; the per-workgroup
    gather stays on the sequential-k kernel, so there both are held to the
    oracle's tolerance instead."""
    k, n = 5120, 2048
    lay, w = oracle_w(k, n, 128, 4242, False, True)
    q4 = build(lay, hip_device)
    lib = _lib.load()
    for m, path in ((8, _lib.DW4_PATH_DECODE), (64, _lib.DW4_PATH_DECODE),
                    (64, _lib.DW4_PATH_PREFILL), (300, _lib.DW4_PATH_PREFILL)):
        say(f"act-order gather-first vs in-kernel gather M={m} path={path}")
        x = make_x(m, k, seed=m + 77)
        xd = x.to(hip_device)
        outs = []
        for with_ws in (True, False):
            # without act-order room: the decode plan's split planes only (the
            # prefill calls below are unsplit)
            size = _lib.workspace_size(m, k, n, 128, True) if with_ws else \
                (_lib.workspace_size(m, k, n, 128, False) if path == _lib.DW4_PATH_DECODE else 0)
            ws = torch.zeros(max(16, size), dtype=torch.uint8, device=hip_device)
            if with_ws:
                assert ws.numel() >= m * k * 2  # room for the gathered activations
            y = torch.empty(m, n, dtype=torch.float16, device=hip_device)
            st = lib.dw4_gemm_path(path, 1, m, k, n, 128, xd.data_ptr(), k,
                                   q4.qweight.data_ptr(), q4.qzeros.data_ptr(),
                                   q4.scales.data_ptr(), q4.perm.data_ptr(), None,
                                   y.data_ptr(), n, ws.data_ptr(),
                                   ws.numel(), torch.cuda.current_stream().cuda_stream)
            assert st == _lib.DW4_OK, _lib.strerror(st)
            torch.cuda.synchronize()
            if with_ws:  # the arrival-counter head stays zero for later split calls
                assert not ws[:4096 * 4].any(), f"counter head written M={m}"
            outs.append(y.cpu())
        ref = gptq.gemm_ref(x.numpy(), w)
        if m <= 64:
            assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16)), f"M={m}"
        else:
            check_tol(outs[1], ref, f"in-kernel gather M={m} path {path}")
        check_tol(outs[0], ref, f"gather-first M={m} path {path}")
        if path == _lib.DW4_PATH_PREFILL:  # automatic split: gathered rows after the planes
            say(f"act-order gather-first after split-K planes M={m}")
            ws = torch.zeros(_lib.workspace_size(m, k, n, 128, True), dtype=torch.uint8,
                             device=hip_device)
            y = torch.empty(m, n, dtype=torch.float16, device=hip_device)
            st = lib.dw4_gemm_path(path, 0, m, k, n, 128, xd.data_ptr(), k,
                                   q4.qweight.data_ptr(), q4.qzeros.data_ptr(),
                                   q4.scales.data_ptr(), q4.perm.data_ptr(), None,
                                   y.data_ptr(), n, ws.data_ptr(), ws.numel(),
                                   torch.cuda.current_stream().cuda_stream)
            assert st == _lib.DW4_OK, _lib.strerror(st)
            torch.cuda.synchronize()
            check_tol(y.cpu(), ref, f"gather-first split M={m}")


@pytest.mark.parametrize("g", [32, 64, 256, 1024])
def test_group_sizes(hip_device, g):
    k, n = 1024, 272  # N = 17 strips: a partial prefill N-tile
    for act in (False, True):
        lay, w = oracle_w(k, n, g, 3000 + g, False, act)
        q4 = build(lay, hip_device)
        for m in (1, 5, 24, 33, 64, 100):
            for path in ((_lib.DW4_PATH_DECODE, _lib.DW4_PATH_PREFILL) if m <= 64
                         else (_lib.DW4_PATH_PREFILL,)):
                say(f"group g={g} act={act} M={m} path={path}")
                x = make_x(m, k, seed=m + g)
                y = q4.matmul(x.to(hip_device), path=path)
                torch.cuda.synchronize()
                check_tol(y, gptq.gemm_ref(x.numpy(), w), f"g={g} act={act} M={m} path {path}")
        # dequantised weight bit-exact for every group size / act-order
        say(f"group g={g} act={act} dequant")
        wd = q4.get_float16_weights_matrix_v2().cpu().numpy()
        assert np.array_equal(wd.view(np.uint16), w.view(np.uint16))


def test_prefill_large_m_and_split_k(hip_device):
    lay, w = oracle_w(4096, 4096, 128, 1000, False, False)
    q4 = build(lay, hip_device)
    x = make_x(2048, 4096, seed=2048)
    ref = gptq.gemm_ref(x.numpy(), w)
    xd = x.to(hip_device)
    for split in (0, 1, 3, 8):
        say(f"prefill M=2048 split={split}")
        q4.tuning_params = TuningParams(PREFILL_SPLIT_K=split)
        y = q4.matmul(xd, path=_lib.DW4_PATH_PREFILL)
        torch.cuda.synchronize()
        check_tol(y, ref, f"M=2048 split {split}")


@pytest.mark.parametrize("kn", SHAPES_7B, ids=lambda kn: f"{kn[0]}x{kn[1]}")
def test_prefill_7b_large_m(hip_device, kn):
    """Config 3 at M = 1024 and 2048 on every 7B shape through the automatic
    path (64, 96 and 128 x 256 tiles of the LDS-streamed kernel, 11008 x 4096
    at M = 1024 split in two)."""
    k, n = kn
    lay, w = oracle_w(k, n, 128, 1000 + SHAPES_7B.index(kn), False, False)
    q4 = build(lay, hip_device)
    for m in (1024, 2048):
        say(f"prefill 7B {k}x{n} M={m}")
        x = make_x(m, k, seed=m + 13)
        y = q4.matmul(x.to(hip_device))
        torch.cuda.synchronize()
        check_tol(y, gptq.gemm_ref(x.numpy(), w), f"prefill {k}x{n} M={m}")


@pytest.mark.parametrize("k,n,m,g,act", [(1024, 400, 600, 128, False), (2048, 4112, 1000, 128, False),
                                         (1024, 400, 700, 64, True), (1024, 272, 520, 32, True),
                                         (1024, 400, 300, 64, True), (1024, 272, 200, 32, False),
                                         (1024, 4112, 2000, 32, True), (2048, 4112, 2000, 64, False),
                                         (4096, 4112, 200, 128, False), (4096, 2064, 300, 32, True),
                                         (2048, 4112, 400, 128, False), (4096, 1040, 250, 64, False),
                                         (4096, 4112, 160, 128, True)],
                         ids=["1024x400_M600", "2048x4112_M1000", "1024x400_M700_g64_act",
                              "1024x272_M520_g32_act", "1024x400_M300_g64_act",
                              "1024x272_M200_g32", "1024x4112_M2000_g32_act",
                              "2048x4112_M2000_g64", "4096x4112_M200_32row",
                              "4096x2064_M300_g32_act_4wave", "2048x4112_M400_4wave",
                              "4096x1040_M250_g64_32row", "4096x4112_M160_act_32row"])
def test_prefill_128_row_tiles_partial(hip_device, k, n, m, g, act):
    """The prefill path from 160 to 2000 rows with a partial last row tile, a
    partial last column tile (N not a multiple of the tile width) and group
    sizes 32 / 64 / 128, unsplit and split along K (the splits of a column
    tile spread over the XCDs as units of their own).  The planner's tiles,
    unsplit: K-sliced 64 x 32, 32 x 64 and 64 x 64 for the narrow and small
    ones, LDS-streamed 64 x 128 (M = 400) and 96 x 256 (M = 1000, 2000); the
    ids name the tiles of an earlier plan (test_gpu_prefill_tiles.py asserts
    a case's tile)."""
    lay, w = oracle_w(k, n, g, 5000 + m, False, act)
    q4 = build(lay, hip_device)
    for split in (0, 1, 2):
        say(f"prefill 128-row tiles {k}x{n} M={m} g={g} act={act} split={split}")
        q4.tuning_params = TuningParams(PREFILL_SPLIT_K=split)
        x = make_x(m, k, seed=m + g)
        y = q4.matmul(x.to(hip_device), path=_lib.DW4_PATH_PREFILL)
        torch.cuda.synchronize()
        check_tol(y, gptq.gemm_ref(x.numpy(), w), f"{k}x{n} M={m} split {split}")


@pytest.mark.parametrize("k,n,m", [(4096, 1040, 200), (4096, 1040, 256), (11008, 1040, 200),
                                   (4096, 1040, 600), (2048, 4112, 2000)],
                         ids=["32x128_M200", "32x128_M256", "64x256_K11008_M200",
                              "128x128_M600", "128x256_M2000"])
def test_prefill_bias_lds_streamed_tiles(hip_device, k, n, m):
    """Bias in the prefill kernels' epilogues, unsplit (split 1: the tile's own
    epilogue adds it) and split along K (2, and the plan's own choice: the
    reduce adds it), against the oracle plus bias.  The planner's tiles for
    these shapes: K-sliced 64 x 32 (K = 4096, M <= 256), 64 x 64 in three
    splits (K = 11008) and unsplit (M = 600), LDS-streamed 96 x 256 (M = 2000);
    the ids name the tiles of an earlier plan."""
    lay, w = oracle_w(k, n, 128, 6060 + m, False, False)
    q4 = build(lay, hip_device)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(6)) * 0.5).half()
    bd = bias.to(hip_device)
    for split in (0, 1, 2):
        say(f"prefill bias {k}x{n} M={m} split={split}")
        q4.tuning_params = TuningParams(PREFILL_SPLIT_K=split)
        x = make_x(m, k, seed=m + 606)
        y = q4.matmul(x.to(hip_device), bias=bd, path=_lib.DW4_PATH_PREFILL)
        torch.cuda.synchronize()
        ref = gptq.gemm_ref(x.numpy(), w) + bias.float().numpy()[None, :]
        check_tol(y, ref, f"bias {k}x{n} M={m} split {split}")


def test_shared_workspace_across_shapes(hip_device):
    """Two matrices share one workspace; decode split-K partials and prefill
    split-K calls of different tile counts alternate on it.  Each result
    stays within tolerance and the arrival counters at the head of the
    workspace are all zero after every call."""
    cache = CacheV2(hip_device)
    mats = {}
    for k, n in ((11008, 4096), (4096, 11008)):
        lay, w = oracle_w(k, n, 128, 1002 + k, False, False)
        d = lay.to(hip_device)
        mats[(k, n)] = (Q4MatrixV2(d.qweight, d.qzeros, d.scales, k, n, None, False,
                                   TuningParams(MAX_M=512), cache), w)
    cache.init_cache()
    head = 4096  # int32 arrival counters
    seq = [((11008, 4096), 16, _lib.DW4_PATH_DECODE, 0), ((4096, 11008), 100, _lib.DW4_PATH_PREFILL, 0),
           ((11008, 4096), 64, _lib.DW4_PATH_PREFILL, 0), ((4096, 11008), 16, _lib.DW4_PATH_PREFILL, 5),
           ((11008, 4096), 16, _lib.DW4_PATH_DECODE, 0), ((4096, 11008), 130, _lib.DW4_PATH_PREFILL, 2),
           ((4096, 11008), 100, _lib.DW4_PATH_PREFILL, 0)]
    for (k, n), m, path, split in seq:
        say(f"shared workspace {k}x{n} M={m} path={path} split={split}")
        q4, w = mats[(k, n)]
        q4.tuning_params = TuningParams(MAX_M=512, PREFILL_SPLIT_K=split)
        x = make_x(m, k, seed=m + k)
        y = q4.matmul(x.to(hip_device), path=path)
        torch.cuda.synchronize()
        check_tol(y, gptq.gemm_ref(x.numpy(), w), f"shared ws {k}x{n} M={m} path {path}")
        counters = cache.workspace[: head * 4].view(torch.int32)
        assert int(torch.count_nonzero(counters)) == 0


def test_operator_routes(hip_device):
    """QuantLinear end to end through every route the reference has:
    no-grad forward (HIP kernel), bias, bf16 activations, must_blas and
    reconstructed-weight dense products, and the input gradient of the
    grad-enabled forward (x @ W.T through the dequantised weight)."""
    from operators.core.linear.real_quant import QuantLinearMaker
    k, n = 1024, 512
    lay, w = oracle_w(k, n, 128, 4242, False, True)
    maker = QuantLinearMaker(quantization_group_size=128, use_act_order=True)
    with torch.device(hip_device):
        lin = maker.make_linear(k, n, bias=True)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(5)) * 0.5).half()
    lin.load_state_dict({"qweight": lay.qweight, "qzeros": lay.qzeros, "scales": lay.scales,
                         "g_idx": lay.g_idx, "bias": bias})
    cache = CacheV2(hip_device)
    maker.post_init(TuningParams(), cache)
    cache.init_cache()
    q4 = lin.q4_matrix
    x = make_x(24, k, seed=77)
    ref = gptq.gemm_ref(x.numpy(), w) + bias.float().numpy()
    xd = x.to(hip_device)
    say("operator: no-grad forward with bias")
    y = lin(xd.view(2, 12, k))
    torch.cuda.synchronize()
    assert tuple(y.shape) == (2, 12, n) and y.dtype == torch.float16
    check_tol(y.reshape(24, n), ref, "forward + bias")
    say("operator: bf16 activations")
    yb = lin(xd.to(torch.bfloat16))
    torch.cuda.synchronize()
    assert yb.dtype == torch.bfloat16
    wb = gptq.bf16_to_float(gptq.bf16_bits(w)).astype(np.float64)
    check_tol(yb.float(), x.to(torch.bfloat16).double().numpy() @ wb
              + bias.to(torch.bfloat16).double().numpy(), "bf16 forward")
    say("operator: must_blas dense route")
    yd = q4.matmul(xd, None, None, True, bias=bias.to(hip_device))
    torch.cuda.synchronize()
    check_tol(yd, ref, "must_blas")
    say("operator: reconstructed weight route")
    q4.reconstruct_weight(torch.float16)
    yr = lin(xd)
    q4.release_weight()
    torch.cuda.synchronize()
    check_tol(yr, ref, "reconstructed")
    say("operator: input gradient")
    xg = xd.clone().requires_grad_(True)
    yg = lin(xg)
    g = make_x(24, n, seed=78)
    yg.backward(g.to(hip_device))
    torch.cuda.synchronize()
    check_tol(yg.detach(), ref, "grad-enabled forward")
    gref = g.numpy().astype(np.float64) @ w.astype(np.float64).T
    check_tol(xg.grad, gref, "input gradient")


def test_unaligned_output_rows(hip_device):
    """y at an odd element offset with a row stride that is not a multiple
    of 8 halves (no 16-byte row segments): same bits as an aligned y."""
    lay, w = oracle_w(4096, 4096, 128, 1000, False, False)
    q4 = build(lay, hip_device)
    lib = _lib.load()
    ws = q4.cache.workspace
    for m, path in ((3, _lib.DW4_PATH_DECODE), (40, _lib.DW4_PATH_PREFILL),
                    (256, _lib.DW4_PATH_PREFILL)):
        say(f"unaligned y M={m} path={path}")
        x = make_x(m, 4096, seed=m + 500).to(hip_device)
        ref = q4.matmul(x, path=path)
        big = torch.full((m * 4100 + 8,), -1, dtype=torch.int16, device=hip_device)
        yv = big[1:1 + m * 4100].view(m, 4100)
        st = lib.dw4_gemm_path(path, 0, m, 4096, 4096, 128, x.data_ptr(), 4096,
                               q4.qweight.data_ptr(), q4.qzeros.data_ptr(), q4.scales.data_ptr(),
                               None, None, yv.data_ptr(), 4100, ws.data_ptr(), ws.numel(),
                               torch.cuda.current_stream().cuda_stream)
        assert st == _lib.DW4_OK
        torch.cuda.synchronize()
        assert torch.equal(yv[:, :4096], ref.view(torch.int16))
        assert bool((yv[:, 4096:] == -1).all()) and int(big[0]) == -1


def test_deterministic(hip_device):
    lay, _ = oracle_w(4096, 11008, 128, 1001, False, False)
    q4 = build(lay, hip_device)
    for m, path in ((1, _lib.DW4_PATH_DECODE), (16, _lib.DW4_PATH_DECODE),
                    (64, _lib.DW4_PATH_PREFILL), (256, _lib.DW4_PATH_PREFILL)):
        say(f"determinism M={m} path={path}")
        x = make_x(m, 4096, seed=99).to(hip_device)
        outs = [q4.matmul(x, path=path).clone() for _ in range(3)]
        torch.cuda.synchronize()
        for o in outs[1:]:
            assert torch.equal(o.view(torch.int16), outs[0].view(torch.int16))


def test_graph_capture_replay(hip_device):
    lay, w = oracle_w(4096, 4096, 128, 1000, False, False)
    q4 = build(lay, hip_device)
    for m in (1, 8, 256):
        say(f"graph capture M={m}")
        x = make_x(m, 4096, seed=5).to(hip_device)
        out = torch.empty(m, 4096, dtype=torch.float16, device=hip_device)
        eager = q4.matmul(x).clone()
        s = torch.cuda.Stream(device=hip_device)
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            q4.matmul(x, output=out)  # warm-up outside capture
        torch.cuda.current_stream().wait_stream(s)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            q4.matmul(x, output=out)
        for rep in range(3):
            out.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out.view(torch.int16), eager.view(torch.int16)), rep
            _ = (x * 2).sum().item()  # eager work between replays


def test_errors_surface(hip_device):
    lay, _ = oracle_w(4096, 4096, 128, 1000, False, False)
    q4 = build(lay, hip_device)
    lib = _lib.load()
    x = torch.zeros(2, 4096 + 8, dtype=torch.float16, device=hip_device)
    y = torch.empty(1, 4096, dtype=torch.float16, device=hip_device)
    say("errors: misaligned x pointer")
    st = lib.dw4_gemm(1, 4096, 4096, 128, x.data_ptr() + 2, 4096, q4.qweight.data_ptr(),
                      q4.qzeros.data_ptr(), q4.scales.data_ptr(), None, None, y.data_ptr(), 4096,
                      None, 0, None)
    assert st == _lib.DW4_ERR_MISALIGNED
    say("errors: unsupported K")
    st = lib.dw4_gemm(1, 96, 4096, 32, x.data_ptr(), 96, q4.qweight.data_ptr(), q4.qzeros.data_ptr(),
                      q4.scales.data_ptr(), None, None, y.data_ptr(), 4096, None, 0, None)
    assert st == _lib.DW4_ERR_UNSUPPORTED
    say("errors: split decode without workspace")
    # M=4 x K=13824 activations exceed one workgroup's LDS share at N=5120:
    # fp32 split-K partials needed (all-zero packed buffers of the right sizes)
    kb, nb = 13824, 5120
    pq = torch.zeros(kb // 8 * nb, dtype=torch.int32, device=hip_device)
    pz = torch.zeros(kb // 128 * nb // 8, dtype=torch.int32, device=hip_device)
    ps = torch.zeros(kb // 128 * nb, dtype=torch.float16, device=hip_device)
    xs = torch.zeros(4, kb, dtype=torch.float16, device=hip_device)
    ys = torch.empty(4, nb, dtype=torch.float16, device=hip_device)
    assert _lib.workspace_size(4, kb, nb, 128, False) > 0
    st = lib.dw4_gemm_path(_lib.DW4_PATH_DECODE, 0, 4, kb, nb, 128, xs.data_ptr(), kb,
                           pq.data_ptr(), pz.data_ptr(), ps.data_ptr(), None,
                           None, ys.data_ptr(), nb, None, 0, None)
    assert st == _lib.DW4_ERR_WORKSPACE
    say("errors: misaligned view goes through an aligned copy")
    xv = x[:, 1:4097]
    out = q4.matmul(xv)
    ref = q4.matmul(xv.contiguous())
    torch.cuda.synchronize()
    assert torch.equal(out, ref)


# ---------------------------------------------------------------------------
# bf16 route (dequantise to bf16, dense bf16 product with fp32 accumulation)
# ---------------------------------------------------------------------------
def test_bf16_dequant_exhaustive_kat(hip_device):
    """bf16 weights: all 16 q x 16 stored zeros x 65,536 fp16 scale patterns,
    bit for bit against bf16(oracle fp16 weight) (NaNs as a class)."""
    say("exhaustive bf16 dequant KAT K=512 N=65536 g=32")
    K, N, G = 512, 65536, 16
    q = np.zeros((K, N), dtype=np.uint8)
    for z in range(16):
        for qq in range(16):
            q[z * 32 + 2 * qq: z * 32 + 2 * qq + 2, :] = qq
    zeros = np.repeat(np.arange(16, dtype=np.uint8)[:, None], N, axis=1)
    srow = np.arange(65536, dtype=np.uint32).astype(np.uint16)
    scales = np.repeat(srow[None, :], G, axis=0).view(np.float16)
    qweight, qzeros = gptq.pack_qweight(q), gptq.pack_qzeros(zeros)
    g_idx = (np.arange(K) // 32).astype(np.int32)
    with np.errstate(all="ignore"):
        ref = gptq.dequantize_bf16(qweight, qzeros, scales, g_idx)
    cache = CacheV2(hip_device)
    q4 = Q4MatrixV2(torch.from_numpy(qweight).to(hip_device), torch.from_numpy(qzeros).to(hip_device),
                    torch.from_numpy(scales).to(hip_device), K, N, None, False, TuningParams(), cache)
    w = q4.get_bfloat16_weights_matrix_v2().view(torch.int16).cpu().numpy().view(np.uint16)
    nan = np.isnan(gptq.bf16_to_float(ref))
    same = (w == ref) | (nan & np.isnan(gptq.bf16_to_float(w)))
    assert same.all(), np.argwhere(~same)[:5]


@pytest.mark.parametrize("act", [False, True], ids=["plain", "act"])
def test_bf16_route_beyond_fp16_range(hip_device, act):
    """bf16 activations whose values exceed fp16's range (|x| up to 3e5):
    the product keeps them (fp16 narrowing would give inf), within the
    GEMM tolerance of the float64 product of x and the bf16 oracle weight;
    the activation gradient takes the same bf16 route."""
    k, n = 1024, 768
    lay, _ = oracle_w(k, n, 128, 515 + act, False, act)
    a = lay.numpy()
    wb = gptq.bf16_to_float(gptq.dequantize_bf16(a["qweight"], a["qzeros"], a["scales"],
                                                 a["g_idx"])).astype(np.float64)
    q4 = build(lay, hip_device)
    gen = torch.Generator().manual_seed(31)
    for m in (1, 16, 300):
        say(f"bf16 route act={act} M={m}")
        x = (torch.randn(m, k, generator=gen) * 1e5).to(torch.bfloat16)
        assert float(x.float().abs().max()) > 65504.0
        xd = x.to(hip_device)
        y = q4.matmul(xd)
        torch.cuda.synchronize()
        assert y.dtype == torch.bfloat16
        ref = x.double().numpy() @ wb
        check_tol(y.float(), ref, f"bf16 forward M={m}")
        g = (torch.randn(m, n, generator=gen) * 1e5).to(torch.bfloat16)
        gx = q4.transpose_matmul(g.to(hip_device))
        torch.cuda.synchronize()
        assert gx.dtype == torch.bfloat16
        check_tol(gx.float(), g.double().numpy() @ wb.T, f"bf16 transpose M={m}")
    say("bf16 reconstructed-weight route")
    q4.reconstruct_weight(torch.bfloat16)
    assert torch.equal(q4.reconstructed_weight_bfloat16.view(torch.int16).cpu(),
                       torch.from_numpy(gptq.dequantize_bf16(
                           a["qweight"], a["qzeros"], a["scales"], a["g_idx"]).view(np.int16)))
    x = (torch.randn(8, k, generator=gen) * 1e5).to(torch.bfloat16)
    y = q4.matmul(x.to(hip_device))
    q4.release_weight(torch.bfloat16)
    torch.cuda.synchronize()
    check_tol(y.float(), x.double().numpy() @ wb, "bf16 reconstructed")


@pytest.mark.parametrize("k,n,g,sym,act", [
    (4096, 4096, 128, False, False),   # 16-wave workgroups, one strip each
    (4096, 11008, 128, False, False),  # 8 waves, two strips per workgroup
    (11008, 4096, 128, True, False),   # symmetric zeros, 86 chunks over 16 waves
    (5120, 5120, 128, False, True),    # act-order, x gathered into the workspace
    (1024, 768, 32, False, False),     # groups of 32 (four per chunk), waves without chunks
    (768, 512, 64, False, True),       # groups of 64, act-order, six chunks
    (1024, 8192, 64, False, False),    # groups of 64, two strips per workgroup up to 48 rows
], ids=["4096sq", "4096x11008", "11008x4096_sym", "5120sq_act", "g32", "g64_act", "g64_wide"])
def test_bf16_native_decode(hip_device, k, n, g, sym, act):
    """bf16 activations at 1 <= M <= BF16_MAX_M take dw4_gemm_bf16 (the
    register-fed kernel's bf16 mode, one to four 16-row tiles in one launch):
    within the GEMM tolerance of the float64 product of x with the dense
    route's weight bf16(fp16(s(q - z))) and with the exact fp16 weight, bias
    added after the bf16 rounding, equal bits on a repeat; q4.matmul returns
    exactly what the C entry point writes; act-order without workspace room
    (every workgroup gathering) gives the same bits; one row past the limit
    takes the prefill kernels' bf16 form (dw4_gemm_bf16_prefill)."""
    lay, w = oracle_w(k, n, g, 7100 + k + n, sym, act)
    a = lay.numpy()
    wb = gptq.bf16_to_float(gptq.dequantize_bf16(a["qweight"], a["qzeros"], a["scales"],
                                                 a["g_idx"])).astype(np.float64)
    q4 = build(lay, hip_device)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(8)) * 0.5).to(torch.bfloat16)
    bd = bias.to(hip_device)
    lib = _lib.load()
    for m in (1, 3, 8, 16, 17, 32, 40, 49, _lib.BF16_MAX_M, _lib.BF16_MAX_M + 1):
        say(f"bf16 native {k}x{n} g={g} sym={sym} act={act} M={m}")
        x = make_x(m, k, seed=m + 7).to(torch.bfloat16)
        xd = x.to(hip_device)
        y = q4.matmul(xd, bias=bd)
        again = q4.matmul(xd, bias=bd)
        torch.cuda.synchronize()
        assert y.dtype == torch.bfloat16 and tuple(y.shape) == (m, n)
        assert torch.equal(y.view(torch.int16), again.view(torch.int16))
        xb = x.double().numpy()
        check_tol(y.float(), xb @ wb + bias.double().numpy(), f"bf16 M={m} vs bf16 weight")
        check_tol(y.float(), xb @ w + bias.double().numpy(), f"bf16 M={m} vs fp16 weight")
        if m > _lib.BF16_MAX_M:
            continue
        perm = q4.perm.data_ptr() if q4.use_act else None
        for ws, ws_bytes in ((q4.cache.workspace.data_ptr(), q4.cache.workspace.numel()),
                             (None, 0)):
            direct = torch.empty(m, n, dtype=torch.bfloat16, device=hip_device)
            _lib.check("dw4_gemm_bf16", lib.dw4_gemm_bf16(
                m, k, n, g, xd.data_ptr(), k, q4.qweight.data_ptr(), q4.qzeros.data_ptr(),
                q4.scales.data_ptr(), perm, bd.data_ptr(), direct.data_ptr(), n, ws, ws_bytes,
                None))
            torch.cuda.synchronize()
            assert torch.equal(direct.view(torch.int16), y.view(torch.int16)), \
                f"M={m} workspace={ws is not None}"


def test_output_argument_contract(hip_device):
    """A caller's output receives the product or the call raises: row-strided
    [M, N] views are written in place; wrong dtype, wrong size or a
    non-row-major layout raise before any launch."""
    lay, w = oracle_w(4096, 4096, 128, 1000, False, False)
    q4 = build(lay, hip_device)
    for m, path in ((4, _lib.DW4_PATH_DECODE), (96, _lib.DW4_PATH_PREFILL)):
        say(f"output contract M={m} path={path}")
        x = make_x(m, 4096, seed=m + 900).to(hip_device)
        ref = q4.matmul(x, path=path)
        big = torch.full((m, 4096 + 64), -7.0, dtype=torch.float16, device=hip_device)
        view = big[:, 32:32 + 4096]
        got = q4.matmul(x, output=view, path=path)
        torch.cuda.synchronize()
        assert got is view
        assert torch.equal(view, ref)
        assert bool((big[:, :32] == -7.0).all()) and bool((big[:, 32 + 4096:] == -7.0).all())
        flat = torch.empty(m * 4096, dtype=torch.float16, device=hip_device)
        got = q4.matmul(x, output=flat, path=path)
        torch.cuda.synchronize()
        assert got is flat and torch.equal(flat.view(m, 4096), ref)
        with pytest.raises(TypeError):
            q4.matmul(x, output=torch.empty(m, 4096, dtype=torch.float32, device=hip_device))
        with pytest.raises(ValueError):
            q4.matmul(x, output=torch.empty(m, 4095, dtype=torch.float16, device=hip_device))
        with pytest.raises(ValueError):
            q4.matmul(x, output=torch.empty(4096, m, dtype=torch.float16, device=hip_device).t())
    for m in (1, 5, 37):
        say(f"output contract bf16 native M={m}, row-strided x and output")
        xb = make_x(m, 4096, seed=m + 950).to(torch.bfloat16).to(hip_device)
        ref = q4.matmul(xb)
        wide = torch.zeros(m, 4096 + 24, dtype=torch.bfloat16, device=hip_device)
        wide[:, 16:16 + 4096] = xb  # ldx = 4120 (a multiple of 8), base 32 bytes in
        big = torch.full((m, 4096 + 64), -7.0, dtype=torch.bfloat16, device=hip_device)
        view = big[:, 32:32 + 4096]
        got = q4.matmul(wide[:, 16:16 + 4096], output=view)
        torch.cuda.synchronize()
        assert got is view and torch.equal(view.view(torch.int16), ref.view(torch.int16))
        assert bool((big[:, :32] == -7.0).all()) and bool((big[:, 32 + 4096:] == -7.0).all())
