"""GPU parity of the transposed W4A16 product (dw4_gemm_t, the PEFT
backward out = g @ W^T) against the oracle, through the C ABI and through
Q4MatrixV2.transpose_matmul / autograd.

Bar: max|out - out_ref| <= 2e-2 * ||out_ref row||_inf, out_ref = g @ W^T in
float64 with W the oracle's dequantised weight.  Covers Llama-2-7B shapes,
act-order 13B, group sizes 32/64/256/1024 and g = K, N-ranges that do not
divide the strips, M across one and several 64-row blocks, determinism and
the error statuses.  Every case prints its name before touching the GPU.
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
from hip_extends.w4a16 import CacheV2, Q4LinearFunction, Q4MatrixV2, TuningParams
from oracle import gptq

pytestmark = pytest.mark.gpu

TOL = 2e-2


def say(msg: str) -> None:
    print(f"[case] {msg}", flush=True)
    sys.stdout.flush()


@functools.lru_cache(maxsize=16)
def _layer(k, n, g, seed, act):
    lay = make_layer(k, n, g, seed=seed, act_order=act)
    a = lay.numpy()
    return lay, gptq.dequantize(a["qweight"], a["qzeros"], a["scales"], a["g_idx"])


def _matrix(lay, dev, max_m=256):
    cache = CacheV2(dev)
    d = lay.to(dev)
    q4 = Q4MatrixV2(d.qweight, d.qzeros, d.scales, d.in_features, d.out_features,
                    d.g_idx if d.act_order else None, d.act_order,
                    TuningParams(MAX_M=max_m, TRANSPOSE_MAX_M=4096), cache)
    cache.init_cache()
    return q4


def _gemm_t(q4, g2):
    m = g2.shape[0]
    out = torch.full((m, q4.height), float("nan"), dtype=torch.float16, device=g2.device)
    nbytes = _lib.gemm_t_workspace_size(m, q4.height, q4.width, q4.group_size)
    ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=g2.device)
    _lib.call("dw4_gemm_t", m, q4.height, q4.width, q4.group_size, g2.data_ptr(), g2.stride(0),
              q4.qweight.data_ptr(), q4.qzeros.data_ptr(), q4.scales.data_ptr(),
              q4.perm.data_ptr() if q4.use_act else None, out.data_ptr(), out.stride(0),
              ws.data_ptr(), ws.numel(), torch.cuda.current_stream(g2.device).cuda_stream)
    return out


def _check(out, g, w, what):
    ref = g.numpy().astype(np.float64) @ w.astype(np.float64).T
    y = out.float().cpu().numpy()
    assert np.all(np.isfinite(y)), what
    ok, worst = gptq.within_tolerance(y, ref, TOL)
    assert ok, f"{what}: worst error ratio {worst:.4f} > 1"


@pytest.mark.parametrize("shape", [(4096, 4096), (4096, 11008), (11008, 4096)],
                         ids=["4096x4096", "4096x11008", "11008x4096"])
def test_transpose_7b(hip_device, shape):
    k, n = shape
    lay, w = _layer(k, n, 128, 3000 + k + n, False)
    q4 = _matrix(lay, hip_device)
    for m in (1, 5, 16, 33, 64, 65, 100, 256):
        say(f"gemm_t {k}x{n} M={m}")
        g = make_x(m, n, seed=4000 + m)
        out = _gemm_t(q4, g.to(hip_device))
        torch.cuda.synchronize()
        _check(out, g, w, f"{k}x{n} M={m}")


@pytest.mark.parametrize("k,n,gs,act", [(5120, 13824, 128, True), (1024, 512, 32, False),
                                        (1024, 512, 64, True), (2048, 272, 256, True),
                                        (1024, 80, 1024, False), (128, 4096, 128, True)])
def test_transpose_groups_and_act(hip_device, k, n, gs, act):
    lay, w = _layer(k, n, gs, 5000 + k + n + gs, act)
    q4 = _matrix(lay, hip_device)
    for m in (1, 8, 70):
        say(f"gemm_t {k}x{n} g={gs} act={act} M={m}")
        g = make_x(m, n, seed=6000 + m)
        out = _gemm_t(q4, g.to(hip_device))
        torch.cuda.synchronize()
        _check(out, g, w, f"{k}x{n} g={gs} act={act} M={m}")


def test_transpose_deterministic_and_routes(hip_device):
    lay, w = _layer(4096, 11008, 128, 7000, True)
    q4 = _matrix(lay, hip_device)
    g = make_x(24, 11008, seed=7001).to(hip_device)
    say("gemm_t determinism")
    a = _gemm_t(q4, g)
    b = _gemm_t(q4, g)
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    say("transpose_matmul native vs dense route")
    native = q4.transpose_matmul(g.view(2, 12, 11008))
    q4.tuning_params = TuningParams(TRANSPOSE_MAX_M=0)
    dense = q4.transpose_matmul(g.view(2, 12, 11008))
    torch.cuda.synchronize()
    assert native.shape == dense.shape == (2, 12, 4096)
    _check(native.view(24, 4096), g.cpu(), w, "native route")
    _check(dense.view(24, 4096), g.cpu(), w, "dense route")
    say("autograd backward through the native kernel")
    q4.tuning_params = TuningParams(TRANSPOSE_MAX_M=256)
    x = make_x(24, 4096, seed=7002).to(hip_device).requires_grad_(True)
    y = Q4LinearFunction.apply(x, q4, None, False)
    y.backward(g)
    torch.cuda.synchronize()
    _check(x.grad, g.cpu(), w, "autograd grad_input")


def test_transpose_status(hip_device):
    lay, _ = _layer(1024, 512, 32, 8000, False)
    q4 = _matrix(lay, hip_device)
    lib = _lib.load()
    g = torch.zeros(4, 512, dtype=torch.float16, device=hip_device)
    out = torch.empty(4, 1024, dtype=torch.float16, device=hip_device)
    args = (q4.qweight.data_ptr(), q4.qzeros.data_ptr(), q4.scales.data_ptr(), None,
            out.data_ptr(), 1024)
    say("gemm_t statuses")
    assert lib.dw4_gemm_t(4, 1024, 500, 32, g.data_ptr(), 512, *args, None, 0, None) == \
        _lib.DW4_ERR_UNSUPPORTED
    assert lib.dw4_gemm_t(4, 1024, 512, 32, g.data_ptr() + 2, 512, *args, None, 0, None) == \
        _lib.DW4_ERR_MISALIGNED
    need = _lib.gemm_t_workspace_size(4, 1024, 512, 32)
    if need:
        assert lib.dw4_gemm_t(4, 1024, 512, 32, g.data_ptr(), 512, *args, None, 0, None) == \
            _lib.DW4_ERR_WORKSPACE
    assert lib.dw4_gemm_t(0, 1024, 512, 32, None, 512, *args, None, 0, None) == _lib.DW4_OK


# Tiles of 48 and 64 rows with their remainders, an odd number of strips (the
# last in a pair of its own), one chunk row, N-ranges, groups of 32 to K.  The
# weight is exact in both, so the bound is the fp16 rounding of the result
# (2^-11) plus fp32 sums of n products (n 2^-24 of the sum of magnitudes).
@pytest.mark.parametrize("k,n,group,act", [
    (128, 16, 32, False), (128, 48, 128, False), (256, 272, 64, True), (1152, 1056, 128, True),
    (512, 4112, 512, False), (4096, 4096, 128, False)])
def test_tall_rows_edges(hip_device, k, n, group, act):
    lay, w = _layer(k, n, group, 8100 + k + n, act)
    q4 = _matrix(lay, hip_device)
    wd = w.astype(np.float64)
    for m in (65, 96, 97, 128, 129, 385):
        say(f"tall gemm_t {k}x{n} g={group} act={act} M={m}")
        g = make_x(m, n, seed=8200 + m)
        gd = g.numpy().astype(np.float64)
        out = _gemm_t(q4, g.to(hip_device)).double().cpu().numpy()
        bound = 2.0 ** -11 * np.abs(gd @ wd.T) + n * 2.0 ** -24 * (np.abs(gd) @ np.abs(wd).T) + 2.0 ** -24
        assert np.all(np.abs(out - gd @ wd.T) <= bound), (m, k, n)


def test_tall_overflowing_weight_stays_at_its_output(hip_device):
    # s (q - z) beyond fp16 in one group of one column: infinite weights at
    # some of its rows k only, and the other outputs as the dense product has them
    lay, _ = _layer(256, 64, 128, 8300, False)
    scales = lay.scales.clone()
    scales[1, 5] = 30000.0
    cache = CacheV2(hip_device)
    q4 = Q4MatrixV2(*(t.to(hip_device) for t in (lay.qweight, lay.qzeros, scales)), 256, 64, None, False,
                    TuningParams(MAX_M=256, TRANSPOSE_MAX_M=128), cache)
    cache.init_cache()
    g = (make_x(200, 64, seed=8301) * 0.01).to(hip_device)
    w = q4.get_float16_weights_matrix_v2()
    finite = torch.isfinite(w).all(dim=1)
    assert finite.any() and not finite.all()
    say("tall gemm_t with overflowing weights")
    out = _gemm_t(q4, g).float()
    ref = g.float() @ w.float().t().contiguous()
    assert torch.isfinite(out[:, finite]).all()
    assert torch.equal(out[:, ~finite], ref[:, ~finite])


def test_transpose_above_limit_keeps_dense_semantics(hip_device):
    lay, w = _layer(1152, 1056, 128, 8400, True)
    q4 = _matrix(lay, hip_device)
    q4.tuning_params = TuningParams(TRANSPOSE_MAX_M=64)
    assert _lib.gemm_t_packed(200, 1152, 1056, 128)
    g = make_x(200, 1056, seed=8401).to(hip_device)
    say("packed above the limit, then the calls that keep the dense product")
    _check(q4.transpose_matmul(g), g.cpu(), w, "packed")
    buf = torch.zeros(1152 * 1056, dtype=torch.float16, device=hip_device)
    q4.transpose_matmul(g, None, buf)
    assert torch.equal(buf.view(1152, 1056), q4.get_float16_weights_matrix_v2())
    tracked = g.clone().requires_grad_(True)
    assert q4.transpose_matmul(tracked).requires_grad
    out = torch.func.vmap(q4.transpose_matmul)(g.view(2, 100, 1056))
    _check(out.view(200, 1152), g.cpu(), w, "vmap")


@pytest.mark.parametrize("m", [1, 384, 3000])
def test_backward_with_kept_weight(hip_device, m):
    lay, w = _layer(1152, 1056, 128, 8500, True)
    q4 = _matrix(lay, hip_device)
    q4.tuning_params = TuningParams(MAX_M=256)
    x = make_x(m, 1152, seed=8501).to(hip_device).requires_grad_(True)
    dy = make_x(m, 1056, seed=8502).to(hip_device)
    say(f"gradient with the weight kept, M={m}: first order, and recorded")
    y = Q4LinearFunction.apply(x, q4, None, True)
    dx, = torch.autograd.grad(y, x, dy, retain_graph=True)
    _check(dx, dy.cpu(), w, "gradient")
    tracked = dy.clone().requires_grad_(True)
    dx2, = torch.autograd.grad(y, x, tracked, create_graph=True)
    q4.cache.temp_weight.zero_()
    ddy, = torch.autograd.grad(dx2, tracked, x.detach())
    _check(ddy, x.detach().cpu(), w.T, "second order")


def _trained(q4, m, seed):
    x = make_x(m, q4.height, seed=seed).to(q4.device).requires_grad_(True)
    dy = make_x(m, q4.width, seed=seed + 1).to(q4.device)
    return x, dy


def _step(q4, x, dy, kept=True):
    y = Q4LinearFunction.apply(x, q4, None, kept)
    return torch.autograd.grad(y, x, dy)[0]


def test_captured_backward_owns_its_planes(hip_device):
    """A forward and backward of 8 rows captured, then larger backwards through
    the same cache, which once shared one buffer of planes, freed as it grew."""
    lay, w = _layer(1152, 1056, 128, 8600, True)
    q4 = _matrix(lay, hip_device)
    q4.tuning_params = TuningParams(MAX_M=256)
    assert _lib.gemm_t_workspace_size(8, 1152, 1056, 128) > 0  # planes there are
    x, dy = _trained(q4, 8, 8601)
    say("captured forward and backward of 8 rows, larger ones between the replays")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        want = _step(q4, x, dy)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = _step(q4, x, dy)
    for i, m in enumerate((64, 100, 128)):
        got.fill_(float("nan"))
        graph.replay()
        big, dbig = _trained(q4, m, 8610 + i)
        dx = _step(q4, big, dbig)
        fill = [torch.full((1 << 18,), float(i), device=hip_device) for _ in range(8)]
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        assert all(bool((f == i).all()) for f in fill)
        _check(dx, dbig.cpu(), w, f"eager backward of {m} rows")


def test_backwards_on_two_streams(hip_device):
    lay, _ = _layer(1152, 1056, 128, 8600, True)
    q4 = _matrix(lay, hip_device)
    q4.tuning_params = TuningParams(MAX_M=256)
    grads = [_trained(q4, m, 8620 + m)[1] for m in (8, 100)]
    want = [q4.transpose_matmul(g) for g in grads]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in grads]
    say("transposed products on two streams")
    outs = [[], []]
    for _ in range(20):
        for i, st in enumerate(streams):
            with torch.cuda.stream(st):
                outs[i].append(q4.transpose_matmul(grads[i]))
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(o, want[i]) for o in outs[i])


def test_kept_backward_is_of_the_forwards_words(hip_device):
    """The matrix pointed at other words, or its limit changed, between the
    forward and the backward: the gradient stays that of the forward; words
    overwritten in place are refused."""
    lay, w = _layer(1152, 1056, 128, 8600, True)
    q4 = _matrix(lay, hip_device)
    q4.tuning_params = TuningParams(MAX_M=256)
    x, dy = _trained(q4, 24, 8630)
    say("backward after rebind, after a new limit, after an overwrite")
    y = Q4LinearFunction.apply(x, q4, None, True)
    words = [t.clone() for t in q4._words()]
    q4.rebind(torch.zeros_like(words[0]), *words[1:])
    _check(torch.autograd.grad(y, x, dy)[0], dy.cpu(), w, "rebound")
    q4.rebind(*words)
    y = Q4LinearFunction.apply(x, q4, None, True)
    q4.set_tuning_params(TuningParams(MAX_M=256, TRANSPOSE_MAX_M=0))
    _check(torch.autograd.grad(y, x, dy)[0], dy.cpu(), w, "new limit")
    q4.set_tuning_params(TuningParams(MAX_M=256))
    y = Q4LinearFunction.apply(x, q4, None, True)
    q4.qweight.zero_()
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(y, x, dy)
