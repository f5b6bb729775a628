"""Performance cases of the quantized-Linear framework.

Each case is the work one call site of a serving or fine-tuning program has
the framework do, through its public entry points.  Projection sizes are the
repository's benchmark shapes (Llama-2 7B and 13B) and, in drawn cases, generic
ones; checkpoints are random GPTQ 4-bit tensors in the checkpoint format with
the value ranges of quantised weights.

Kinds of cases:

* ``linear``    ``QuantLinear.forward`` of one projection, from one decode row
                to a long prompt, fp16 or bf16, with or without act-order;
* ``finetune``  the same with the input's gradient: forward and backward of a
                frozen projection under adapter training;
* ``step``      one decode token through every projection of several layers,
                captured in a graph, as a serving loop replays it per batch size;
* ``stage``     a whole decode step of several decoder layers (norms, q/k/v,
                rotary embedding, cache write, paged attention, MLP), captured
                in a graph;
* ``tail``      the decoder layer after attention (o, norm, gate/up, down);
* ``prompt``    the layer before attention on a prompt: norm, q/k/v, rotary
                embedding and the prompt's keys and values into cache blocks;
* ``attention`` paged-attention decode alone;
* ``swap``      a sequence's keys and values into cache blocks and back, as
                swapping a request in and out does.

``exact`` restates each path in float64 torch (weights s * (q - z), no
intermediate rounding).  Tolerances are about four times the difference
measured between two correct roundings of the same product (fp16 results:
one rounding of 2^-12 rms on the output and at most one on the weights; bf16
results: the same at 2^-9).
"""
import os
import sys

import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "drofell-for-revision_amd")
for _p in (PKG, REPO):
    if _p not in sys.path:
        sys.path.insert(0, _p)

from hip_extends.w4a16 import (CacheV2, TuningParams, attention_forward_qkv_stage_v2_py,  # noqa: E402
                               attention_forward_rope_stage_v2_py, decoder_after_stage_v2_py,
                               gemm_group)
from operators import flags  # noqa: E402
from operators.core.attention.common import AttentionConfig  # noqa: E402
from operators.core.attention.real_page import PagedAttention  # noqa: E402
from operators.core.block.common import BlockInfo  # noqa: E402
from operators.core.block.real import LayerBlocksHolder  # noqa: E402
from operators.core.linear.real_quant import QuantLinearMaker  # noqa: E402

EPS = 1e-5
# hidden size, MLP width, heads of head size 128
LAYERS = {"7b": (4096, 11008, 32), "13b": (5120, 13824, 40)}


def listed():
    return [
        # one decode row through one projection: the smallest call there is,
        # where the call itself counts
        dict(name="linear-1row", kind="linear", rows=1, k=4096, n=4096, group=128, act=False,
             bias=False, dtype="fp16"),
        # a decode batch on an act-order checkpoint's widest projection
        dict(name="linear-45rows-act", kind="linear", rows=45, k=5120, n=13824, group=128, act=True,
             bias=False, dtype="fp16"),
        # a short prompt (or a chunk of one) through an MLP projection
        dict(name="linear-300rows", kind="linear", rows=300, k=4096, n=11008, group=128, act=False,
             bias=False, dtype="fp16"),
        # several long prompts at once
        dict(name="linear-3500rows-g64", kind="linear", rows=3500, k=11008, n=4096, group=64,
             act=False, bias=False, dtype="fp16"),
        # a prompt with bf16 activations
        dict(name="linear-700rows-bf16", kind="linear", rows=700, k=4096, n=4096, group=128,
             act=False, bias=True, dtype="bf16"),
        # adapter training over a frozen projection, one sequence
        dict(name="finetune-384rows", kind="finetune", rows=384, k=4096, n=11008, group=128,
             act=False, bias=False, dtype="fp16"),
        # one token of one request through all projections of four layers
        dict(name="step-1row", kind="step", rows=1, size="7b", layers=4, group=128, act=False),
        # one token of eight requests through four whole decoder layers
        dict(name="stage-8seqs", kind="stage", seqs=8, ctx=600, size="7b", layers=4, group=128,
             block=16),
        # the layer after attention on a chunk of a prompt
        dict(name="tail-100rows", kind="tail", rows=100, size="7b", group=128, act=False),
        # the layer before attention on a prompt
        dict(name="prompt-1000rows", kind="prompt", rows=1000, size="7b", group=128, block=32),
        # long-context decode with grouped query heads
        dict(name="attention-gqa-long", kind="attention", seqs=24, ctx=3000, heads=32, kv_heads=8,
             head_dim=128, block=32),
        # a request's cached keys and values written and read back
        dict(name="swap-1500rows", kind="swap", rows=1500, kv_heads=32, head_dim=128, block=32),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


# a drawn case stays below the largest listed one
_MOST_FLOPS = 2 * 3500 * 11008 * 4096


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "finetune", "step", "stage", "tail", "prompt",
                       "attention", "swap"])
    if kind in ("linear", "finetune"):
        k, n = rng.choice([(4096, 4096), (4096, 11008), (11008, 4096), (4096, 12288), (4096, 22016),
                           (5120, 5120), (5120, 13824), (13824, 5120),
                           (128 * rng.randint(8, 90), 32 * rng.randint(32, 400))])
        groups = [g for g in (32, 64, 128, 128, 128, 256) if k % g == 0]
        most = min(3500 if kind == "linear" else 1500, _MOST_FLOPS // (2 * k * n))
        return dict(kind=kind, rows=_log_int(rng, 1, most), k=k, n=n, group=rng.choice(groups),
                    act=rng.random() < 0.3, bias=rng.random() < 0.3,
                    dtype=rng.choice(["fp16", "fp16", "bf16"]))
    size = rng.choice(["7b", "13b"])
    group = rng.choice([64, 128, 128])
    if kind == "step":
        return dict(kind=kind, rows=_log_int(rng, 1, 32), size=size, layers=rng.randint(1, 4),
                    group=group, act=rng.random() < 0.3)
    if kind == "stage":
        return dict(kind=kind, seqs=_log_int(rng, 1, 24), ctx=_log_int(rng, 16, 2000), size=size,
                    layers=rng.randint(1, 3), group=group, block=rng.choice([16, 32]))
    if kind == "tail":
        return dict(kind=kind, rows=_log_int(rng, 1, 1000), size=size, group=group,
                    act=rng.random() < 0.3)
    if kind == "prompt":
        return dict(kind=kind, rows=_log_int(rng, 16, 1500), size=size, group=group,
                    block=rng.choice([16, 32]))
    if kind == "attention":
        heads, kv_heads = rng.choice([(32, 32), (40, 40), (32, 8), (64, 8), (8, 2)])
        return dict(kind=kind, seqs=_log_int(rng, 1, 32), ctx=_log_int(rng, 16, 4000), heads=heads,
                    kv_heads=kv_heads, head_dim=rng.choice([64, 80, 96, 128, 128, 128, 256]),
                    block=rng.choice([16, 32]))
    return dict(kind=kind, rows=_log_int(rng, 16, 3000), kv_heads=rng.choice([8, 32, 40]),
                head_dim=rng.choice([64, 128]), block=rng.choice([16, 32]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(gen, *shape):
    return torch.randn(*shape, device="cuda", generator=gen)


def _checkpoint(gen, k, n, group, perm):
    """A GPTQ projection: 4-bit codes around the middle of the range, stored
    zeros (effective zero - 1) around 7, scales that give weights of about
    1 / sqrt(k), and for act-order (perm) a permuted group index."""
    q = (_normal(gen, k, n) * 3.0 + 7.5).round_().clamp_(0, 15).to(torch.int32)
    z = (_normal(gen, k // group, n) * 1.5 + 7.0).round_().clamp_(0, 15).to(torch.int32)
    scales = ((0.7 + 0.6 * torch.rand(k // group, n, device="cuda", generator=gen))
              * (0.3 / k ** 0.5)).to(torch.float16)
    rank = torch.arange(k, device="cuda") if perm is None else perm
    return q, z, scales, torch.div(rank, group, rounding_mode="floor").to(torch.int32)


def _checkpoints(gen, mats, group, act):
    """One checkpoint per (k, n, input): with act-order, projections of the
    same input (q, k, v; gate, up) are quantised in the same row order."""
    last, perm = None, None
    for k, n, source in mats:
        if act and (perm is None or source != last):
            perm = torch.randperm(k, device="cuda", generator=gen)
        last = source
        yield k, n, _checkpoint(gen, k, n, group, perm)


def _packed(q, z):
    qweight = torch.zeros(q.shape[0] // 8, q.shape[1], dtype=torch.int32, device=q.device)
    qzeros = torch.zeros(z.shape[0], z.shape[1] // 8, dtype=torch.int32, device=q.device)
    for i in range(8):
        qweight |= q[i::8] << (4 * i)
        qzeros |= z[:, i::8] << (4 * i)
    return qweight, qzeros


def _linears(gen, mats, group, act, rows, bias=False):
    """QuantLinear modules of these (k, n, input) with one shared workspace."""
    maker = QuantLinearMaker(quantization_group_size=group, use_act_order=act)
    out = []
    for k, n, (q, z, scales, g_idx) in _checkpoints(gen, mats, group, act):
        qweight, qzeros = _packed(q, z)
        with torch.device("cuda"):
            lin = maker.make_linear(k, n, bias=bias)
        state = {"qweight": qweight, "qzeros": qzeros, "scales": scales, "g_idx": g_idx}
        if bias:
            state["bias"] = _normal(gen, n).to(torch.float16)
        lin = lin.to(torch.device("cuda", torch.cuda.current_device()))
        lin.load_state_dict(state)
        out.append(lin)
    cache = CacheV2(torch.device("cuda", torch.cuda.current_device()))
    maker.post_init(TuningParams(MAX_M=max(rows, 1)), cache)
    cache.init_cache()
    return out


def _weights(gen, mats, group, act, bias=False):
    """The same projections' weights (and biases) in float64, drawn in the same order."""
    out = []
    for k, n, (q, z, scales, g_idx) in _checkpoints(gen, mats, group, act):
        g = g_idx.long()
        w = scales.double()[g] * (q.double() - (z.double() + 1.0)[g])
        out.append((w, _normal(gen, n).to(torch.float16).double() if bias else None))
    return out


def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float16


def _layer(size):
    """A layer's projections (k, n, input): q, k, v, o, gate, up, down."""
    h, i, _ = LAYERS[size]
    return [(h, h, "x"), (h, h, "x"), (h, h, "x"), (h, h, "attention"), (h, i, "mlp"), (h, i, "mlp"),
            (i, h, "gated")]


def _norm_weight(gen, n):
    return (1.0 + 0.1 * _normal(gen, n)).to(torch.float16)


def _rope_tables(positions, hd):
    inv = 1.0 / 10000.0 ** (torch.arange(0, hd, 2, dtype=torch.float64) / hd)
    ang = torch.outer(torch.arange(positions, dtype=torch.float64), inv)
    ang = torch.cat([ang, ang], dim=1)
    return ang.sin().to("cuda", torch.float16), ang.cos().to("cuda", torch.float16)


def _contexts(gen, seqs, ctx):
    """Context lengths of a running batch: the longest is ctx, the others from half of it up."""
    lens = torch.randint(max(1, ctx // 2), ctx + 1, (seqs,), device="cuda", generator=gen)
    lens[0] = ctx
    return lens.to(torch.int32)


def _cacher(gen, seqs, ctx, kv_heads, hd, block):
    """Cache blocks holding earlier tokens, and the block table of each sequence."""
    flags.BLOCK_SIZE = block
    per = (ctx + block - 1) // block
    holder = LayerBlocksHolder.create_contigious_cacher(
        BlockInfo(head_dim=hd, num_key_value_heads=kv_heads), seqs * per, torch.device("cuda"))
    kc, vc = holder.contigious_kv_tenosr
    for t in (kc, vc):
        t.normal_(generator=gen)
    tables = torch.randperm(seqs * per, device="cuda", generator=gen).to(torch.int32)
    return holder, tables.view(seqs, per)


def _slots(gen, rows, block):
    """Slots of one sequence's tokens: consecutive within blocks, the blocks in any order."""
    blocks = (rows + block - 1) // block
    table = torch.randperm(blocks, device="cuda", generator=gen)
    t = torch.arange(rows, device="cuda")
    return table[t // block] * block + t % block, blocks


# ---------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------
def prepare(case, seed):
    return {"kind": case["kind"], **_PREPARE[case["kind"]](case, _gen(seed))}


def _prepare_linear(case, gen):
    lin, = _linears(gen, [(case["k"], case["n"], "x")], case["group"], case["act"], case["rows"],
                    case["bias"])
    return {"lin": lin, "x": _normal(gen, case["rows"], case["k"]).to(_dtype(case))}


def _prepare_finetune(case, gen):
    state = _prepare_linear(case, gen)
    state["x"].requires_grad_(True)
    state["dy"] = (_normal(gen, case["rows"], case["n"])).to(_dtype(case))
    return state


def _captured(call):
    """A graph of call(), captured after one plain run, and what call() returned."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    return {"graph": graph, "out": out}


def _prepare_step(case, gen):
    h, inter, _ = LAYERS[case["size"]]
    rows = case["rows"]
    lins = _linears(gen, _layer(case["size"]) * case["layers"], case["group"], case["act"], rows)
    mats = [lin.q4_matrix for lin in lins]
    x = _normal(gen, rows, h).to(torch.float16)
    xi = _normal(gen, rows, inter).to(torch.float16)

    def call():
        out = []
        for i in range(0, len(mats), 7):
            q, k, v, o, gate, up, down = mats[i:i + 7]
            out += gemm_group(x, [q, k, v]) + [o.matmul(x)]
            out += gemm_group(x, [gate, up]) + [down.matmul(xi)]
        return out

    return {"lins": lins, "inputs": (x, xi), **_captured(call)}


def _stage_inputs(case, gen):
    h, inter, heads = LAYERS[case["size"]]
    seqs, ctx = case["seqs"], case["ctx"]
    x = _normal(gen, seqs, h).to(torch.float16)
    norms = [(_norm_weight(gen, h), _norm_weight(gen, h)) for _ in range(case["layers"])]
    caches = [_cacher(gen, seqs, ctx, heads, 128, case["block"]) for _ in range(case["layers"])]
    lens = _contexts(gen, seqs, ctx)
    return h, inter, heads, x, norms, caches, lens


def _prepare_stage(case, gen):
    lins = _linears(gen, _layer(case["size"]) * case["layers"], case["group"], False, case["seqs"])
    h, inter, heads, x, norms, caches, lens = _stage_inputs(case, gen)
    seqs, ctx, layers = case["seqs"], case["ctx"], case["layers"]
    sin, cos = _rope_tables(ctx, 128)
    pos = lens - 1
    att = PagedAttention(AttentionConfig(h, 128, heads, heads, 1))
    att.workspace(seqs, ctx, x.device)

    def buf(width):
        return torch.empty(seqs, width, dtype=torch.float16, device="cuda")

    rms, q, k, v, x2 = (buf(h) for _ in range(5))
    gate_out, up_out = buf(inter), buf(inter)
    hidden = [buf(h) for _ in range(layers)]
    ctx_lens = torch.empty_like(lens)

    def call():
        xin = x
        for i in range(layers):
            wq, wk, wv, wo, wg, wu, wd = (lin.q4_matrix for lin in lins[7 * i:7 * i + 7])
            holder, tables = caches[i]
            attention_forward_qkv_stage_v2_py(norms[i][0], EPS, wq, wk, wv, rms, q, k, v, None, xin,
                                              0, 0, 0, 1, seqs)
            holder.rope_and_cache(q.view(seqs, heads, 128), k.view(seqs, heads, 128),
                                  v.view(seqs, heads, 128), sin, cos, pos, tables, ctx_lens)
            o = att.forward(q.view(seqs, heads, 128), ctx, ctx_lens, tables, holder)
            decoder_after_stage_v2_py(wo, wg, wu, wd, norms[i][1], EPS, o.view(seqs, h), xin, x2, rms,
                                      gate_out, up_out, hidden[i])
            xin = hidden[i]
        return {"hidden": hidden, "cache": [c.contigious_kv_tenosr for c, _ in caches]}

    keep = (lins, att, norms, caches, x, pos, sin, cos, rms, q, k, v, x2, gate_out, up_out, ctx_lens)
    return {"keep": keep, **_captured(call)}


def _prepare_tail(case, gen):
    h, inter, _ = LAYERS[case["size"]]
    lins = _linears(gen, _layer(case["size"])[3:], case["group"], case["act"], case["rows"])
    rows = case["rows"]

    def buf(width):
        return torch.empty(rows, width, dtype=torch.float16, device="cuda")

    return {"lins": lins, "norm": _norm_weight(gen, h),
            "attn": _normal(gen, rows, h).to(torch.float16), "x": _normal(gen, rows, h).to(torch.float16),
            "bufs": (buf(h), buf(h), buf(inter), buf(inter)), "out": buf(h)}


def _prepare_prompt(case, gen):
    h, _, heads = LAYERS[case["size"]]
    rows = case["rows"]
    lins = _linears(gen, _layer(case["size"])[:3], case["group"], False, rows)
    flags.BLOCK_SIZE = case["block"]
    x = _normal(gen, rows, h).to(torch.float16)
    norm = _norm_weight(gen, h)
    slots, blocks = _slots(gen, rows, case["block"])
    holder = LayerBlocksHolder.create_contigious_cacher(
        BlockInfo(head_dim=128, num_key_value_heads=heads), blocks, torch.device("cuda"))
    for t in holder.contigious_kv_tenosr:
        t.zero_()
    sin, cos = _rope_tables(rows, 128)
    bufs = tuple(torch.empty(rows, h, dtype=torch.float16, device="cuda") for _ in range(4))
    return {"lins": lins, "norm": norm, "x": x, "slots": slots, "holder": holder, "sin": sin,
            "cos": cos, "bufs": bufs, "heads": heads, "rows": rows}


def _prepare_attention(case, gen):
    seqs, ctx, heads, kvh, hd = (case[k] for k in ("seqs", "ctx", "heads", "kv_heads", "head_dim"))
    holder, tables = _cacher(gen, seqs, ctx, kvh, hd, case["block"])
    lens = _contexts(gen, seqs, ctx)
    att = PagedAttention(AttentionConfig(heads * hd, hd, heads, kvh, heads // kvh))
    att.workspace(seqs, ctx, lens.device)
    q = (_normal(gen, seqs, heads, hd) * 1.5).to(torch.float16)
    return {"att": att, "q": q, "ctx": ctx, "lens": lens, "tables": tables, "holder": holder}


def _prepare_swap(case, gen):
    kvh, hd, rows = case["kv_heads"], case["head_dim"], case["rows"]
    flags.BLOCK_SIZE = case["block"]
    slots, blocks = _slots(gen, rows, case["block"])
    holder = LayerBlocksHolder.create_contigious_cacher(
        BlockInfo(head_dim=hd, num_key_value_heads=kvh), blocks, torch.device("cuda"))
    for t in holder.contigious_kv_tenosr:
        t.zero_()
    k, v = (_normal(gen, rows, kvh, hd).to(torch.float16) for _ in range(2))
    return {"holder": holder, "slots": slots, "k": k, "v": v}


_PREPARE = {"linear": _prepare_linear, "finetune": _prepare_finetune, "step": _prepare_step,
            "stage": _prepare_stage, "tail": _prepare_tail, "prompt": _prepare_prompt,
            "attention": _prepare_attention, "swap": _prepare_swap}


# ---------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------
def run(state):
    return _RUN[state["kind"]](state)


def _run_linear(s):
    return s["lin"](s["x"])


def _run_finetune(s):
    y = s["lin"](s["x"])
    dx, = torch.autograd.grad(y, s["x"], s["dy"])
    return y.detach(), dx


def _run_graph(s):
    s["graph"].replay()
    return s["out"]


def _run_tail(s):
    o, gate, up, down = (lin.q4_matrix for lin in s["lins"])
    x2, rms, gate_out, up_out = s["bufs"]
    decoder_after_stage_v2_py(o, gate, up, down, s["norm"], EPS, s["attn"], s["x"], x2, rms, gate_out,
                              up_out, s["out"])
    return x2, s["out"]


def _run_prompt(s):
    q4, k4, v4 = (lin.q4_matrix for lin in s["lins"])
    rms, q, k, v = s["bufs"]
    rows, heads = s["rows"], s["heads"]
    attention_forward_qkv_stage_v2_py(s["norm"], EPS, q4, k4, v4, rms, q, k, v, None, s["x"], 0, 0, 0,
                                      rows, 1)
    attention_forward_rope_stage_v2_py(q, k, s["sin"], s["cos"], rows, 1, heads, heads, 128, 0, None)
    s["holder"].kv_tensor_to_slots_with_convert(k.view(rows, heads, 128), v.view(rows, heads, 128),
                                                s["slots"])
    return (q,) + s["holder"].contigious_kv_tenosr


def _run_attention(s):
    return s["att"].forward(s["q"], s["ctx"], s["lens"], s["tables"], s["holder"])


def _run_swap(s):
    s["holder"].kv_tensor_to_slots_with_convert(s["k"], s["v"], s["slots"])
    k, v = s["holder"].kv_tensor_from_slots_with_convert_with_create(s["slots"])
    return s["holder"].contigious_kv_tenosr + (k, v)


_RUN = {"linear": _run_linear, "finetune": _run_finetune, "step": _run_graph, "stage": _run_graph,
        "tail": _run_tail, "prompt": _run_prompt, "attention": _run_attention, "swap": _run_swap}


# ---------------------------------------------------------------------------
# work, tolerance
# ---------------------------------------------------------------------------
def _gemm(rows, k, n, group, act=False):
    weight = k * n // 2 + (k // group) * (2 * n + n // 2) + (4 * k if act else 0)
    return {"bytes": weight + 2 * rows * (k + n), "flops": 2 * rows * k * n}


def _sum(parts):
    return {"bytes": sum(p["bytes"] for p in parts), "flops": sum(p["flops"] for p in parts)}


def _attention_work(lens, heads, kv_heads, hd):
    return {"bytes": 4 * lens * kv_heads * hd, "flops": 4 * lens * heads * hd}


def work(case):
    kind = case["kind"]
    if kind == "linear":
        return _gemm(case["rows"], case["k"], case["n"], case["group"], case["act"])
    if kind == "finetune":  # the weight is needed in both directions, x and dy once each
        a = _gemm(case["rows"], case["k"], case["n"], case["group"], case["act"])
        return _sum([a, a])
    if kind == "swap":  # k and v read, written to blocks, read from them, written again
        return {"bytes": 4 * 2 * 2 * case["rows"] * case["kv_heads"] * case["head_dim"], "flops": 0}
    if kind == "attention":
        lens = case["seqs"] * case["ctx"] * 3 // 4
        w = _attention_work(lens, case["heads"], case["kv_heads"], case["head_dim"])
        w["bytes"] += 4 * case["seqs"] * case["heads"] * case["head_dim"]
        return w
    mats = _layer(case["size"])
    rows = case["seqs"] if kind == "stage" else case["rows"]
    mats = mats[3:] if kind == "tail" else mats[:3] if kind == "prompt" else mats * case["layers"]
    parts = [_gemm(rows, k, n, case["group"], case.get("act", False)) for k, n, _ in mats]
    if kind == "prompt":  # k and v go to the cache too
        parts.append({"bytes": 4 * rows * LAYERS[case["size"]][0], "flops": 0})
    if kind == "stage":
        heads = LAYERS[case["size"]][2]
        parts += [_attention_work(rows * case["ctx"] * 3 // 4, heads, heads, 128)] * case["layers"]
    return _sum(parts)


def tolerance(case):
    kind = case["kind"]
    if kind == "swap":
        return "exact"
    if kind in ("linear", "finetune") and case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 8e-2}
    if kind in ("linear", "finetune", "step", "attention"):
        return {"rel": 1.2e-3, "max": 1.2e-2}
    # several roundings in a row (norm, products, gate, residuals)
    return {"rel": 4e-3, "max": 4e-2}


# ---------------------------------------------------------------------------
# exact
# ---------------------------------------------------------------------------
def exact(case, seed):
    return _EXACT[case["kind"]](case, _gen(seed))


def _exact_linear(case, gen):
    (w, b), = _weights(gen, [(case["k"], case["n"], "x")], case["group"], case["act"], case["bias"])
    y = _normal(gen, case["rows"], case["k"]).to(_dtype(case)).double() @ w
    return y if b is None else y + b


def _exact_finetune(case, gen):
    (w, b), = _weights(gen, [(case["k"], case["n"], "x")], case["group"], case["act"], case["bias"])
    y = _normal(gen, case["rows"], case["k"]).to(_dtype(case)).double() @ w
    dy = _normal(gen, case["rows"], case["n"]).to(_dtype(case)).double()
    return (y if b is None else y + b), dy @ w.t()


def _exact_step(case, gen):
    h, inter, _ = LAYERS[case["size"]]
    ws = _weights(gen, _layer(case["size"]) * case["layers"], case["group"], case["act"])
    x = _normal(gen, case["rows"], h).to(torch.float16).double()
    xi = _normal(gen, case["rows"], inter).to(torch.float16).double()
    return [(xi if w.shape[0] == inter else x) @ w for w, _ in ws]


def _rms(x, w):
    return x * w.double() * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + EPS)


def _rotate(t, sin, cos):
    """t [tokens, heads, hd], tables [tokens, hd]."""
    half = t.shape[-1] // 2
    s, c = sin.double()[:, None, :], cos.double()[:, None, :]
    return t * c + torch.cat([-t[..., half:], t[..., :half]], dim=-1) * s


def _to_slots(cache, slots, k, v):
    """k, v [tokens, heads, hd] into blocks [.., heads, hd / 8, bs, 8] and [.., heads, hd, bs]."""
    kc, vc = cache
    bs = vc.shape[-1]
    blk, off = slots.long() // bs, slots.long() % bs
    kc[blk, :, :, off, :] = k.reshape(k.shape[0], k.shape[1], -1, 8)
    vc[blk, :, :, off] = v


def _attend(q, cache, tables, lens):
    """q [seqs, heads, hd] against the cached keys and values of each sequence."""
    kc, vc = cache
    kvh, hd = vc.shape[1], vc.shape[2]
    out = torch.empty_like(q)
    for s in range(q.shape[0]):
        n, t = int(lens[s]), tables[s].long()
        k = kc[t].permute(1, 0, 3, 2, 4).reshape(kvh, -1, hd)[:, :n].double()
        v = vc[t].permute(1, 0, 3, 2).reshape(kvh, -1, hd)[:, :n].double()
        qs = q[s].reshape(kvh, -1, hd)
        p = torch.softmax(torch.matmul(qs, k.transpose(1, 2).contiguous()) * hd ** -0.5, dim=-1)
        out[s] = torch.matmul(p, v).reshape(q.shape[1], hd)
    return out


def _exact_tail_of(attn, x, norm, wo, wg, wu, wd):
    x2 = x + attn @ wo
    r = _rms(x2, norm)
    return x2, x2 + (torch.nn.functional.silu(r @ wg) * (r @ wu)) @ wd


def _exact_stage(case, gen):
    ws = [w for w, _ in _weights(gen, _layer(case["size"]) * case["layers"], case["group"], False)]
    h, _, heads, x, norms, caches, lens = _stage_inputs(case, gen)
    sin, cos = _rope_tables(case["ctx"], 128)
    seqs, pos = case["seqs"], (lens - 1).long()
    x, hidden, out_caches = x.double(), [], []
    for i in range(case["layers"]):
        wq, wk, wv, wo, wg, wu, wd = ws[7 * i:7 * i + 7]
        holder, tables = caches[i]
        cache = tuple(t.double() for t in holder.contigious_kv_tenosr)
        r = _rms(x, norms[i][0])
        q = _rotate((r @ wq).view(seqs, heads, 128), sin[pos], cos[pos])
        k = _rotate((r @ wk).view(seqs, heads, 128), sin[pos], cos[pos])
        block = tables.gather(1, (pos // case["block"])[:, None])[:, 0].long()
        _to_slots(cache, block * case["block"] + pos % case["block"], k, (r @ wv).view(seqs, heads, 128))
        o = _attend(q, cache, tables, lens).view(seqs, h)
        _, x = _exact_tail_of(o, x, norms[i][1], wo, wg, wu, wd)
        hidden.append(x)
        out_caches.append(cache)
    return {"hidden": hidden, "cache": out_caches}


def _exact_tail(case, gen):
    h = LAYERS[case["size"]][0]
    wo, wg, wu, wd = (w for w, _ in _weights(gen, _layer(case["size"])[3:], case["group"], case["act"]))
    norm = _norm_weight(gen, h)
    attn = _normal(gen, case["rows"], h).to(torch.float16).double()
    x = _normal(gen, case["rows"], h).to(torch.float16).double()
    return _exact_tail_of(attn, x, norm, wo, wg, wu, wd)


def _exact_prompt(case, gen):
    h, _, heads = LAYERS[case["size"]]
    rows, bs = case["rows"], case["block"]
    wq, wk, wv = (w for w, _ in _weights(gen, _layer(case["size"])[:3], case["group"], False))
    x = _normal(gen, rows, h).to(torch.float16).double()
    r = _rms(x, _norm_weight(gen, h))
    slots, blocks = _slots(gen, rows, bs)
    sin, cos = _rope_tables(rows, 128)
    q = _rotate((r @ wq).view(rows, heads, 128), sin, cos)
    k = _rotate((r @ wk).view(rows, heads, 128), sin, cos)
    cache = (torch.zeros(blocks, heads, 16, bs, 8, dtype=torch.float64, device="cuda"),
             torch.zeros(blocks, heads, 128, bs, dtype=torch.float64, device="cuda"))
    _to_slots(cache, slots, k, (r @ wv).view(rows, heads, 128))
    return (q.view(rows, h),) + cache


def _exact_attention(case, gen):
    s = _prepare_attention(case, gen)
    return _attend(s["q"].double(), s["holder"].contigious_kv_tenosr, s["tables"], s["lens"])


def _exact_swap(case, gen):
    kvh, hd, bs = case["kv_heads"], case["head_dim"], case["block"]
    slots, blocks = _slots(gen, case["rows"], bs)
    k, v = (_normal(gen, case["rows"], kvh, hd).to(torch.float16).double() for _ in range(2))
    cache = (torch.zeros(blocks, kvh, hd // 8, bs, 8, dtype=torch.float64, device="cuda"),
             torch.zeros(blocks, kvh, hd, bs, dtype=torch.float64, device="cuda"))
    _to_slots(cache, slots, k, v)
    return cache + (k, v)


_EXACT = {"linear": _exact_linear, "finetune": _exact_finetune, "step": _exact_step,
          "stage": _exact_stage, "tail": _exact_tail, "prompt": _exact_prompt,
          "attention": _exact_attention, "swap": _exact_swap}
