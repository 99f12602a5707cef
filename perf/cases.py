"""The work that a program has this library do, as cases that can be timed and checked: one TP=8 rank's share of a
GLM-5.3 MoE layer (hidden size 6144, 256 columns of every expert's intermediate, 256 experts, 8 a token) and the EXL3
linears beside it, each through the public entry points of ea_exl3.

    listed()               the cases
    draw(rng)              one more case of the ranges they stand for
    prepare(case, seed)    weights, inputs and scratch on the GPU
    run(state)             one pass; its outputs
    work(case)             the bytes and operations a pass cannot do without
    tolerance(case)        how far two correct implementations may differ
    exact(case, seed)      the same outputs in 64-bit arithmetic, without the library
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "expertatlas-glm5.3_amd"))  # the package of the tree that is run

DIMS, EXPERTS, SLOTS, SCALE = 6144, 256, 8, 2.5
MCG, MUL1 = 1, 2  # codebooks
DTYPE = {"f16": 0, "bf16": 1, "f32": 2}
TORCH = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


# ---- the cases ------------------------------------------------------------------------------------------------------

def listed():
    return [
        # One quantized projection of a decode step: the smallest call, where latency is all there is.
        dict(name="linear_1row", kind="linear", rows=1, k=6144, n=2048, jobs=1, k2=8, cb=MCG, x="bf16", y="f32"),
        # The same projection over the widest decode window (and the tail of a prompt).
        dict(name="linear_128rows", kind="linear", rows=128, k=6144, n=2048, jobs=1, k2=8, cb=MCG, x="bf16", y="f32"),
        # The shared expert of a speculative window at the checkpoints' own 5-bit mul1: gate|up in one call, SwiGLU, down.
        dict(name="shared_mlp_12rows", kind="mlp", rows=12, width=256, k2=10, cb=MUL1),
        # The same over a wide window.
        dict(name="shared_mlp_70rows", kind="mlp", rows=70, width=256, k2=10, cb=MUL1),
        # One token of a decode step through eight resident layers (routing, routed experts, shared expert, sum).
        dict(name="decode_1row_8layers", kind="decode", rows=1, layers=8, widths="8", router=False, x="bf16"),
        # A few sequences, or a short speculative window, from the router's own GEMM on; experts at 3 and 4 bits.
        dict(name="decode_5rows_router", kind="decode", rows=5, layers=1, widths="6x0.7 8x0.3", router=True, x="bf16"),
        # The most rows the decode layer takes: about a hundred distinct experts.
        dict(name="decode_16rows", kind="decode", rows=16, layers=1, widths="6x0.7 8x0.3", router=False, x="f16"),
        # A decode window of an odd size, as the engine issues one: top-8, routed experts, shared expert, sum.
        dict(name="window_37rows", kind="window", rows=37, widths="6x0.7 8x0.3", x="bf16"),
        # The widest decode window.
        dict(name="window_128rows", kind="window", rows=128, widths="6x0.7 8x0.3", x="bf16"),
        # A short prompt, summed in slot order (the same bits on every run).
        dict(name="prefill_512rows", kind="prefill", rows=512, widths="8", planes=True, round=False, x="bf16"),
        # A long prompt in the default mode (no pair plane).
        dict(name="prefill_2048rows", kind="prefill", rows=2048, widths="8", planes=False, round=True, x="bf16"),
        # A prompt of an odd size on a wider bank: most experts at 5 bits, some at 6 and 8.
        dict(name="prefill_777rows_wide", kind="prefill", rows=777, widths="10x0.6 12x0.3 16x0.1", planes=True, round=True,
             x="bf16"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "mlp", "decode", "decode", "window", "prefill", "prefill"])
    x = rng.choice(["bf16", "bf16", "f16"])
    if kind == "linear":
        k2, cb = rng.choice([(8, MCG), (6, MCG), (4, MCG), (10, MUL1), (8, MUL1), (12, MUL1)])
        return dict(kind=kind, rows=_log_int(rng, 1, 128), k=128 * _log_int(rng, 4, 48), n=128 * _log_int(rng, 1, 48),
                    jobs=rng.choice([1, 1, 2, 3]), k2=k2, cb=cb, x=x, y=rng.choice(["f32", "bf16", "f16"]))
    if kind == "mlp":
        k2, cb = rng.choice([(10, MUL1), (8, MCG), (6, MCG)])
        return dict(kind=kind, rows=_log_int(rng, 1, 128), width=rng.choice([128, 256]), k2=k2, cb=cb)
    widths = rng.choice(["8", "6", "6x0.7 8x0.3", "4x0.3 6x0.5 8x0.2", "10"])
    if kind == "decode":
        return dict(kind=kind, rows=_log_int(rng, 1, 16), layers=rng.choice([1, 1, 3]), widths=widths, router=rng.random() < 0.5, x=x)
    if kind == "window":
        return dict(kind=kind, rows=_log_int(rng, 17, 128), widths=widths, x=x)
    planes = rng.random() < 0.5
    if rng.random() < 0.3:
        widths = rng.choice(["12", "10x0.6 12x0.3 16x0.1"])
    return dict(kind=kind, rows=_log_int(rng, 129, 2048), widths=widths, planes=planes, round=rng.random() < 0.7, x=x)


# ---- weights and inputs ---------------------------------------------------------------------------------------------

def _width_table(text):
    """K2 (twice the bits a weight) of every expert: one width, or 'K2xshare' parts spread over the experts."""
    parts = [p.split("x") for p in text.split()]
    if len(parts) == 1:
        return np.full(EXPERTS, int(parts[0][0]), np.int32)
    table = []
    for k2, share in parts:
        table += [int(k2)] * int(round(EXPERTS * float(share)))
    table = (table + [int(parts[0][0])] * EXPERTS)[:EXPERTS]
    return np.random.default_rng(77).permutation(np.array(table, np.int32))


def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + what) & 0x7FFFFFFF)
    return g


def _normal(shape, gen, dtype):
    return torch.randn(shape, device="cuda", generator=gen).to(TORCH[dtype])


def _popularity(gen):
    """log-probabilities of a Zipf(1.1) popularity over a random ranking of the experts (prompts route unevenly)."""
    p = -1.1 * torch.log(torch.arange(1, EXPERTS + 1, device="cuda", dtype=torch.float32))
    return p[torch.randperm(EXPERTS, device="cuda", generator=gen)]


def _picks(seed, rows):
    """A prompt's picks int32 [rows, 8] (Zipf(1.1), without replacement) and weights fp32 [rows, 8] that sum to 2.5."""
    gen = _gen(seed, 21)
    u = torch.rand((rows, EXPERTS), device="cuda", generator=gen).clamp_min(1e-20)
    pick = torch.topk(_popularity(gen) - torch.log(-torch.log(u)), SLOTS, dim=1).indices.to(torch.int32).contiguous()
    w = torch.rand((rows, SLOTS), device="cuda", generator=gen) * 0.95 + 0.05
    return pick, (w / w.sum(1, keepdim=True) * SCALE).contiguous()


class _State:
    """What one case keeps: device, module handles and tensors, by name."""

    def __init__(self, case):
        self.case = case


def _linears(case, seed):
    from ea_exl3 import resident

    gen = _gen(seed, 31)
    return [resident.DeviceLinear(gen, case["k"], case["n"], case["k2"], case["cb"]) for _ in range(case["jobs"])]


def _shared(seed, width, k2, cb):
    from ea_exl3 import resident

    return resident.DeviceShared((int(seed) * 7919 + 5) & 0x7FFFFFFF, DIMS, width, k2, cb)


def _routed(seed, layer, widths):
    from ea_exl3 import resident

    return resident.DeviceRouted((int(seed) * 104729 + layer) & 0x7FFFFFFF, EXPERTS, DIMS, 256, k2=_width_table(widths))


def _decode_inputs(case, seed):
    """x [rows, D], router weight (bf16) or logits (fp32) and bias of every layer."""
    gen, rows = _gen(seed, 41), case["rows"]
    x = _normal((rows, DIMS), gen, case["x"])
    bias = 0.1 * torch.randn(EXPERTS, device="cuda", generator=gen)
    layers = case.get("layers", 1)
    if case.get("router"):
        return x, bias, [(0.02 * torch.randn((EXPERTS, DIMS), device="cuda", generator=gen)).to(torch.bfloat16)
                         for _ in range(layers)]
    return x, bias, [torch.randn((rows, EXPERTS), device="cuda", generator=gen) for _ in range(layers)]


def prepare(case, seed):
    from ea_exl3 import device, linear, moe, prompt_experts

    device.init(0)
    s, kind, R = _State(case), case["kind"], case["rows"]
    if kind == "linear":
        s.lins = _linears(case, seed)
        s.x = _normal((R, case["k"]), _gen(seed, 11), case["x"])
        s.y = [torch.zeros((R, case["n"]), dtype=TORCH[case["y"]], device="cuda") for _ in s.lins]
        s.scratch = linear.Scratch(R, case["k"], s.lins[0].sk * R * case["n"])
    elif kind == "mlp":
        s.shared = _shared(seed, case["width"], case["k2"], case["cb"])
        s.x = _normal((R, DIMS), _gen(seed, 11), "bf16")
        _mlp_buffers(s, R, case["width"])
    elif kind == "decode":
        s.x, s.bias, s.route = _decode_inputs(case, seed)
        s.layers = [_routed(seed, l, case["widths"]) for l in range(case["layers"])]
        sh = [_shared(seed + l, 256, 8, MCG) for l in range(case["layers"])]
        s.keep, s.shared = sh, [(h.gate.c, h.up.c, h.down.c) for h in sh]
        s.logits = [torch.zeros((R, EXPERTS), device="cuda") for _ in s.layers] if case["router"] else s.route
        s.pick = [torch.zeros((R, SLOTS), dtype=torch.int32, device="cuda") for _ in s.layers]
        s.wts = [torch.zeros((R, SLOTS), device="cuda") for _ in s.layers]
        s.out = [torch.zeros((R, DIMS), device="cuda") for _ in s.layers]
        s.scratch = moe.Scratch(s.layers[0], R, SLOTS)
    elif kind == "window":
        s.x, s.bias, logits = _decode_inputs(case, seed)
        s.logits = logits[0]
        s.ex = _routed(seed, 0, case["widths"])
        s.shared = _shared(seed, 256, 8, MCG)
        s.pick = torch.zeros((R, SLOTS), dtype=torch.int32, device="cuda")
        s.wts = torch.zeros((R, SLOTS), device="cuda")
        s.out = torch.zeros((R, DIMS), device="cuda")
        s.scratch = moe.Scratch(s.ex, R, SLOTS)
        _mlp_buffers(s, R, 256)
    else:
        s.ex = _routed(seed, 0, case["widths"])
        s.x = _normal((R, DIMS), _gen(seed, 11), case["x"])
        s.pick, s.wts = _picks(seed, R)
        s.out = torch.zeros((R, DIMS), device="cuda")
        s.scratch = prompt_experts.Scratch(s.ex, R, SLOTS, planes=case["planes"])
    return s


def _mlp_buffers(s, R, width):
    from ea_exl3 import linear

    s.g, s.u, s.act = (torch.zeros((R, width), dtype=torch.bfloat16, device="cuda") for _ in range(3))
    s.sy = torch.zeros((R, DIMS), device="cuda")
    s.lscratch = linear.Scratch(R, DIMS, max(s.shared.gate.sk * width, s.shared.down.sk * DIMS) * R)


# ---- one pass -------------------------------------------------------------------------------------------------------

def _mlp(s, stream, R, width, x_dtype):
    """The shared expert as forward.mlp issues it: gate|up, SwiGLU, down."""
    from ea_exl3 import linear, ops

    linear.call(stream, s.lscratch, [s.shared.gate, s.shared.up], s.x.data_ptr(), x_dtype, R,
                [s.g.data_ptr(), s.u.data_ptr()], [1, 1])
    ops.swiglu2(stream, s.g.data_ptr(), s.u.data_ptr(), s.act.data_ptr(), R, width)
    linear.call(stream, s.lscratch, [s.shared.down], s.act.data_ptr(), 1, R, [s.sy.data_ptr()], [2])


def run(s):
    from ea_exl3 import device, linear, moe, ops, prompt_experts

    case, kind, R, q = s.case, s.case["kind"], s.case["rows"], device.stream()
    if kind == "linear":
        linear.call(q, s.scratch, s.lins, s.x.data_ptr(), DTYPE[case["x"]], R, [y.data_ptr() for y in s.y],
                    [DTYPE[case["y"]]] * len(s.lins))
        return s.y
    if kind == "mlp":
        _mlp(s, q, R, case["width"], 1)
        return [s.g, s.u, s.act, s.sy]
    if kind == "decode":
        for l, ex in enumerate(s.layers):
            args = (s.bias.data_ptr(), SCALE, s.pick[l].data_ptr(), s.wts[l].data_ptr(), ex, s.shared[l], s.scratch,
                    s.out[l].data_ptr(), R, DTYPE[case["x"]])
            if case["router"]:
                moe.ffn_decode_router(q, s.x.data_ptr(), DIMS, s.route[l].data_ptr(), s.logits[l].data_ptr(), *args)
            else:
                moe.ffn_decode(q, s.x.data_ptr(), DIMS, s.logits[l].data_ptr(), *args)
        return {"out": s.out, "pick": s.pick, "wts": s.wts, "logits": s.logits}
    if kind == "window":
        ops.topk(q, s.logits.data_ptr(), s.bias.data_ptr(), s.pick.data_ptr(), s.wts.data_ptr(), R, SCALE)
        moe.routed(q, s.x.data_ptr(), DIMS, s.pick.data_ptr(), s.wts.data_ptr(), s.ex, s.scratch, s.out.data_ptr(), R,
                   DTYPE[case["x"]])
        _mlp(s, q, R, 256, DTYPE[case["x"]])
        ops.add_f32(q, s.out.data_ptr(), s.sy.data_ptr(), R * DIMS)
        return {"out": s.out, "pick": s.pick, "wts": s.wts}
    prompt_experts.run(q, s.x.data_ptr(), DIMS, s.pick.data_ptr(), s.wts.data_ptr(), s.ex, s.scratch, s.out.data_ptr(),
                       R, do_round=case["round"], x_dtype=DTYPE[case["x"]])
    return s.out


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

def _touched(rows, zipf):
    """The experts that `rows` rows are expected to touch."""
    if not zipf:
        return EXPERTS * (1 - (1 - SLOTS / EXPERTS) ** rows)
    rng = np.random.default_rng(9)
    p = -1.1 * np.log(np.arange(1, EXPERTS + 1))
    g = p - np.log(-np.log(rng.uniform(1e-20, 1, (rows, EXPERTS))))
    return float(len(np.unique(np.argpartition(-g, SLOTS, axis=1)[:, :SLOTS])))


def _matrix_bytes(k, n, k2):
    return k * n * k2 // 16 + 2 * (k + n)


def work(case):
    kind, R = case["kind"], case["rows"]
    size = {"f16": 2, "bf16": 2, "f32": 4}
    if kind == "linear":
        k, n, j = case["k"], case["n"], case["jobs"]
        return {"bytes": j * _matrix_bytes(k, n, case["k2"]) + R * k * 2 + j * R * n * size[case["y"]],
                "flops": 2 * j * R * k * n}
    if kind == "mlp":
        w = case["width"]
        return {"bytes": 3 * _matrix_bytes(DIMS, w, case["k2"]) + R * (DIMS * 6 + 3 * w * 2),
                "flops": 6 * R * DIMS * w}
    expert = 3 * _matrix_bytes(DIMS, 256, float(np.mean(_width_table(case["widths"]))))
    touched = _touched(R, kind == "prefill")
    flops, moved = 6 * R * SLOTS * DIMS * 256, touched * expert + R * (DIMS * 6 + SLOTS * 8)
    if kind != "prefill":  # the shared expert, the logits and the bias
        flops += 6 * R * DIMS * 256
        moved += 3 * _matrix_bytes(DIMS, 256, 8) + R * EXPERTS * 4
        if case.get("router"):
            flops += 2 * R * DIMS * EXPERTS
            moved += EXPERTS * DIMS * 2
    n = case.get("layers", 1)
    return {"bytes": int(n * moved), "flops": int(n * flops)}


def tolerance(case):
    # fp16 products summed in fp32: another order of sums moves an output by about 1e-6 of its size, and where a rounding
    # to 16 bits follows (the rotated inputs, gate, up, the down inputs, 16-bit outputs) some values then round the other
    # way. Atomic sums in another order were measured 1e-5 apart (bf16-rounded outputs, 2048 rows).
    if case["kind"] == "linear" and case["y"] == "f32":
        return {"rel": 1e-4}
    if case["kind"] in ("linear", "mlp") or case.get("round"):
        return {"rel": 1e-3}
    return {"rel": 5e-4, "differ": 0.0}


# ---- the same in 64-bit arithmetic ----------------------------------------------------------------------------------

def _codebook(cb):
    """The value of each of the 65,536 states, as the format defines it in fp16."""
    s = np.arange(65536, dtype=np.uint64)
    half = lambda v: (v & np.uint64(0xFFFF)).astype(np.uint16).view(np.float16)  # noqa: E731
    if cb == MUL1:
        v = (s * np.uint64(0x83DCD12D)) & np.uint64(0xFFFFFFFF)
        total = sum(((v >> np.uint64(8 * i)) & np.uint64(255)) for i in range(4))
        # (1024 + byte sum) * c1 + c0, rounded to fp16 once
        c1, c0 = (float(np.array([b], np.uint16).view(np.float16)[0]) for b in (0x1EEE, 0xC931))
        return ((1024.0 + total.astype(np.float64)) * c1 + c0).astype(np.float16).astype(np.float64)
    v = (s * np.uint64(0xCBAC1FED)) & np.uint64(0xFFFFFFFF)
    v = (v & np.uint64(0x8FFF8FFF)) ^ np.uint64(0x3B603B60)
    return (half(v) + half(v >> np.uint64(16))).astype(np.float64)


_TABLES = {}


def _tables(k2, cb):
    """(first word, second word, shift) of each of a tile's 256 values, its place in the tile, and the codebook."""
    if (k2, cb) not in _TABLES:
        p = np.arange(256)
        end = ((p + 1) * k2 - ((p + 1) & 1 if k2 & 1 else 0)) // 2  # value p's state ends at this bit of the stream
        start = (end - 16) % (128 * k2)
        L, j = p >> 3, p & 7
        row, col = 2 * (L & 3) + (j & 1) + 8 * ((j >> 1) & 1), (L >> 2) + 8 * (j >> 2)
        place = np.empty(256, np.int64)
        place[row * 16 + col] = p  # value of (row, col)
        to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
        w0 = (start >> 5)[place]
        _TABLES[(k2, cb)] = (to(w0), to((w0 + 1) % (4 * k2)), to((32 - (start & 31))[place]), to(_codebook(cb)))
    return _TABLES[(k2, cb)]


def _tiles(words, k2, cb):
    """Tiles [T, 4 k2] (32-bit words) -> their values [T, 16, 16] in float64."""
    w0, w1, shift, book = _tables(k2, cb)
    w = words.to(torch.int64) & 0xFFFFFFFF
    state = (((w[:, w0] << 16) | (w[:, w1] >> 16)) >> shift) & 0xFFFF
    return book[state].reshape(-1, 16, 16)


def _hadamard():
    h = torch.ones((1, 1), dtype=torch.float64, device="cuda")
    while h.shape[0] < 128:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(128.0)


def _rotate(v):
    """The orthonormal 128-point Walsh-Hadamard transform of every 128 columns."""
    return (v.reshape(-1, 128) @ _hadamard()).reshape(v.shape)


def _project(x, w, suh, svh):
    """x through one quantized matrix w [K, N]: the input and output rotations and scales around the product."""
    return _rotate(_rotate(x * suh.double()) @ w) * svh.double()


def _linear_matrix(l):
    """A linear's words [N / 128, K / 16, 8, 4 k2] as [K, N]."""
    t = _tiles(l.words.reshape(-1, 4 * l.k2), l.k2, l.cb).reshape(l.n // 128, l.k // 16, 8, 16, 16)
    return t.permute(1, 3, 0, 2, 4).reshape(l.k, l.n)


def _expert_matrix(ex, m, e):
    """Expert e's gate (0), up (1) or down (2) matrix [K, N]."""
    K, N = ((ex.dims, ex.width), (ex.dims, ex.width), (ex.width, ex.dims))[m]
    k2, at = int(ex.k2_host[e]), int(ex.offs[m][e]) // 4
    words = ex.slabs[m][at:at + int(ex.bytes[m][e]) // 4].reshape(-1, 4 * k2)
    return _tiles(words, k2, ex.cb).reshape(K // 16, N // 16, 16, 16).permute(0, 2, 1, 3).reshape(K, N)


def _silu(v):
    return v * torch.sigmoid(v)


def _experts(ex, x, pick, wts):
    out = torch.zeros((x.shape[0], ex.dims), dtype=torch.float64, device="cuda")
    sc = lambda t, n: t.reshape(ex.count, n)  # noqa: E731
    for e in torch.unique(pick).tolist():
        rows, slot = torch.nonzero(pick == e, as_tuple=True)
        v = x[rows]
        g = _project(v, _expert_matrix(ex, 0, e), sc(ex.suh_g, ex.dims)[e], sc(ex.svh_g, ex.width)[e])
        u = _project(v, _expert_matrix(ex, 1, e), sc(ex.suh_u, ex.dims)[e], sc(ex.svh_u, ex.width)[e])
        y = _project(_silu(g) * u, _expert_matrix(ex, 2, e), sc(ex.suh_d, ex.width)[e], sc(ex.svh_d, ex.dims)[e])
        out.index_add_(0, rows, y * wts[rows, slot].double()[:, None])
    return out


def _exact_mlp(sh, x):
    g, u = (_project(x, _linear_matrix(l), l.suh, l.svh) for l in (sh.gate, sh.up))
    act = _silu(g) * u
    return g, u, act, _project(act, _linear_matrix(sh.down), sh.down.suh, sh.down.svh)


def _exact_route(logits, bias):
    sig = torch.sigmoid(logits)
    pick = torch.topk(sig + bias.double(), SLOTS, dim=1).indices
    w = torch.gather(sig, 1, pick)
    return pick, w / (w.sum(1, keepdim=True) + 1e-20) * SCALE


def exact(case, seed):
    kind, R = case["kind"], case["rows"]
    if kind == "linear":
        x = _normal((R, case["k"]), _gen(seed, 11), case["x"]).double()
        return [_project(x, _linear_matrix(l), l.suh, l.svh) for l in _linears(case, seed)]
    if kind == "mlp":
        return list(_exact_mlp(_shared(seed, case["width"], case["k2"], case["cb"]),
                               _normal((R, DIMS), _gen(seed, 11), "bf16").double()))
    if kind == "prefill":
        x = _normal((R, DIMS), _gen(seed, 11), case["x"]).double()
        pick, wts = _picks(seed, R)
        return _experts(_routed(seed, 0, case["widths"]), x, pick.long(), wts)
    x, bias, route = _decode_inputs(case, seed)
    x = x.double()
    outs, picks, wtss, logitss = [], [], [], []
    for l in range(case.get("layers", 1)):
        logits = x @ route[l].double().t() if case.get("router") else route[l].double()
        pick, wts = _exact_route(logits, bias)
        out = _experts(_routed(seed, l, case["widths"]), x, pick, wts)
        outs.append(out + _exact_mlp(_shared(seed + l, 256, 8, MCG), x)[3])
        picks.append(pick.to(torch.int32))
        wtss.append(wts)
        logitss.append(logits)
    if kind == "window":
        return {"out": outs[0], "pick": picks[0], "wts": wtss[0]}
    return {"out": outs, "pick": picks, "wts": wtss, "logits": logitss}
