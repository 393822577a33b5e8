"""The work a program built on this library has it do, as cases that can be timed.

    listed()             the cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what the program holds before the call: operands on the GPU, weights, tables, handles
    run(state)           one pass through the public entry points; returns its outputs
    work(case)           bytes and operations the pass cannot do without
    tolerance(case)      how far another correct implementation of the same precision may be off

Six kinds of case:

    plain    standalone attention as `attention_fast.run` (operands in host memory) or
             `mattn.Context.runOnHandles` (resident f32 rows) serve it
    klein    fused QK-norm + rope + attention of `blocks` Klein blocks in one batch, each block with
             its own operands and norm weights (text rows under the added-stream weights)
    zimage   the same for the Z-Image form (three-axis rope from positions, no text weights)
    segment  the attention segment of `layers` Z-Image layers in one batch
    wide     the one-head, 512-wide attention of the VAE mid-block
    project  the projections either side of attention: of a Klein double block (two streams, q/k/v
             and output) or of a single block (q/k/v, and the output projection of width 4 x hidden)

A batch is opened, filled and ended (which waits for it) inside run(), as a denoising step does.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from zdraw_amd import hip, host
from zdraw_amd import workloads as wl

D = wl.HEAD_DIM
WIDE = 512
KLEIN_TXT = 512         # text slots of a Klein sequence
KLEIN_THETA = 10000.0
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
ACT = {"f32": hip.F32, "bf16": hip.BF16, "f16": hip.F16}
WEIGHT = {"f32": hip.W_F32, "bf16": hip.W_BF16, "f16": hip.W_F16}
SIZE = {"f32": 4, "bf16": 2, "f16": 2}

_ctx = None


def context():
    """One context per process: device, queue, pipelines."""
    global _ctx
    if _ctx is None:
        torch.zeros(1, device="cuda")  # torch's runtime first: both then use the same device context
        _ctx = host.Context.init()
    return _ctx


# ------------------------------------------------------------------------ cases
def klein(name, grid, *, batch=1, ref=(0, 0), txt=KLEIN_TXT, heads=24, blocks=1, act="bf16", out="bf16", bound=True,
          masked=False, staging="bf16", concat=False, site="prepass"):
    return {"name": name, "kind": "klein", "grid_h": grid[0], "grid_w": grid[1], "ref_h": ref[0], "ref_w": ref[1], "txt": txt,
            "batch": batch, "heads": heads, "blocks": blocks, "act": act, "out": out, "bound": bound, "masked": masked,
            "staging": staging, "concat": concat, "site": site}


def listed():
    return [
        # the reference's plumbing configuration: one small attention on host arrays; all latency
        {"name": "plain_256_host", "kind": "plain", "tokens": 256, "heads": 2, "valid": 0, "host": True},
        # a 256 x 256 preview: the attention of the five double-stream blocks of one step
        klein("klein_256", (16, 16), blocks=5),
        # four seeds of a 512 x 512 render side by side
        klein("klein_512_x4", (32, 32), batch=4, blocks=2),
        # a 1024 x 1024 render, the headline configuration
        klein("klein_1024", (64, 64), blocks=2),
        # an 832 x 1216 portrait with a short prompt, in the reference's resident form: f32 activations,
        # padded text keys masked, no score bound from the caller, half-precision concat operand out
        klein("klein_portrait_resident", (76, 52), act="f32", out="f16", bound=False, masked=True, concat=True, blocks=2),
        # edit mode: target and reference image, two prompts of different length
        klein("klein_edit_ragged", (64, 64), ref=(64, 64), batch=2, masked=True, blocks=2),
        # the Z-Image layer at 1024 x 1024, 16-bit activations
        {"name": "zimage_1024_segment", "kind": "segment", "grid_h": 64, "grid_w": 64, "cap": 512, "heads": 30, "layers": 2,
         "act": "bf16", "weight": "bf16", "norm": "f32"},
        # the same layer at 512 x 768 with a short caption, as the reference keeps it: f32 activations, f16 weights
        {"name": "zimage_512x768_segment_f32", "kind": "segment", "grid_h": 48, "grid_w": 32, "cap": 77, "heads": 30, "layers": 2,
         "act": "f32", "weight": "f16", "norm": "bf16"},
        # the VAE mid-block of a 1024 x 1024 render
        {"name": "wide_16384", "kind": "wide", "tokens": 16384},
        # the reference's own test length for that kernel: no power of two, half a tile left over
        {"name": "wide_6208", "kind": "wide", "tokens": 6208},
        # both streams' projections of a double block at 512 x 512, f32 activations
        {"name": "project_double_512", "kind": "project", "block": "double", "txt": 512, "img": 1024, "hidden": 3072, "act": "f32",
         "out": "f32", "weight": "bf16"},
        # a single block's projections at 1024 x 1024, 16-bit activations
        {"name": "project_single_1024", "kind": "project", "block": "single", "txt": 512, "img": 4096, "hidden": 3072, "act": "bf16",
         "out": "bf16", "weight": "bf16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, most_tokens):
    """An image of 128 to 1024-odd pixels a side in 16-pixel patches, any aspect up to 1 : 2.5."""
    while True:
        h, w = _log(rng, 8, 96), _log(rng, 8, 96)
        if h <= 2.5 * w and w <= 2.5 * h and h * w <= most_tokens:
            return h, w


def draw(rng):
    kind = rng.choice(("plain", "klein", "klein", "klein", "zimage", "segment", "segment", "wide", "project", "project"))
    if kind == "plain":
        host_side = rng.random() < 0.4
        tokens = _log(rng, 16, 1536 if host_side else 4224)
        return {"kind": "plain", "tokens": tokens, "heads": rng.choice((1, 2, 3, 8, 24, 30)),
                "valid": rng.randint(1, tokens) if rng.random() < 0.25 else 0, "host": host_side}
    if kind == "klein":
        batch = rng.choice((1, 1, 1, 2, 3, 4))
        gh, gw = _grid(rng, 4608 // (1 if batch < 3 else 2))
        c = klein("", (gh, gw), batch=batch, txt=KLEIN_TXT if rng.random() < 0.7 else _log(rng, 16, KLEIN_TXT),
                  heads=24 if rng.random() < 0.7 else rng.choice((2, 5, 16, 32)), act=rng.choice(("bf16", "bf16", "f32", "f16")),
                  bound=rng.random() < 0.6, masked=rng.random() < 0.4, blocks=2)
        del c["name"]
        if batch < 3 and rng.random() < 0.25 and gh * gw <= 4096:
            c["ref_h"], c["ref_w"] = gh, gw
        c["out"] = rng.choice(("bf16", "bf16", "f16", "f32"))
        c["concat"] = c["out"] != "f32" and rng.random() < 0.3
        if rng.random() < 0.15:
            c["staging"] = "f16"
        elif c["act"] != "f16" and rng.random() < 0.1:
            c["site"] = "tile"
        return c
    if kind == "zimage":
        gh, gw = _grid(rng, 6144)
        return {"kind": "zimage", "grid_h": gh, "grid_w": gw, "cap": _log(rng, 16, 512), "heads": rng.choice((30, 30, 30, 4, 16)),
                "blocks": 2, "act": rng.choice(("bf16", "bf16", "f32")), "out": rng.choice(("bf16", "f32")), "bound": rng.random() < 0.6}
    if kind == "segment":
        gh, gw = _grid(rng, 4608)
        act, weight = rng.choice((("bf16", "bf16"), ("bf16", "bf16"), ("f32", "bf16"), ("f32", "f16")))
        return {"kind": "segment", "grid_h": gh, "grid_w": gw, "cap": _log(rng, 16, 512), "heads": rng.choice((30, 30, 30, 8, 20)),
                "layers": rng.choice((1, 2)), "act": act, "weight": weight, "norm": rng.choice(("f32", "bf16", "f16"))}
    if kind == "wide":
        return {"kind": "wide", "tokens": 64 * _log(rng, 4, 288)}
    act, out, weight = rng.choice((("bf16", "bf16", "bf16"), ("f32", "f32", "bf16"), ("f32", "bf16", "bf16"), ("f16", "f32", "f16"), ("f32", "f32", "f16")))
    return {"kind": "project", "block": rng.choice(("double", "single")), "txt": KLEIN_TXT if rng.random() < 0.6 else _log(rng, 16, KLEIN_TXT),
            "img": _log(rng, 64, 4608), "hidden": rng.choice((3072, 3072, 3840, 1024, 2568)), "act": act, "out": out, "weight": weight}


# ---------------------------------------------------------------------- operands
class Resident:
    """A tensor in GPU memory that the library sees through a wrapping handle."""

    def __init__(self, t):
        self.t = t.contiguous()
        self.handle = hip.lib().zdraw_hip_wrap_device_memory(context().device, self.t.data_ptr(), self.t.numel() * self.t.element_size())
        if not self.handle:
            raise RuntimeError(hip.last_error())

    def __del__(self):
        if getattr(self, "handle", None):
            hip.lib().zdraw_hip_release_buffer(self.handle)
            self.handle = None


def _check(rc, what):
    if rc != 0:
        raise RuntimeError(f"{what} rc={rc}: {hip.last_error()}")


def _randn(g, shape, dtype, scale=1.0):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * scale).to(TORCH[dtype])


def _norm_weight(rng):
    """Learned QK-norm weights: around one."""
    return (1.0 + 0.1 * rng.standard_normal(D)).astype(np.float32)


def _typed(a, dtype):
    if dtype == "bf16":
        return host.f32_to_bf16_bits(a)
    return a.astype(np.float16 if dtype == "f16" else np.float32)


def _tokens(case):
    if case["kind"] == "klein":
        return case["txt"] + case["grid_h"] * case["grid_w"] + case["ref_h"] * case["ref_w"]
    pad = lambda n: -(-n // 32) * 32  # sequences are padded to whole blocks of 32 (zimage/zseq.zig:23-34)
    return pad(case["grid_h"] * case["grid_w"]) + pad(case["cap"])


def _text_lens(case):
    """Real text lengths of the segments when the padded text keys are masked."""
    return [max(1, case["txt"] * (15 + 44 * (b % 2)) // 100) for b in range(case["batch"])]


def _strides(dst, tokens, row, batch):
    dst[0] = tokens * row if batch > 1 else 0
    dst[1] = row
    dst[2] = D


def _fused_block(case, g, rng, tables):
    """Operands, weights and argument structs of one block of the fused entry."""
    ctx, tokens, heads = context(), _tokens(case), case["heads"]
    batch, hidden = case.get("batch", 1), case["heads"] * D
    b = {"q": Resident(_randn(g, (batch, tokens, heads, D), case["act"])), "k": Resident(_randn(g, (batch, tokens, heads, D), case["act"])),
         "v": Resident(_randn(g, (batch, tokens, heads, D), case["act"]))}
    pitch = 4 * hidden if case.get("concat") else hidden  # the concat operand of a single block: attention output beside the MLP's
    b["o"] = Resident(torch.zeros((batch, tokens, pitch), device="cuda", dtype=TORCH[case["out"]]))
    x, ops = hip.AttnExt(), hip.QkOperands()
    for s in (x.q_stride, x.k_stride, x.v_stride):
        _strides(s, tokens, hidden, batch)
    _strides(x.out_stride, tokens, pitch, batch)
    x.batch, x.in_dtype, x.out_dtype = batch, ACT[case["act"]], ACT[case["out"]]
    x.k_site = hip.K_IN_TILE_LOAD if case.get("site") == "tile" else hip.K_PREPASS
    x.staging = ACT[case.get("staging", "bf16")]
    w = [_norm_weight(rng) for _ in range(4 if case["kind"] == "klein" else 2)]
    wb = [ctx.buffer(a) for a in w]
    ops.q_weight, ops.k_weight = wb[0].handle, wb[1].handle
    if case["kind"] == "klein":
        x.qk_mode, x.eps, x.txt_rows = hip.QK_KLEIN, wl.KLEIN_EPS, case["txt"]
        ops.q_weight_txt, ops.k_weight_txt = wb[2].handle, wb[3].handle
        ops.rope_cos, ops.rope_sin = tables["cos"].handle, tables["sin"].handle
        if case["masked"]:
            ops.key_pad, x.mask_batch_bytes = tables["pad"].handle, tokens
    else:
        x.qk_mode, x.eps = hip.QK_ZIMAGE, wl.ZIMAGE_EPS
        ops.pos, ops.rope_pairs = tables["pos"].handle, tables["pairs"].handle
        for a in range(3):
            x.zimage_dims[a], x.zimage_base[a] = wl.ZIMAGE_DIMS[a], tables["bases"][a]
    if case["bound"]:
        x.score_bound = host.score_bound(*w)
    b.update(weights=wb, ext=x, ops=ops, params=hip.AttnParams(tokens, heads, heads, D, 0, 0))
    return b


def _zimage_tables(case):
    ctx = context()
    pos = host.zimage_sequence_positions(case["grid_h"], case["grid_w"], case["cap"])
    pairs, bases = host.zimage_rope_fill(wl.ZIMAGE_DIMS, wl.ZIMAGE_LENS, wl.ZIMAGE_THETA)
    return {"pos": ctx.buffer(np.ascontiguousarray(pos, np.uint64)), "pairs": ctx.buffer(pairs), "bases": bases}


def _prepare_fused(case, g, rng):
    ctx = context()
    if case["kind"] == "klein":
        cos, sin = host.klein_build_rope_ref(case["grid_h"], case["grid_w"], case["ref_h"], case["ref_w"], theta=KLEIN_THETA, txt_len=case["txt"])
        tables = {"cos": ctx.buffer(cos), "sin": ctx.buffer(sin)}
        if case["masked"]:
            pad = np.zeros((case["batch"], _tokens(case)), np.uint8)
            for b, n in enumerate(_text_lens(case)):
                pad[b, n:case["txt"]] = 1
            tables["pad"] = ctx.buffer(pad)
    else:
        tables = _zimage_tables(case)
    return {"tables": tables, "blocks": [_fused_block(case, g, rng, tables) for _ in range(case["blocks"])]}


def _prepare_plain(case, g, rng):
    tokens, heads = case["tokens"], case["heads"]
    cfg = host.Config(tokens, heads, heads, D, False, case["valid"])
    if case["host"]:
        q, k, v = (rng.standard_normal((tokens, heads, D), dtype=np.float32) for _ in range(3))
        return {"cfg": cfg, "q": q, "k": k, "v": v}
    s = {n: Resident(_randn(g, (tokens, heads, D), "f32")) for n in "qkv"}
    s.update(cfg=cfg, o=Resident(torch.zeros((tokens, heads, D), device="cuda")))
    return s


def _prepare_segment(case, g, rng):
    ctx, tokens, heads = context(), _tokens(case), case["heads"]
    inner = hidden = heads * D
    tables = _zimage_tables(case)
    layers = []
    for _ in range(case["layers"]):
        act = case["act"]
        t = {n: Resident(torch.zeros((tokens, inner), device="cuda", dtype=TORCH[act])) for n in ("q", "k", "v", "mix", "attn")}
        t["norm"] = Resident(_randn(g, (tokens, hidden), act))
        t["w"] = Resident(_randn(g, (4, inner, hidden), case["weight"], hidden ** -0.5))
        nw = [_norm_weight(rng) for _ in range(2)]
        t["nw"] = [ctx.buffer(_typed(a, case["norm"])) for a in nw]
        p = hip.ChainAttnParams()
        for i, name in enumerate(("q", "k", "v", "proj")):
            setattr(p, name, hip.GemmParams(tokens, hidden, inner, WEIGHT[case["weight"]], hip.GEMM_HALF, i * inner * hidden * 2))
        code = WEIGHT[case["norm"]]
        p.qk = hip.QkNormParams(tokens, heads, heads, D, code, code, *wl.ZIMAGE_DIMS, wl.ZIMAGE_EPS, 0, 0, *tables["bases"])
        p.attn = hip.AttnParams(tokens, heads, heads, D, 0, 0)
        p.act_dtype = ACT[act]
        p.score_bound = host.score_bound(*nw)
        t["params"] = p
        t["bufs"] = hip.ChainAttnBuffers(*(t[n].handle for n in ("norm", "q", "k", "v", "mix", "attn")))
        wh = t["w"].handle
        t["weights"] = hip.ChainAttnWeights(wh, wh, wh, t["nw"][0].handle, t["nw"][1].handle, tables["pos"].handle, tables["pairs"].handle, wh)
        layers.append(t)
    return {"tables": tables, "layers": layers}


def _prepare_wide(case, g, rng):
    s = {n: Resident(_randn(g, (case["tokens"], 1, WIDE), "f32")) for n in "qkv"}
    s.update(cfg=host.Config(case["tokens"], 1, 1, WIDE), o=Resident(torch.zeros((case["tokens"], 1, WIDE), device="cuda")))
    return s


def _products(case):
    """(rows, k, n, how many side by side) of each product of a block, in order."""
    h, txt, img = case["hidden"], case["txt"], case["img"]
    if case["block"] == "double":
        return [(img, h, h, 3), (txt, h, h, 3), (img, h, h, 1), (txt, h, h, 1)]
    return [(txt + img, h, h, 3), (txt + img, 4 * h, h, 1)]


def _prepare_project(case, g, rng):
    products = []
    for m, k, n, count in _products(case):
        a = Resident(_randn(g, (m, k), case["act"]))
        w = Resident(_randn(g, (count, n, k), case["weight"], k ** -0.5))
        c = [Resident(torch.zeros((m, n), device="cuda", dtype=TORCH[case["out"]])) for _ in range(count)]
        params = [hip.GemmParams(m, k, n, WEIGHT[case["weight"]], hip.GEMM_HALF, i * n * k * 2) for i in range(count)]
        products.append({"a": a, "w": w, "c": c, "params": params, "ext": hip.GemmExt(0, 0, 0, 0, 0, ACT[case["act"]], ACT[case["out"]]),
                         "ws": (C.c_void_p * count)(*([w.handle] * count)), "cs": (C.c_void_p * count)(*(x.handle for x in c)),
                         "ps": (C.POINTER(hip.GemmParams) * count)(*(C.pointer(p) for p in params)), "count": count})
    return {"products": products}


def prepare(case, seed):
    context()
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    rng = np.random.default_rng(seed)
    make = {"plain": _prepare_plain, "klein": _prepare_fused, "zimage": _prepare_fused, "segment": _prepare_segment,
            "wide": _prepare_wide, "project": _prepare_project}[case["kind"]]
    state = make(case, g, rng)
    state["case"] = dict(case)
    torch.cuda.synchronize()  # torch's stream made the operands, the library's queue reads them
    return state


# ------------------------------------------------------------------------- a pass
def _run_plain(s):
    if s["case"]["host"]:
        return host.attention_fast_run(context(), s["q"], s["k"], s["v"], s["cfg"])
    context().run_on_handles(s["q"].handle, s["k"].handle, s["v"].handle, s["o"].handle, s["cfg"])
    return s["o"].t


def _run_fused(s):
    lib, batch = hip.lib(), hip.lib().zdraw_hip_batch_begin(context().queue)
    for b in s["blocks"]:
        rc = lib.zdraw_hip_run_attention_fused_enc(batch, b["q"].handle, b["k"].handle, b["v"].handle, b["o"].handle,
                                                   C.byref(b["params"]), C.byref(b["ext"]), C.byref(b["ops"]))
        _check(rc, "fused attention")
    _check(lib.zdraw_hip_batch_end(batch), "batch_end")
    return [b["o"].t for b in s["blocks"]]


def _run_segment(s):
    lib, batch = hip.lib(), hip.lib().zdraw_hip_batch_begin(context().queue)
    for t in s["layers"]:
        _check(lib.zdraw_hip_run_chain_attn_enc(batch, C.byref(t["bufs"]), C.byref(t["weights"]), C.byref(t["params"])), "segment")
    _check(lib.zdraw_hip_batch_end(batch), "batch_end")
    return [{"attn": t["attn"].t, "mix": t["mix"].t} for t in s["layers"]]


def _run_wide(s):
    context().run_on_handles(s["q"].handle, s["k"].handle, s["v"].handle, s["o"].handle, s["cfg"])
    return s["o"].t


def _run_project(s):
    lib, batch = hip.lib(), hip.lib().zdraw_hip_batch_begin(context().queue)
    for p in s["products"]:
        rc = lib.zdraw_hip_run_gemm_group_ext_enc(batch, p["a"].handle, p["ws"], p["cs"], p["ps"], p["count"], C.byref(p["ext"]))
        _check(rc, "projection")
    _check(lib.zdraw_hip_batch_end(batch), "batch_end")
    return [[c.t for c in p["c"]] for p in s["products"]]


def run(state):
    return {"plain": _run_plain, "klein": _run_fused, "zimage": _run_fused, "segment": _run_segment, "wide": _run_wide,
            "project": _run_project}[state["case"]["kind"]](state)


# --------------------------------------------------------------------------- work
def work(case):
    kind = case["kind"]
    if kind == "plain":
        s, h = case["tokens"], case["heads"]
        return {"bytes": 4 * s * h * D * 4, "flops": 4 * D * h * s * (case["valid"] or s)}
    if kind == "wide":
        return {"bytes": 4 * case["tokens"] * WIDE * 4, "flops": 4 * WIDE * case["tokens"] ** 2}
    if kind in ("klein", "zimage"):
        s, h, batch, n = _tokens(case), case["heads"], case.get("batch", 1), case["blocks"]
        keys = [s - case["txt"] + t for t in _text_lens(case)] if case.get("masked") else [s] * batch
        table = 2 * s * D * 4 if kind == "klein" else s * (24 + D * 4)
        return {"bytes": n * (batch * s * h * D * (3 * SIZE[case["act"]] + SIZE[case["out"]]) + table), "flops": n * 4 * D * h * s * sum(keys)}
    if kind == "segment":
        s, hid, n = _tokens(case), case["heads"] * D, case["layers"]
        return {"bytes": n * (2 * s * hid * SIZE[case["act"]] + 4 * hid * hid * 2), "flops": n * (8 * s * hid * hid + 4 * hid * s * s)}
    out = {"bytes": 0, "flops": 0}
    for m, k, n, count in _products(case):
        out["bytes"] += m * k * SIZE[case["act"]] + count * (n * k * 2 + m * n * SIZE[case["out"]])
        out["flops"] += 2 * m * k * n * count
    return out


# The differences from the same paths in float64 on the operands as given, measured over these
# ranges (2-norm of the difference over the 2-norm of the result, and the largest): attention 3.7e-3
# and 2.9e-2, a segment 4.5e-3 and 2.5e-2; products with f32 results 3.5e-7 and 2.4e-6 (16-bit
# operands: only the order of the sums is free), with 16-bit results 1.7e-3 and 3.9e-3. Stated at
# about four times that; the f32 products at a little more for the longest sums.
def tolerance(case):
    if case["kind"] == "project":
        return {"rel": 3e-6, "max": 2e-5} if case["out"] == "f32" else {"rel": 6e-3, "max": 1.6e-2}
    return {"rel": 1.8e-2 if case["kind"] == "segment" else 1.5e-2, "max": 1.1e-1}
