"""The work that programs have this package do, as cases that can be timed and compared.

A case is a dict of plain values; its ``kind`` names the entry points that one
pass goes through:

  routed   ``switched.switched_lora_routed_``: one projection of a batch, from
           the requested ids to the updated y, called eagerly
  layer    one decoder layer's four projections (segments built once, then
           ``switched.switched_lora_`` for each), captured in a HIP graph as a
           serving loop keeps it; a pass is one replay
  hf       ``hf_layers`` forward: base linear, segments, shrink, expand
  vllm     ``vllm_layers.SwitchedLoRALinear.forward``: x . w_ext^T through this
           package's GEMM (or torch's), then the segment expand or the fused
           SwiGLU expand
  expand, swiglu, shunt   the three ``torch.ops.granite_switch`` expand ops on
           an x_ext that the caller's GEMM made
  meta     a step's routing and metadata: ``route_latest_wins`` and
           ``FusedLoRAKernelMeta.prepare_and_store``
  gemm     ``switched.linear_bf16``

Sizes are those of the benchmark and test configurations: hidden sizes 2048 to
32768, the QKV, output, gate/up and down projections, 2 to 48 adapters of rank
8 to 64, also with one rank-512 adapter among them, 1 to 8192 tokens (32768
for the metadata).
"""

from __future__ import annotations

import math

import numpy as np
import torch

import __graft_entry__

__graft_entry__.load_package()
from granite_switch_amd import hf_layers, kernels, meta, ops, switched, vllm_layers  # noqa: E402

ALPHA = 16.0
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
# projections: hidden size and output slices
QKV, O, GATE_UP, DOWN = (4096, "4096,1024,1024"), (4096, "4096"), (4096, "12800,12800"), (12800, "4096")
PROJECTIONS = (QKV, O, GATE_UP, DOWN, (2048, "2048"),
               (2560, "2560,512,512"), (2560, "8192,8192"), (8192, "2560"), (32768, "4096"))
ODD_PROJECTIONS = ((1000, "96"), (264, "32,64"), (520, "256,128,128"), (1024, "512,256"))


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def _case(kind, proj, tokens, adapters, ranks, routing, *, dtype="bf16", extra=0, seqs=0, name=None, **more):
    c = {"kind": kind, "hidden": proj[0], "slices": proj[1], "tokens": tokens, "adapters": adapters, "ranks": ranks,
         "extra": extra, "routing": routing, "seqs": seqs, "dtype": dtype, **more}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the last few requests of an idle server: one projection of a 7-token decode batch (latency only)
        _case("routed", O, 7, 12, "32", "decode", name="decode_o_t7"),
        # a full decode batch: QKV, 20 % of the requests not yet past their invocation point
        _case("routed", QKV, 256, 12, "32", "decode", name="decode_qkv_t256"),
        # fp32 evaluation of a small model: four sequences switching on inside the batch
        _case("routed", (2048, "2048"), 512, 4, "8", "prefill", seqs=4, dtype="fp32", name="fp32_proj_t512"),
        # a large chunked prefill into the widest projection
        _case("routed", GATE_UP, 8192, 12, "32", "prefill", seqs=16, name="prefill_gate_up_t8192"),
        # conversations that switch adapters every few tokens, mixed ranks
        _case("routed", DOWN, 4096, 48, "8,16,32,64", "switch", seqs=64, name="switch_down_t4096"),
        # a serving step: decode rows and prefill chunks together, one layer of it, as a captured graph
        _case("layer", (4096, ""), 4144, 24, "32", "mix", seqs=64, name="step_layer_t4144"),
        # a decode step with one rank-512 adapter loaded beside the rank-32 ones, as a captured graph
        _case("layer", (4096, ""), 256, 12, "32", "decode", extra=512, name="decode_layer_r512_t256"),
        # the HF model's fused QKV at an odd prompt length
        _case("hf", QKV, 1531, 8, "16,32", "prefill", seqs=3, name="hf_qkv_t1531"),
        # the vLLM layer at decode: GEMM over [W; A...] and the expand over its shrink columns
        _case("vllm", QKV, 256, 12, "32", "decode", native=True, fused=False, name="vllm_qkv_t256"),
        # the vLLM layer's largest call: gate/up of a mixed step with the fused SwiGLU expand
        _case("vllm", GATE_UP, 4144, 24, "32", "mix", seqs=64, native=True, fused=True, name="vllm_gate_up_t4144"),
        # the reference-form op on an odd batch of decode and short prompts, three rank tiers
        _case("expand", QKV, 777, 24, "16,32,64", "mix", seqs=40, name="expand_op_qkv_t777"),
        # routing and metadata of a long-prompt step for all the projections of a 40-layer model
        _case("meta", (0, ""), 32768, 24, "32", "prefill", seqs=5, modules=160, name="meta_t32768"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["routed", "routed", "routed", "layer", "hf", "vllm", "vllm", "expand", "swiglu", "shunt",
                       "meta", "gemm"])
    routing = rng.choice(["decode", "prefill", "switch", "mix"])
    tokens = _log_int(rng, 1, 512) if routing == "decode" else _log_int(rng, 33, 8192)
    seqs = tokens if routing == "decode" else max(1, min(tokens // 8, _log_int(rng, 1, 64)))
    adapters = _log_int(rng, 2, 48)
    ranks = rng.choice(["8", "16", "32", "32", "64", "8,16,32,64", "24,40", "16,32"])
    proj = rng.choice(PROJECTIONS[:5] * 2 + PROJECTIONS[5:] + ODD_PROJECTIONS)
    extra = 512 if rng.random() < 0.12 and proj[0] <= 4096 else 0
    if kind == "meta":
        return _case("meta", (0, ""), _log_int(rng, 1, 32768), adapters, "32", rng.choice(["decode", "prefill"]),
                     seqs=_log_int(rng, 1, 64), modules=rng.choice([4, 80, 128, 160]))
    if kind == "layer":
        return _case("layer", (4096, ""), min(tokens, 4144), min(adapters, 24), rng.choice(["16", "32", "16,32"]),
                     routing, seqs=seqs, extra=extra)
    if kind == "hf":
        return _case("hf", proj, min(tokens, 3000), min(adapters, 24), ranks, routing, seqs=seqs,
                     dtype=rng.choice(["bf16", "bf16", "fp32"]))
    if kind == "routed":
        return _case("routed", proj, tokens, adapters, ranks, routing, seqs=seqs, extra=extra,
                     dtype=rng.choice(["bf16", "bf16", "bf16", "fp32"]))
    if kind == "shunt":
        return _case("shunt", rng.choice((O, (2048, "2048"), (2560, "2560"))), min(tokens, 4144), min(adapters, 24),
                     rng.choice(["16", "32", "16,32"]), routing, seqs=seqs, dtype=rng.choice(["bf16", "fp32"]))
    adapters = min(adapters, 24)
    if kind in ("expand", "swiglu"):
        proj = rng.choice((GATE_UP, (2560, "8192,8192")) if kind == "swiglu" else (QKV, O, DOWN, (2560, "2560,512,512")))
        return _case(kind, proj, tokens, adapters, rng.choice(["16", "32", "16,32", "16,32,64"]), routing, seqs=seqs)
    if kind == "gemm":
        proj = rng.choice((QKV, O, GATE_UP, DOWN, (2048, "2048"), (1000, "96"), (2560, "2560")))
    else:
        proj = rng.choice((QKV, O, GATE_UP, DOWN, (2048, "2048"), (2560, "2560,512,512")))
    return _case(kind, proj, min(tokens, 4096), adapters, rng.choice(["16", "32"]), routing, seqs=seqs,
                 **({} if kind == "gemm" else {"native": rng.random() < 0.75,
                                               "fused": proj is GATE_UP and rng.random() < 0.7}))


# ---------------------------------------------------------------------------
# Routing: requested ids, positions, sequence bounds and activation offsets
# ---------------------------------------------------------------------------
def _lengths(rng, total, n):
    """n lengths that sum to total, log-uniform over a factor of 32."""
    n = max(1, min(n, total))
    raw = np.exp(rng.uniform(0.0, math.log(32.0), size=n))
    ends = np.maximum(np.floor(np.cumsum(raw) / raw.sum() * total).astype(np.int64), np.arange(1, n + 1))
    ends[-1] = total
    ends = np.minimum(ends, total - np.arange(n - 1, -1, -1))
    return np.diff(np.concatenate([[0], ends]))


def _num_adapters(case):
    return case["adapters"] + (1 if case["extra"] else 0)


def _rank_list(case):
    given = [int(r) for r in case["ranks"].split(",")]
    ranks = [given[a % len(given)] for a in range(case["adapters"])]
    return ranks + [case["extra"]] if case["extra"] else ranks


def _slice_list(case):
    return tuple(int(s) for s in case["slices"].split(","))


def _routing(case, seed):
    """(requested ids, positions, cu_seqlens, activation offsets or None, effective ids), numpy."""
    rng = np.random.default_rng(int(seed) % (1 << 31))
    T, NA, kind = case["tokens"], _num_adapters(case), case["routing"]
    if kind == "switch":
        lens = _lengths(rng, T, case["seqs"])
        req = np.zeros(T, dtype=np.int64)
        at = 0
        while at < T:
            run = int(rng.integers(4, 17))
            req[at:at + run] = 0 if rng.random() < 0.15 else rng.integers(1, NA + 1)
            at += run
        pos = np.concatenate([np.arange(n) for n in lens])
        off = None
    else:
        decode = T if kind == "decode" else (min(T - 1, case["seqs"] * 3 // 4) if kind == "mix" else 0)
        lens = np.ones(decode, dtype=np.int64)
        start = rng.integers(16, 2048, size=decode)
        offs = start + np.where(rng.random(decode) < 0.2, 1, 0) * rng.integers(1, 16, size=decode)
        if decode < T:
            plen = _lengths(rng, T - decode, max(1, case["seqs"] - decode))
            pstart = rng.integers(0, 8, size=len(plen)) * 256 * (kind == "mix")
            lens = np.concatenate([lens, plen])
            start = np.concatenate([start, pstart])
            # the invocation point lies anywhere in the prompt so far
            offs = np.concatenate([offs, (rng.random(len(plen)) * (pstart + plen)).astype(np.int64)])
        req = np.repeat(rng.integers(1, NA + 1, size=len(lens)), lens)
        pos = np.concatenate([s + np.arange(n) for s, n in zip(start, lens)])
        off = offs
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    eff = req if off is None else np.where(pos >= np.repeat(off, lens), req, 0)
    return req, pos, cu, off, eff


def _dev():
    return torch.device("cuda", torch.cuda.current_device())


def _gen(seed):
    return torch.Generator(device=_dev()).manual_seed(int(seed))


def _normal(g, *shape, std=1.0, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=g, device=_dev()).mul_(std).to(dtype)


def _adapters(g, ranks, hidden, slices, dtype):
    """Checkpoint layout: lora_A [NA, 1, R, H] and pre-scaled lora_B [NA, 1, O_s, R] per slice, zero past each rank."""
    NA, R = len(ranks), max(ranks)
    A_sl, B_sl = [], []
    for width in slices:
        A = torch.zeros(NA, 1, R, hidden, dtype=dtype, device=_dev())
        B = torch.zeros(NA, 1, width, R, dtype=dtype, device=_dev())
        for a, r in enumerate(ranks):
            A[a, 0, :r] = _normal(g, r, hidden, std=hidden ** -0.5, dtype=dtype)
            B[a, 0, :, :r] = _normal(g, width, r, std=0.02 * ALPHA / r, dtype=dtype)
        A_sl.append(A)
        B_sl.append(B)
    return A_sl, B_sl


def _layer_projections():
    return {"qkv": QKV, "o": O, "gate_up": GATE_UP, "down": DOWN}


def _on_gpu(routing):
    req, pos, cu, off, _ = routing
    return tuple(None if v is None else torch.tensor(v, device=_dev()) for v in (req, pos, cu, off))


# ---------------------------------------------------------------------------
# Inputs (from the seed alone), shared by prepare() and exact()
# ---------------------------------------------------------------------------
def _projection_inputs(case, seed, proj=None):
    """x, y and the adapters of one projection."""
    hidden, slices = (case["hidden"], _slice_list(case)) if proj is None else (proj[0], tuple(map(int, proj[1].split(","))))
    g, dtype = _gen(seed), DTYPES[case["dtype"]]
    x = _normal(g, case["tokens"], hidden, dtype=dtype)
    y = _normal(g, case["tokens"], sum(slices), dtype=dtype)
    A_sl, B_sl = _adapters(g, _rank_list(case), hidden, slices, dtype)
    return x, y, A_sl, B_sl


def _weight_inputs(case, seed):
    """x, the base weight and the adapters of one layer."""
    hidden, slices = case["hidden"], _slice_list(case)
    g, dtype = _gen(seed), DTYPES[case["dtype"]]
    x = _normal(g, case["tokens"], hidden, dtype=dtype)
    W = _normal(g, sum(slices), hidden, std=hidden ** -0.5, dtype=dtype)
    A_sl, B_sl = _adapters(g, _rank_list(case), hidden, slices, dtype)
    return x, W, A_sl, B_sl


def _vllm_layer(case, W, A_sl, B_sl):
    slices, S = _slice_list(case), len(_slice_list(case))
    base = torch.nn.Linear(case["hidden"], sum(slices), bias=False, device="meta")
    base.weight = torch.nn.Parameter(W.clone(), requires_grad=False)
    layer = vllm_layers.SwitchedLoRALinear(base, _num_adapters(case), max(_rank_list(case)), num_slices=S,
                                           output_slices=slices if S > 1 else None,
                                           fuse_swiglu=case.get("fused", case["kind"] == "swiglu"))
    for p, v in zip([layer.lora_A] if S == 1 else layer.lora_A_slices, A_sl):
        p.data.copy_(v)
    for p, v in zip([layer.lora_B] if S == 1 else layer.lora_B_slices, B_sl):
        p.data.copy_(v)
    layer.finalize_weights(_rank_list(case))
    layer.native_gemm = bool(case.get("native", False))
    return layer


def _context(layer, eff):
    fm = meta.FusedLoRAKernelMeta(_dev())
    fm.register_remap_tables(layer.remap_table.unsqueeze(0),
                             [(layer.in_features, layer._N_total, layer._num_applicable)])
    ctx = meta.LoRAContext()
    fm.prepare_and_store(torch.tensor(eff, device=_dev()), ctx)
    return ctx


def _xext_adapters(case, seed):
    """lora_B [sum(slices), r] per adapter, and each adapter's first column in x_ext (tier, then index)."""
    g, slices, ranks = _gen(seed + 1), _slice_list(case), _rank_list(case)
    S, at = len(slices), 0 if case["kind"] == "shunt" else sum(slices)
    Bs, cols = {}, {}
    for tier in kernels.SUPPORTED_RANKS:
        for a, r in enumerate(ranks):
            if kernels.promote_rank(r) == tier:
                Bs[a] = _normal(g, sum(slices), tier, std=0.02 * ALPHA / r)
                cols[a] = at
                at += S * tier
    x_ext = _normal(g, case["tokens"], at)
    return Bs, cols, x_ext


def _xext_tables(case, Bs, eff):
    """The op's tables for those adapters: every adapter applies, numbered by tier and index."""
    slices, ranks, dev = _slice_list(case), _rank_list(case), _dev()
    S, N = len(slices), sum(slices)
    order = sorted(range(len(ranks)), key=lambda a: (kernels.promote_rank(ranks[a]), a))
    tiers = [kernels.promote_rank(ranks[a]) for a in order]
    na = tuple(tiers.count(t) for t in kernels.SUPPORTED_RANKS)
    remap = torch.zeros(len(ranks) + 1, dtype=torch.int64)
    for local, a in enumerate(order):
        remap[a + 1] = local + 1
    base = (0 if case["kind"] == "shunt" else N) + np.cumsum([0] + [n * S * r for n, r in zip(na, kernels.SUPPORTED_RANKS)])
    scr = [[int(base[t]) + s * r for t, r in enumerate(kernels.SUPPORTED_RANKS)] for s in range(S)]
    ends = np.cumsum(slices)
    tile_slice = [int(np.searchsorted(ends, j, side="right")) for j in range(0, N, kernels.BLOCK_N)]
    remapped = remap.to(dev)[torch.tensor(eff, device=dev)].contiguous()
    masks = kernels.compute_per_module_bitmasks(torch.tensor(eff, device=dev), remap.to(dev).unsqueeze(1).contiguous())
    return {"lb": torch.cat([Bs[a].reshape(-1) for a in order]), "na": na, "ids": remapped, "masks": masks[0],
            "tile_slice": torch.tensor(tile_slice, dtype=torch.int32, device=dev),
            "scr": torch.tensor(scr, dtype=torch.int32, device=dev), "S": S, "N": N}


CONTROL_0 = 49160     # token id of the first adapter's control token


def _meta_inputs(case, seed):
    """Prompt tokens with a control token at each sequence's invocation point, and the remap tables.

    The case alone fixes the step's shape (lengths, invocation points, which
    sequences carry an adapter over), the seed what is in it.
    """
    shape = np.random.default_rng([case["tokens"], case["seqs"], case["modules"]])
    rng = np.random.default_rng(int(seed) % (1 << 31))
    T, NA = case["tokens"], case["adapters"]
    lens = _lengths(shape, T, case["seqs"] if case["routing"] == "prefill" else T)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    start = (shape.random(len(lens)) < (0.8 if case["routing"] == "decode" else 0.3)) * rng.integers(1, NA + 1, size=len(lens))
    tokens = rng.integers(0, CONTROL_0, size=T)
    at = cu[:-1] + (shape.random(len(lens)) * lens).astype(np.int64)
    at = at[lens > 1]
    tokens[at] = CONTROL_0 + rng.integers(0, NA, size=len(at))
    remap = np.zeros((case["modules"], NA + 1), dtype=np.int64)
    for m in range(case["modules"]):
        applies = np.flatnonzero(rng.random(NA) < 0.8)
        remap[m, 1 + applies] = rng.permutation(len(applies)) + 1
    seq, fired = np.repeat(np.arange(len(lens)), lens), np.zeros(T, dtype=np.int64)
    fired[at] = tokens[at] - CONTROL_0 + 1
    last = np.maximum.accumulate(np.where(fired > 0, np.arange(T), -1))
    ids = np.where(last >= cu[:-1][seq], fired[np.maximum(last, 0)], start[seq])
    return tokens, cu, start, remap, ids


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    kind, dev = case["kind"], _dev()
    if kind == "meta":
        tokens, cu, start, remap, ids = _meta_inputs(case, seed)
        fm = meta.FusedLoRAKernelMeta(dev)
        fm.register_remap_tables(torch.tensor(remap, device=dev), [None] * case["modules"])
        return {"kind": kind, "fm": fm, "tokens": torch.tensor(tokens, device=dev), "cu": torch.tensor(cu, device=dev),
                "start": torch.tensor(start, device=dev),
                "control": torch.arange(CONTROL_0, CONTROL_0 + case["adapters"], device=dev),
                "adapted": int((ids > 0).sum())}
    if kind == "gemm":
        x, w = _gemm_inputs(case, seed)
        return {"kind": kind, "x": x, "w": w}
    routing = _routing(case, seed)
    if kind == "routed":
        x, y, A_sl, B_sl = _projection_inputs(case, seed)
        req, pos, cu, off = _on_gpu(routing)
        return {"kind": kind, "x": x, "y": y, "ids": req, "pos": pos, "cu": cu, "off": off,
                "pack": switched.PackedAdapters.from_slices(A_sl, B_sl, _rank_list(case))}
    if kind == "layer":
        return _prepare_layer(case, seed, routing)
    if kind == "hf":
        x, W, A_sl, B_sl = _weight_inputs(case, seed)
        return {"kind": kind, "x": x, "layer": _hf_layer(case, W, A_sl, B_sl), "ids": torch.tensor(routing[4], device=dev)}
    if kind == "vllm":
        x, W, A_sl, B_sl = _weight_inputs(case, seed)
        layer = _vllm_layer(case, W, A_sl, B_sl)
        layer._lora_ctx = _context(layer, routing[4])
        return {"kind": kind, "x": x, "layer": layer}
    Bs, _, x_ext = _xext_adapters(case, seed)
    return {"kind": kind, "x_ext": x_ext, "dtype": DTYPES[case["dtype"]], **_xext_tables(case, Bs, routing[4])}


def _gemm_inputs(case, seed):
    slices, S = _slice_list(case), len(_slice_list(case))
    n = sum(slices) + S * sum(kernels.promote_rank(r) for r in _rank_list(case))
    g = _gen(seed)
    return _normal(g, case["tokens"], case["hidden"]), _normal(g, n, case["hidden"], std=case["hidden"] ** -0.5)


def _hf_layer(case, W, A_sl, B_sl):
    slices, NA, R = _slice_list(case), _num_adapters(case), max(_rank_list(case))
    with _dev():
        if len(slices) == 1:
            layer = hf_layers.SwitchedLoRALinear(case["hidden"], slices[0], NA, R, bias=False)
        else:
            layer = hf_layers.MergedSwitchedLoRALinear(case["hidden"], slices, NA, R)
    layer = layer.to(DTYPES[case["dtype"]])
    with torch.no_grad():
        layer.weight.copy_(W)
        for p, v in zip(*((layer.lora_A, layer.lora_B), (A_sl[0], B_sl[0])) if len(slices) == 1 else
                        ([*layer.lora_A_slices, *layer.lora_B_slices], [*A_sl, *B_sl])):
            p.copy_(v)
    layer.freeze(_rank_list(case))
    return layer


def _prepare_layer(case, seed, routing):
    """The four projections of a layer as one HIP graph over static buffers."""
    req, pos, cu, off = _on_gpu(routing)
    NA, parts = _num_adapters(case), {}
    for k, (name, proj) in enumerate(_layer_projections().items()):
        x, y, A_sl, B_sl = _projection_inputs(case, seed + 101 * k, proj)
        parts[name] = (y, x, switched.PackedAdapters.from_slices(A_sl, B_sl, _rank_list(case)))
        del A_sl, B_sl
    segs = switched.build_segments(req, NA, pos, cu, off)

    def step(copies=False):
        switched.build_segments(req, NA, pos, cu, off, out=segs)
        for y, x, pack in parts.values():
            switched.switched_lora_(y.clone() if copies else y, x, segs, pack)

    step(copies=True)          # workspaces are allocated before the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    return {"kind": "layer", "graph": graph, "parts": parts, "segs": segs, "inputs": (req, pos, cu, off),
            "y": {name: p[0] for name, p in parts.items()}}


def run(state):
    kind = state["kind"]
    if kind == "routed":
        return switched.switched_lora_routed_(state["y"], state["x"], state["ids"], state["pack"], state["pos"],
                                              state["cu"], state["off"])
    if kind == "layer":
        state["graph"].replay()
        return state["y"]
    if kind == "hf":
        with torch.no_grad():
            return state["layer"](state["x"], state["ids"])
    if kind == "vllm":
        return state["layer"](state["x"])[0]
    if kind == "gemm":
        return switched.linear_bf16(state["x"], state["w"])
    if kind == "meta":
        ids = switched.route_latest_wins(state["tokens"], state["control"], cu_seqlens=state["cu"], start_ids=state["start"])
        ctx = meta.LoRAContext()
        state["fm"].prepare_and_store(ids, ctx)
        return {"ids": ids, "masks": ctx.per_module_bitmasks, "remapped": ctx.remapped_indices,
                "eff": ctx.segments.eff_ids, "offsets": ctx.segments.seg_offsets,
                "perm": ctx.segments.perm[:state["adapted"]]}        # the rest of perm is not written
    x_ext, N, tail = state["x_ext"], state["N"], (*state["na"], state["S"], kernels.BLOCK_N)
    if kind == "expand":
        ops.op("switch_lora_expand")(x_ext, state["ids"], state["masks"], state["lb"], state["tile_slice"],
                                     state["scr"], *tail, N)
        return x_ext[:, :N]
    if kind == "swiglu":
        out = torch.empty(x_ext.shape[0], N // 2, dtype=x_ext.dtype, device=x_ext.device)
        ops.op("switch_lora_expand_swiglu")(out, x_ext, state["ids"], state["masks"], state["lb"], state["scr"], *tail,
                                            N // 2, N)
        return out
    out = torch.empty(x_ext.shape[0], N, dtype=state["dtype"], device=x_ext.device)
    ops.op("switch_lora_shrink_expand")(out, x_ext, state["ids"], state["masks"], state["lb"], state["tile_slice"],
                                        state["scr"], *tail, N)
    return out


# ---------------------------------------------------------------------------
# The least work, the exact results and their tolerances
# ---------------------------------------------------------------------------
def _lora_work(case, eff, hidden, slices, e):
    """(bytes, flops) of y += (x A^T) B^T over the adapted rows."""
    ranks, S, N = _rank_list(case), len(slices), sum(slices)
    rows = np.bincount(eff, minlength=len(ranks) + 1)[1:]
    act, used = int(rows.sum()), sum(r for r, n in zip(ranks, rows) if n)
    flops = sum(2 * int(n) * r * (S * hidden + N) for r, n in zip(ranks, rows))
    return e * (act * hidden + S * hidden * used + N * used + 2 * act * N) + 8 * len(eff), flops


def work(case):
    kind = case["kind"]
    T, e = case["tokens"], 4 if case["dtype"] == "fp32" else 2
    if kind == "meta":
        m = case["modules"]
        return {"bytes": 8 * T + 8 * T + 4 * T + 4 * T + 8 * T * m + 8 * m * -(-T // 32), "flops": 0}
    eff = _routing(case, 0)[4]
    if kind == "layer":
        both = [_lora_work(case, eff, h, tuple(map(int, s.split(","))), e) for h, s in _layer_projections().values()]
        return {"bytes": sum(b for b, _ in both), "flops": sum(f for _, f in both)}
    H, slices, ranks = case["hidden"], _slice_list(case), _rank_list(case)
    S, N = len(slices), sum(slices)
    if kind == "routed":
        b, f = _lora_work(case, eff, H, slices, e)
        return {"bytes": b, "flops": f}
    if kind == "hf":
        _, f = _lora_work(case, eff, H, slices, e)
        used = sum(r for a, r in enumerate(ranks) if (eff == a + 1).any())
        return {"bytes": e * (T * H + N * H + T * N + used * (S * H + N)) + 8 * T, "flops": f + 2 * T * N * H}
    shrink = S * sum(kernels.promote_rank(r) for r in ranks)
    rows = np.bincount(eff, minlength=len(ranks) + 1)[1:]
    delta = sum(2 * int(n) * kernels.promote_rank(r) * N for r, n in zip(ranks, rows))
    lb = 2 * N * sum(kernels.promote_rank(r) for r, n in zip(ranks, rows) if n)
    z = 2 * S * sum(int(n) * kernels.promote_rank(r) for r, n in zip(ranks, rows))
    if kind in ("gemm", "vllm"):
        w = N + shrink
        out = N // 2 if case.get("fused") else (N if kind == "vllm" else w)
        return {"bytes": 2 * (T * H + w * H + T * out) + (lb + 8 * T if kind == "vllm" else 0),
                "flops": 2 * T * w * H + (delta if kind == "vllm" else 0)}
    if kind == "expand":
        return {"bytes": 4 * int(rows.sum()) * N + z + lb + 8 * T, "flops": delta}
    if kind == "swiglu":
        return {"bytes": 3 * T * N + z + lb + 8 * T, "flops": delta + 4 * T * N}
    return {"bytes": e * T * N + z + lb + 8 * T, "flops": delta}


def _delta64(x, eff, A_sl, B_sl, ranks, out):
    """out += switched-LoRA delta of x, everything in 64 bits."""
    for a, r in enumerate(ranks):
        rows = torch.tensor(np.flatnonzero(eff == a + 1), device=out.device)
        if rows.numel():
            z = [x[rows].double() @ A[a, 0, :r].double().t() for A in A_sl]
            out[rows] += torch.cat([zs @ B[a, 0, :, :r].double().t() for zs, B in zip(z, B_sl)], dim=1)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "meta":
        return None
    if kind == "gemm":
        x, w = _gemm_inputs(case, seed)
        return x.double() @ w.double().t()
    ranks, eff = _rank_list(case), _routing(case, seed)[4]
    if kind == "layer":
        got = {}
        for k, (name, proj) in enumerate(_layer_projections().items()):
            x, y, A_sl, B_sl = _projection_inputs(case, seed + 101 * k, proj)
            got[name] = _delta64(x, eff, A_sl, B_sl, ranks, y.double())
        return got
    if kind == "routed":
        x, y, A_sl, B_sl = _projection_inputs(case, seed)
        return _delta64(x, eff, A_sl, B_sl, ranks, y.double())
    if kind in ("hf", "vllm"):
        x, W, A_sl, B_sl = _weight_inputs(case, seed)
        out = _delta64(x, eff, A_sl, B_sl, ranks, x.double() @ W.double().t())
        if case.get("fused"):
            gate, up = out.chunk(2, dim=1)
            out = gate * torch.sigmoid(gate) * up
        return out
    Bs, cols, x_ext = _xext_adapters(case, seed)
    slices, N = _slice_list(case), sum(_slice_list(case))
    out = torch.zeros(case["tokens"], N, dtype=torch.float64, device=x_ext.device) if kind == "shunt" \
        else x_ext[:, :N].double()
    for a, B in Bs.items():
        rows = torch.tensor(np.flatnonzero(eff == a + 1), device=out.device)
        r, lo = B.shape[1], 0
        for s, width in enumerate(slices):
            z = x_ext[rows, cols[a] + s * r:cols[a] + (s + 1) * r].double()
            out[rows, lo:lo + width] += z @ B[lo:lo + width].double().t()
            lo += width
    if kind == "swiglu":
        gate, up = out.chunk(2, dim=1)
        out = gate * torch.sigmoid(gate) * up
    return out


def tolerance(case):
    """About four times the error against exact() (2-norm, and of the worst value) that
    two orders of summation and two kernels of each path were measured at."""
    kind = case["kind"]
    if kind == "meta":
        return "exact"
    if case["dtype"] == "fp32":
        return {"rel": 8e-6, "max": 5e-5} if kind == "hf" else {"rel": 4e-7, "max": 4e-6}
    if kind in ("hf", "vllm"):          # base output and shrink values rounded before the expand
        return {"rel": 1.3e-2, "max": 0.05} if case.get("fused") else {"rel": 1e-2, "max": 0.032}
    return {"rel": 7e-3, "max": 0.02}
