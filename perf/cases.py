"""Performance cases of the expert-paging path, through its public entry points.

The path of one MoE layer: acquire slots, bring the missing experts' rows from
pinned RAM (raw or compressed), expand compressed rows, run the fp8 expert FFN
on the slab; at load time, compress the rows. The kinds below stand for:

- ``step``: the expert FFN of small batches (decode steps, one to a few dozen
  tokens) over experts resident in the slab. A serving loop captures these
  steps in a graph, layer after layer, so a case is ``layers`` layers captured
  once in ``prepare`` and replayed in ``run``. The choice between the decode
  step and the separate calls is the pager's own (``moe.decode_pays``).
- ``ffn``: the expert FFN of a prefill, one eager call of ``moe.fused_moe``.
- ``expand``: the batched expansion of compressed rows resident in HBM.
- ``expand_ram``: the same for the few misses of a decode step, their records
  read straight from the pinned RAM tier.
- ``encode``: compression of expert rows at load time, one row per call
  (a weight loader that hands over one expert at a time) up to a layer's.
- ``prefill``: a whole layer forward of the pager whose routing overflows the
  cache slots, so the experts go through the working slab in chunks.
- ``trace``: decode steps of the pager with hits and misses, captured.

Expert sizes: hidden 2048 and intermediate 512 over 256 experts with top-8 (the
benchmark's model), and generic multiples of 128 around them. Weights are
N(0, 0.02) quantised to fp8 e4m3 with one scale per 128x128 block, tokens
N(0, 1) in bf16, routing by the top-k of random logits with a per-expert bias,
so that some experts get several times the tokens of others.
"""

import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "vllm-expert-pager_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from vllm_expert_pager import codec, moe  # noqa: E402
from vllm_expert_pager import pager as pg  # noqa: E402

B = moe.BLOCK
GROUP = codec.GROUP  # values per codec group: rows are multiples of it
PITCH = 0.89  # the pager's default pitch ratio
SKEW = 0.4  # standard deviation of the router's per-expert bias


def listed():
    big = {"E": 256, "H": 2048, "I": 512, "topk": 8, "act": "silu", "ids": "int64"}
    return [
        # One sequence decoding: 8 pairs, 8 resident experts, 16 layers a graph.
        {"name": "step_1_token", "kind": "step", "T": 1, "layers": 16, **big},
        # Four sequences: 32 pairs, the most that the default 32 cache slots take.
        {"name": "step_4_tokens", "kind": "step", "T": 4, "layers": 8, **big},
        # A batch of sequences over a larger cache: 184 pairs, mostly one or two per expert.
        {"name": "step_23_tokens", "kind": "step", "T": 23, "layers": 4, **big},
        # A short ragged prefill of a smaller GELU model, int32 ids.
        {"name": "ffn_333_tokens_gelu", "kind": "ffn", "T": 333, "E": 64, "H": 2048, "I": 768, "topk": 8,
         "act": "gelu", "ids": "int32"},
        # The benchmark's prefill layer.
        {"name": "ffn_2048_tokens", "kind": "ffn", "T": 2048, **big},
        # The largest prefill batch a scheduler usually allows.
        {"name": "ffn_8192_tokens", "kind": "ffn", "T": 8192, **big},
        # The benchmark's headline: all 256 experts of a layer expanded from HBM.
        {"name": "expand_256_experts", "kind": "expand", "rows": 256, "H": 2048, "I": 512},
        # A decode step's misses expanded from pinned RAM.
        {"name": "expand_ram_3_experts", "kind": "expand_ram", "rows": 3, "H": 2048, "I": 512},
        # Loading expert by expert: one w13 row (2 MiB) a call.
        {"name": "encode_1_row", "kind": "encode", "rows": 1, "groups": 128},
        # Loading a layer at once: 256 w13 rows.
        {"name": "encode_256_rows", "kind": "encode", "rows": 256, "groups": 128},
        # A prefill through the tiers: 2048 tokens, every expert in a compressed RAM tier.
        {"name": "prefill_2048_tokens", "kind": "prefill", "T": 2048, "compress": True, "slots": 32, "W": 64, **big},
        # Decode steps with paging from a raw RAM tier: 2 layers, 16 steps a graph.
        {"name": "trace_16_steps", "kind": "trace", "T": 1, "layers": 2, "steps": 16, "compress": False,
         "slots": 32, "W": 16, **{**big, "E": 128}},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_model(rng, most_values):
    """A random expert shape with at most ``most_values`` weights in all."""
    while True:
        E = rng.choice([16, 48, 64, 128, 160, 256])
        H, I = B * rng.randint(4, 32), B * rng.randint(1, 12)
        topk = rng.choice([1, 2, 4, 6, 8, 8, 10])
        if E * 3 * H * I <= most_values:
            return {"E": E, "H": H, "I": I, "topk": topk, "act": rng.choice(["silu", "silu", "gelu"]),
                    "ids": rng.choice(["int64", "int32"])}


def draw(rng):
    kind = rng.choice(["step", "step", "ffn", "ffn", "expand", "expand_ram", "encode", "encode", "prefill", "trace"])
    if kind == "step":
        return {"kind": kind, "T": _log_int(rng, 1, 64), "layers": 4, **_draw_model(rng, 256 * 3 * 2048 * 512)}
    if kind == "ffn":
        c = _draw_model(rng, 256 * 3 * 2048 * 512)
        most = 8192 * 8 * 2048 * 512 // (c["topk"] * c["H"] * c["I"])  # no more work than the largest listed case
        return {"kind": kind, "T": _log_int(rng, 65, max(66, min(8192, most))), **c}
    if kind in ("expand", "expand_ram"):
        while True:
            H, I = B * rng.randint(4, 32), B * rng.randint(1, 12)
            rows = _log_int(rng, 1, 256 if kind == "expand" else 12)
            if H * I % GROUP == 0 and rows * H * I <= 256 * 2048 * 512:
                return {"kind": kind, "rows": rows, "H": H, "I": I}
    if kind == "encode":
        return {"kind": kind, "rows": _log_int(rng, 1, 256), "groups": _log_int(rng, 3, 160)}
    c = {"E": rng.choice([16, 48, 64, 96]), "H": B * 2 * rng.randint(2, 8), "I": B * rng.randint(1, 4),
         "topk": rng.choice([4, 6, 8]), "act": rng.choice(["silu", "gelu"]), "ids": rng.choice(["int64", "int32"])}
    compress = rng.random() < 0.5
    if kind == "prefill":
        return {"kind": kind, "T": _log_int(rng, 5, 1024), "compress": compress, "slots": 16,
                "W": rng.choice([8, 16, 32]), **c}
    return {"kind": kind, "T": rng.choice([1, 2]), "layers": rng.randint(1, 3), "steps": rng.choice([4, 8]),
            "compress": compress, "slots": 16, "W": 8, **c}


# ---- inputs ----


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1009 + salt)


def _fp8_blocks(g, n, blocks):
    """(n, blocks * GROUP) bytes: N(0, 0.02) weights, one amax / 448 scale per 128x128 block; and the scales."""
    rows = torch.empty((n, blocks * GROUP), dtype=torch.uint8, device="cuda")
    scales = torch.empty((n, blocks), dtype=torch.float32, device="cuda")
    step = max(1, (1 << 26) // (blocks * GROUP))
    for i in range(0, n, step):
        w = torch.randn((min(step, n - i), blocks, GROUP), generator=g, device="cuda") * 0.02
        s = (w.abs().amax(dim=2) / 448.0).clamp_min(1e-10)
        rows[i : i + step] = (w / s[:, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8).flatten(1)
        scales[i : i + step] = s
    return rows, scales


def _weights(g, E, n, k):
    """E fp8 matrices (n, k) as bytes with their block scales: the blocks' 16384 values become 128x128 tiles."""
    rows, scales = _fp8_blocks(g, E, n * k // (B * B))
    w = rows.view(E, n // B, k // B, B, B).transpose(2, 3).reshape(E, n, k)
    return w, scales.view(E, n // B, k // B)


def _experts(case, seed):
    """(w13, w13_scale, w2, w2_scale) of a case's experts."""
    g = _gen(seed, 1)
    E, H, I = case["E"], case["H"], case["I"]
    return (*_weights(g, E, 2 * I, H), *_weights(g, E, H, I))


def _tokens(case, seed, steps=1):
    """Per step: tokens (T, H) bf16, routed weights (T, topk) and expert ids (T, topk)."""
    g = _gen(seed, 2)
    E, T = case["E"], case["T"]
    bias = SKEW * torch.randn((E,), generator=g, device="cuda")
    out = []
    for _ in range(steps):
        x = torch.randn((T, case["H"]), generator=g, device="cuda").to(torch.bfloat16)
        top, ids = (torch.randn((T, E), generator=g, device="cuda") + bias).topk(case["topk"], dim=1)
        out.append((x, torch.softmax(top, dim=1).contiguous(), ids.to(getattr(torch, case["ids"])).contiguous()))
    return out


def _capture(fn):
    """fn's launches as a graph (run once before, as every capture is), and what the captured call returned."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def _step(case, x, tw, ids, emap, w):
    """The pager's expert FFN of a batch whose experts are all in the slab."""
    E = case["E"]
    if moe.decode_pays(x, ids, case["I"]):
        return moe.decode_experts(x, tw, ids, emap, E, *w, E, activation=case["act"])
    xq, xs, routing = moe.quant_route(x, ids, emap, E)
    contrib = torch.empty((ids.numel(), x.shape[1]), dtype=torch.bfloat16, device=x.device)
    moe.run_experts(xq, xs, tw, *w, routing, contrib, case["act"])
    return moe.topk_sum(contrib, ids, E)


def _compressed(case, seed):
    """The expert rows of a case, w13 then w2, compressed: (pitch records, LUTs (rows, 2, 512))."""
    g = _gen(seed, 3)
    n, HI = case["rows"], case["H"] * case["I"]
    records, luts = [], []
    for blocks in (2 * HI // GROUP, HI // GROUP):
        raw, _ = _fp8_blocks(g, n, blocks)
        rec, lut, _ = codec.encode_rows(raw, codec.pitch_of(raw.shape[1], PITCH, 4096))
        records.append(rec)
        luts.append(lut)
    return records, torch.stack(luts, dim=1).contiguous()


def _pager(case, seed, layers):
    """A pager with every expert in its RAM tier, its layers loaded and set up."""
    settings = pg.Settings(cache_slots=case["slots"], compress="on" if case["compress"] else "off",
                           pitch_ratio=1.0 if case["compress"] and case["H"] * case["I"] < 1 << 18 else PITCH,
                           working_rows=case["W"], log_interval=0)
    p = pg.Pager(settings, layers, case["E"], case["H"], case["I"], torch.device("cuda"))
    made = []
    for layer in range(layers):
        w13, w13s, w2, w2s = _experts(case, seed + 31 * layer)
        eng = p.add_layer(case["act"])
        p.store.write_rows(layer, "w13_weight", w13.flatten(1))
        p.store.write_rows(layer, "w2_weight", w2.flatten(1))
        eng.setup({"w13_weight_scale_inv": w13s, "w2_weight_scale_inv": w2s})
        made.append(eng)
    return p, made


def _trace_steps(case, seed):
    """Per step and layer (x, weights, ids); half of the steps route as the one before, as decoding does."""
    steps = []
    for layer in range(case["layers"]):
        mine = _tokens(case, seed + 17 * layer, case["steps"])
        for t in range(1, case["steps"], 2):
            mine[t] = (mine[t][0], mine[t][1], mine[t - 1][2])
        steps.append(mine)
    return [[steps[layer][t] for layer in range(case["layers"])] for t in range(case["steps"])]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        w = _experts(case, seed)
        emap = torch.arange(case["E"], dtype=torch.int32, device="cuda")
        steps = _tokens(case, seed, case["layers"])
        graph, out = _capture(lambda: [_step(case, *s, emap, w) for s in steps])
        return {"kind": kind, "graph": graph, "out": out, "keep": (w, emap, steps)}
    if kind == "ffn":
        return {"kind": kind, "w": _experts(case, seed), "x": _tokens(case, seed)[0], "act": case["act"]}
    if kind in ("expand", "expand_ram"):
        records, luts = _compressed(case, seed)
        n, HI = case["rows"], case["H"] * case["I"]
        order = torch.randperm(n, generator=_gen(seed, 4), device="cuda")
        st = {"kind": kind, "todo": torch.arange(n, device="cuda"), "dst_row": order,
              "no_cache": torch.full((n,), -1, dtype=torch.int64, device="cuda"), "lut": luts,
              "dst": [torch.empty((n, k * HI), dtype=torch.uint8, device="cuda") for k in (2, 1)]}
        if kind == "expand":
            st["src"] = records
            return st
        st["src"] = [torch.empty(r.shape, dtype=torch.uint8, pin_memory=True) for r in records]
        for host, r in zip(st["src"], records):
            host.copy_(r)
        st["src_row"] = torch.arange(n, device="cuda")
        g = _gen(seed, 5)
        st["scale"] = [torch.rand((n, k * HI // (B * B)), generator=g, device="cuda") for k in (2, 1)]
        st["scale_dst"] = [torch.empty_like(s) for s in st["scale"]]
        return st
    if kind == "encode":
        raw, _ = _fp8_blocks(_gen(seed, 6), case["rows"], case["groups"])
        # Rows of a few groups do not average the code lengths of larger ones out.
        ratio = PITCH if case["groups"] >= 32 else 1.0
        return {"kind": kind, "raw": raw, "pitch": codec.pitch_of(raw.shape[1], ratio, 4096)}
    if kind == "prefill":
        p, (eng,) = _pager(case, seed, 1)
        # Decode steps before it, so that the cache slots hold experts.
        few = max(1, case["slots"] // case["topk"])
        for x, tw, ids in _tokens({**case, "T": few}, seed + 7, 2):
            eng.forward(x, tw, ids)
        return {"kind": kind, "pager": p, "eng": eng, "x": _tokens(case, seed)[0]}
    if kind == "trace":
        p, engines = _pager(case, seed, case["layers"])
        steps = _trace_steps(case, seed)
        graph, out = _capture(lambda: [e.forward(*s) for step in steps for e, s in zip(engines, step)])
        return {"kind": kind, "graph": graph, "out": out, "pager": p, "engines": engines, "keep": steps}
    raise ValueError(kind)


def run(state):
    kind = state["kind"]
    if kind == "step":
        state["graph"].replay()
        return state["out"]
    if kind == "ffn":
        x, tw, ids = state["x"]
        return moe.fused_moe(x, tw, ids, *state["w"], activation=state["act"])
    if kind == "expand":
        codec.decode_rows(state["todo"], state["dst_row"], state["no_cache"], state["src"], state["dst"],
                          state["lut"])
        return state["dst"]
    if kind == "expand_ram":
        codec.decode_rows_from_ram(state["todo"], state["dst_row"], state["no_cache"], state["src_row"], 0,
                                   state["src"], state["dst"], state["lut"], state["scale"], state["scale_dst"])
        return [state["dst"], state["scale_dst"]]
    if kind == "encode":
        return codec.encode_rows(state["raw"], state["pitch"])
    if kind == "prefill":
        return state["eng"].forward(*state["x"])
    state["graph"].replay()
    return {"out": state["out"], "slot_of": [e.table.slot_of for e in state["engines"]]}


# ---- work and tolerance ----


def _row_bytes(case, values):
    """Bytes of an expansion or compression of ``values`` fp8 values: raw, nibbles, Huffman words of about 2.7 bits."""
    return values * (1 + 0.5 + 2.7 / 8)


def _touched(case, T):
    """Experts that T tokens reach, on average, if routing is even."""
    E = case["E"]
    return E * (1.0 - (1.0 - min(1.0, case["topk"] / E)) ** T)


def _ffn_work(case, T, times=1):
    H, I, topk = case["H"], case["I"], case["topk"]
    weights = _touched(case, T) * (3 * H * I + 12 * H * I / (B * B))
    return {"bytes": times * (weights + 2 * T * 2 * H + 12 * T * topk), "flops": times * 6.0 * T * topk * H * I}


def work(case):
    kind = case["kind"]
    if kind == "step":
        return _ffn_work(case, case["T"], case["layers"])
    if kind == "ffn":
        return _ffn_work(case, case["T"])
    if kind in ("expand", "expand_ram"):
        return {"bytes": _row_bytes(case, 3 * case["rows"] * case["H"] * case["I"]), "flops": 0}
    if kind == "encode":
        return {"bytes": _row_bytes(case, case["rows"] * case["groups"] * GROUP), "flops": 0}
    if kind == "prefill":
        return _ffn_work(case, case["T"])
    return _ffn_work(case, case["T"], case["layers"] * case["steps"])


def tolerance(case):
    """Bytes are exact. Of the FFN, the order of a block's fp8 products differs between
    implementations, so a gate, up or activation value at a rounding boundary moves to its bf16
    or fp8 neighbour, which is up to 1/16 of a value away, or takes its whole scale group along.
    Activations are heavy-tailed: one large value that moves is 2-3% of a single token's output
    (measured against 64-bit sums: 0.2% where none moves, 1.2-3% where one does)."""
    if case["kind"] in ("expand", "expand_ram", "encode"):
        return "exact"
    return {"rel": 0.03, "max": 0.5}


# ---- 64-bit results ----


def _quant64(v):
    """Values (n, K) rounded to fp8 per 128-column group as the format has it, in 64 bits."""
    n, K = v.shape
    b = v.float().view(n, K // B, B)
    s = b.abs().amax(dim=2, keepdim=True).clamp_min(1e-10) / 448.0
    return ((b / s).clamp(-448, 448).to(torch.float8_e4m3fn).double() * s.double()).view(n, K)


def _matrix64(q, s):
    n, k = q.shape
    v = q.view(torch.float8_e4m3fn).double().view(n // B, B, k // B, B)
    return (v * s.double()[:, None, :, None]).view(n, k)


def _ffn64(case, x, tw, ids, w):
    """The w8a8 expert FFN with its roundings to fp8 and bf16 kept and every sum in 64 bits."""
    w13, w13s, w2, w2s = w
    I = case["I"]
    xd = _quant64(x)
    out = torch.zeros(x.shape, dtype=torch.float64, device=x.device)
    for e in torch.unique(ids).tolist():
        t, k = (ids == e).nonzero(as_tuple=True)
        h = (xd[t] @ _matrix64(w13[e], w13s[e]).T).bfloat16().double()
        g, u = h[:, :I], h[:, I:]
        a = g / (1 + torch.exp(-g)) if case["act"] == "silu" else g * 0.5 * (1 + torch.erf(g / math.sqrt(2.0)))
        y = _quant64((a.bfloat16().double() * u).bfloat16()) @ _matrix64(w2[e], w2s[e]).T
        out.index_add_(0, t, y * tw[t, k].double()[:, None])
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        w = _experts(case, seed)
        return [_ffn64(case, *s, w) for s in _tokens(case, seed, case["layers"])]
    if kind in ("ffn", "prefill"):
        return _ffn64(case, *_tokens(case, seed)[0], _experts(case, seed))
    if kind == "trace":
        w = [_experts(case, seed + 31 * layer) for layer in range(case["layers"])]
        out = [_ffn64(case, *s, w[layer]) for step in _trace_steps(case, seed) for layer, s in enumerate(step)]
        return {"out": out, "slot_of": [None] * case["layers"]}
    return None  # bytes: the same or wrong
