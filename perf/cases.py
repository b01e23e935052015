"""Timed cases of the W4A16 grouped-expert MoE path.

Each case is one call that a serving program makes for one MoE layer, through
the package's public entry points:

  * "experts": ``fused_experts_w4a16`` on activations and a finished routing;
  * "layer":   ``W4A16MoELayer``, the router step and the experts;
  * "routing": ``router_topk_softmax`` and ``moe_align_block_size``, for a
               program that runs expert kernels of its own.

The layer of the benchmark has E=256 experts, top-10 routing, hidden K=3072,
intermediate N=1024 and int4 weights in groups of 32.  Beside it stand the
shapes one GPU holds when that layer is split over eight (N=128 of every
expert, or 32 of the experts), and generic layers with the larger groups and
with sizes that are not multiples of 256.
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

from __graft_entry__ import load_package

DEVICE = "cuda:0"
SKEW_STD = 1.5  # per-expert logit bias of skewed routing

LAYER = dict(E=256, topk=10, K=3072, N=1024, group=32)


def _case(name, M, *, kind="experts", skewed=False, local=1, ids="int32", **shape):
    """`local` > 1: the GPU holds the first E of local * E experts; the router
    picks among all of them and the pairs of the others carry the id -1."""
    c = dict(LAYER)
    c.update(shape)
    c.update(name=name, kind=kind, M=M, skewed=skewed, local=local, ids=ids)
    return c


def listed():
    return [
        # One user decoding one token: latency, 10 experts' weights.
        _case("decode_1", 1),
        # A decode step of a small server (the benchmark's headline batch).
        _case("decode_16", 16),
        # A decode step of a busy server, with the uneven expert load of real
        # routers: a few hot experts, most with one to four tokens.
        _case("decode_64_skewed", 64, skewed=True),
        # A large decode batch, or a short prompt: about ten tokens an expert.
        _case("batch_250", 250),
        # A prefill chunk that does not fill its size.
        _case("prefill_1000", 1000),
        # A full prefill chunk.
        _case("prefill_4096", 4096),
        # The same layer split over eight GPUs by its intermediate size.
        _case("slice_prefill_2048", 2048, N=128),
        # ... and by its experts: most pairs belong to other GPUs.
        _case("local_experts_1500", 1500, E=32, local=8, skewed=True),
        # Another layer, whose intermediate size is no multiple of 256, with
        # one scale per 128 elements and the router's int64 ids.
        _case("ragged_prefill_777", 777, E=64, topk=6, K=2048, N=1408, group=128, ids="int64"),
        # A decode step of a smaller layer.
        _case("small_decode_12", 12, E=64, topk=8, K=2048, N=768, group=64),
        # The whole step from the router's logits, few tokens.
        _case("layer_step_4", 4, kind="layer"),
        # Routing and sorting a prefill chunk.
        _case("routing_4096", 4096, kind="routing"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["experts"] * 8 + ["layer", "routing"])
    skewed = rng.random() < 0.35
    ids = rng.choice(["int32", "int32", "int64"])
    local = 1
    form = rng.choice(["layer", "layer", "slice", "local", "other", "other"])
    s = dict(LAYER)
    if form == "slice":
        s["N"] = rng.choice([128, 256, 512])
    elif form == "local" and kind == "experts":
        local = rng.choice([2, 4, 8])
        s["E"] = 256 // local
    elif form == "other":
        s["group"] = rng.choice([32, 64, 128])
        s["E"] = rng.choice([8, 16, 32, 60, 64, 128, 160])
        s["topk"] = rng.choice([2, 4, 6, 8])
        unit = max(64, s["group"])
        s["K"] = unit * rng.randint(1024 // unit, 4096 // unit)
        s["N"] = unit * rng.randint(256 // unit, 2048 // unit)
    M = _log_int(rng, 1, 4096)
    # no dearer than the largest listed case
    top = 4096 * LAYER["topk"] * LAYER["K"] * LAYER["N"]
    M = max(1, min(M, top // (s["topk"] * s["K"] * s["N"])))
    return dict(s, kind=kind, M=M, skewed=skewed, local=local, ids=ids)


# ---- inputs -----------------------------------------------------------------


def _gen(seed, salt):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed * 1000003 + salt)
    return g


def _logits(case, seed):
    M, E = case["M"], case["E"] * case["local"]
    x = torch.randn((M, E), generator=_gen(seed, 1), device=DEVICE)
    if case["skewed"]:
        x += torch.randn((E,), generator=_gen(seed, 2), device=DEVICE) * SKEW_STD
    return x


def _routing(case, seed):
    """(weights fp32, ids) of the top-k of the logits; pairs of experts on
    other GPUs get the id -1."""
    vals, ids = torch.topk(_logits(case, seed), case["topk"], dim=-1)
    w = torch.softmax(vals, dim=-1)
    if case["local"] > 1:
        ids = torch.where(ids < case["E"], ids, -1)
    return w.contiguous(), ids.to(getattr(torch, case["ids"])).contiguous()


def _weights(case, seed):
    E, K, N, G = case["E"], case["K"], case["N"], case["group"]
    g = _gen(seed, 3)

    def packed(rows, cols):  # uniform int4 codes, eight to a word
        return torch.randint(0, 256, (E, rows, cols // 2), generator=g, device=DEVICE,
                             dtype=torch.uint8).view(torch.int32)

    def scales(rows, cols):
        s = torch.rand((E, rows, cols // G), generator=g, device=DEVICE)
        return (s * 0.015 + 0.005).to(torch.bfloat16)

    return packed(2 * N, K), packed(K, N), scales(2 * N, K), scales(K, N)


def _hidden(case, seed):
    x = torch.randn((case["M"], case["K"]), generator=_gen(seed, 4), device=DEVICE)
    return x.to(torch.bfloat16)


def prepare(case, seed):
    moe = load_package()
    st = {"moe": moe, "kind": case["kind"], "topk": case["topk"], "E": case["E"],
          "group": case["group"]}
    if case["kind"] == "routing":
        st["logits"] = _logits(case, seed)
        return st
    w13, w2, s13, s2 = _weights(case, seed)
    st["x"] = _hidden(case, seed)
    if case["kind"] == "layer":
        st["logits"] = _logits(case, seed)
        weights = moe.MoELayerWeights(w13=w13, w2=w2, s13=s13, s2=s2, group_size=case["group"])
        st["layer"] = moe.W4A16MoELayer(weights, case["topk"])
    else:
        st["w"] = (w13, w2, s13, s2)
        st["tw"], st["ids"] = _routing(case, seed)
    return st


def run(state):
    moe = state["moe"]
    if state["kind"] == "routing":
        w, ids = moe.router_topk_softmax(state["logits"], state["topk"])
        sorted_ids, expert_ids, num_post = moe.moe_align_block_size(ids, 16, state["E"])
        return w, ids, sorted_ids, expert_ids, num_post
    if state["kind"] == "layer":
        return state["layer"](state["x"], state["logits"])
    w13, w2, s13, s2 = state["w"]
    return moe.fused_experts_w4a16(state["x"], w13, w2, s13, s2, state["tw"], state["ids"],
                                   state["group"])


# ---- what a pass cannot do without --------------------------------------------


@functools.lru_cache(maxsize=None)
def _routed(M, E_all, E, topk, skewed):
    """(experts with a routed pair, routed pairs) of one sample routing."""
    rng = np.random.default_rng(0)
    x = rng.standard_normal((M, E_all), dtype=np.float32)
    if skewed:
        x += (rng.standard_normal(E_all) * SKEW_STD).astype(np.float32)
    ids = np.argpartition(-x, topk - 1, axis=1)[:, :topk]
    here = ids[ids < E]
    return int(np.unique(here).size), int(here.size)


def work(case):
    M, E, topk, K, N = (case[k] for k in ("M", "E", "topk", "K", "N"))
    id_bytes = 8 if case["ids"] == "int64" else 4
    if case["kind"] == "routing":
        slots = (M * topk + E * 15 + 15) // 16 * 16  # the sorted list, padded per expert
        return {"bytes": M * E * 4 + M * topk * 8 + slots * 4 + slots // 16 * 4 + 4, "flops": 0}
    touched, pairs = _routed(M, E * case["local"], E, topk, case["skewed"])
    elems = 3 * N * K  # weights of one expert
    expert_bytes = elems // 2 + elems // case["group"] * 2
    nbytes = touched * expert_bytes + 2 * M * K * 2
    nbytes += M * E * 4 if case["kind"] == "layer" else M * topk * (4 + id_bytes)
    return {"bytes": nbytes, "flops": 2 * pairs * elems}


def tolerance(case):
    if case["kind"] == "routing":
        # fp32 softmax weights; ids and sort are whole numbers
        return {"rel": 1e-6, "max": 1e-5}
    # bf16 activations between the two products, bf16 weighted rows, bf16 out:
    # 2.3e-3 to 3.7e-3 of the result's norm against 64 bits.
    return {"rel": 1e-2, "max": 8e-2}


# ---- the same in 64 bits --------------------------------------------------------


def _dequant64(packed, scale, group):
    """(code - 8) * scale of one expert's rows, code i of a word in bits 4i."""
    shifts = torch.arange(0, 32, 4, device=packed.device, dtype=torch.int32)
    codes = (packed.unsqueeze(-1) >> shifts) & 0xF
    rows = packed.shape[0]
    w = (codes - 8).reshape(rows, -1, group).to(torch.float64)
    return (w * scale.to(torch.float64).unsqueeze(-1)).reshape(rows, -1)


def _exact_experts(case, seed, tw, ids):
    w13, w2, s13, s2 = _weights(case, seed)
    x = _hidden(case, seed).to(torch.float64)
    N, G, topk = case["N"], case["group"], case["topk"]
    out = torch.zeros((case["M"], case["K"]), dtype=torch.float64, device=DEVICE)
    flat = ids.reshape(-1).long()
    w_flat = tw.reshape(-1).to(torch.float64)
    for e in torch.unique(flat[flat >= 0]).tolist():
        at = torch.nonzero(flat == e).reshape(-1)
        rows = at // topk
        y = x[rows] @ _dequant64(w13[e], s13[e], G).T
        h = torch.nn.functional.silu(y[:, :N]) * y[:, N:]
        out.index_add_(0, rows, (h @ _dequant64(w2[e], s2[e], G).T) * w_flat[at].unsqueeze(1))
    return out


def exact(case, seed):
    topk = case["topk"]
    if case["kind"] == "experts":
        return _exact_experts(case, seed, *_routing(case, seed))
    vals, ids = torch.topk(_logits(case, seed).to(torch.float64), topk, dim=-1)
    tw = torch.softmax(vals, dim=-1)
    if case["kind"] == "layer":
        return _exact_experts(case, seed, tw, ids)
    E, block = case["E"], 16
    flat = ids.reshape(-1)
    counts = torch.bincount(flat, minlength=E)
    padded = (counts + block - 1) // block * block
    ends = torch.cumsum(padded, 0)
    size = (flat.numel() + E * (block - 1) + block - 1) // block * block
    order = torch.argsort(flat, stable=True)
    experts = flat[order]
    first = torch.cumsum(counts, 0) - counts
    place = (ends - padded)[experts] + torch.arange(flat.numel(), device=DEVICE) - first[experts]
    sorted_ids = torch.full((size,), flat.numel(), dtype=torch.int32, device=DEVICE)
    sorted_ids[place] = order.to(torch.int32)
    starts = torch.arange(size // block, device=DEVICE) * block
    blocks = torch.searchsorted(ends, starts, right=True)
    expert_ids = torch.where(starts < ends[-1], blocks, -1).to(torch.int32)
    return tw, ids.to(torch.int32), sorted_ids, expert_ids, ends[-1:].to(torch.int32)
