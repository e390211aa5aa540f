"""Performance cases of the W4A16 MoE path: the work that a program using this package has it do.

A case is a dict of plain values. `prepare` makes what such a program holds before the call (expert
stacks, router, hidden states, a captured decode graph), `run` makes one pass through the public
entry points, `work` states the bytes and operations that the pass cannot do without, and `exact`
gives the same outputs in 64 bits with plain torch.

Kinds:
  step     a decode step of a layer stack: residual add + RMSNorm + MoE layer, each layer's input the
           previous one's output, captured once in a graph and replayed (the decode loop of a server)
  decode   the MoE layers of a decode step at their own hidden states, captured and replayed alike
  routed   the same with the routing given by the caller (a router of the caller's own)
  layer    one MoE layer called eagerly: chunked prefill and prefill batches
  dequant  a projection's int4 stack to dense weights (the reference's dequantise entry point)
  awq      a projection of an AWQ checkpoint repacked to the GPTQ layout (loading a model)
  hr       the hidden-residual predictor: the experts to prefetch for (layer, token) examples
  heads    the per-layer MLP predictor: the experts to prefetch, one head per layer

The decode kinds run several layers per pass, so that the weights of a pass and of the states that
are used in turn do not stay in the 256 MB cache behind the HBM: each layer of a model finds its
weights in HBM. Offloaded decoding (experts in host memory) is left out: its time is the host link's
and the host's waits; its device work is the decode and predictor kinds.

Shapes: hidden 2048, 256 experts of intermediate size 512, top-8, group 128 with router logits
skewed to Zipf(1.1) per layer (the package's synthetic model), and generic ones.
"""

from __future__ import annotations

import math

import torch

from mtp_amd import ops, synth
from mtp_amd.awq import awq_to_gptq
from mtp_amd.moe import MoeBlock
from mtp_amd.predictor import HiddenResidualExpertPredictor

BASE = {"hidden": 2048, "inter": 512, "experts": 256, "top_k": 8, "group": 128}
AWQ_ORDER = (0, 2, 4, 6, 1, 3, 5, 7)


def _moe(name: str, kind: str, tokens: int, **more) -> dict:
    return {"name": name, "kind": kind, "tokens": tokens, "layers": 1, "shared": False,
            **BASE, **more}


def listed() -> list[dict]:
    return [
        # one user's decode step through a stack of layers: the smallest call, all latency
        _moe("step_1", "step", 1, layers=8),
        # a small serving batch
        _moe("decode_8", "decode", 8, layers=8),
        # a serving batch of a model with a sigmoid-gated shared expert
        _moe("decode_shared_32", "decode", 32, layers=8, shared=True),
        # the largest batch of the decode benchmark
        _moe("decode_64", "decode", 64, layers=8),
        # a caller's own routing, on a smaller model with finer quantisation groups
        _moe("routed_48", "routed", 48, layers=8, hidden=1024, inter=256, experts=64, top_k=4,
             group=64),
        # a large decode batch or a short prompt: between the two benchmark sizes, not a multiple
        # of any tile
        _moe("layer_203", "layer", 203),
        # prefill of the benchmark's prompt
        _moe("layer_2048", "layer", 2048),
        # the largest prefill chunk
        _moe("layer_8192", "layer", 8192),
        # dense bf16 weights of part of a layer's gate projections, as a dense fallback holds them
        {"name": "dequant_64", "kind": "dequant", "experts": 64, "hidden": 2048, "inter": 512,
         "group": 128, "linear": True, "dtype": "bfloat16", "g_idx": False},
        # one projection of one layer while an AWQ checkpoint is loaded
        {"name": "awq_wna16_256", "kind": "awq", "experts": 256, "hidden": 2048, "inter": 512,
         "group": 128, "layout": "wna16", "zeros": True, "bf16_scales": False},
        # prefetch of 40 layers for a batch of 4 tokens, by either predictor
        {"name": "hr_160", "kind": "hr", "examples": 160, "hidden": 2048, "experts": 256,
         "layers": 40, "width": 256, "window": 4, "top_k": 16},
        {"name": "heads_4", "kind": "heads", "tokens": 4, "hidden": 2048, "experts": 256,
         "layers": 40, "width": 1024, "top_k": 16},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def _shape(rng) -> dict:
    """The package's model in half of the draws, a generic one otherwise."""
    if rng.random() < 0.5:
        return dict(BASE)
    top_k = rng.choice((1, 2, 4, 6, 8))
    return {"hidden": rng.choice((512, 1024, 1536, 2048)), "inter": rng.choice((256, 512, 1024)),
            "experts": max(16, 4 * _log_int(rng, 4, 64)), "top_k": top_k,
            "group": rng.choice((64, 128, 256))}


def draw(rng) -> dict:
    kind = rng.choices(("step", "decode", "routed", "layer", "dequant", "awq", "hr", "heads"),
                       (3, 6, 3, 7, 2, 2, 1, 1))[0]
    if kind in ("step", "decode", "routed"):
        shape = _shape(rng)
        return {"kind": kind, "tokens": _log_int(rng, 1, 64), "layers": 8,
                "shared": kind != "routed" and rng.random() < 0.4, **shape}
    if kind == "layer":
        shape = _shape(rng)
        # no more multiplications than the largest listed prefill
        cap = 8192 * 8 * 2048 * 512 // (shape["top_k"] * shape["hidden"] * shape["inter"])
        return {"kind": kind, "tokens": _log_int(rng, 65, min(8192, cap)), "layers": 1,
                "shared": rng.random() < 0.4, **shape}
    hidden, inter = rng.choice(((2048, 512), (1024, 512), (512, 2048), (2048, 1024)))
    if kind == "dequant":
        return {"kind": kind, "experts": _log_int(rng, 1, 128), "hidden": hidden, "inter": inter,
                "group": rng.choice((64, 128)), "linear": rng.random() < 0.6,
                "dtype": rng.choice(("bfloat16", "bfloat16", "float16", "float32")),
                "g_idx": rng.random() < 0.25}
    if kind == "awq":
        layout = rng.choice(("wna16", "wna16", "awq"))
        return {"kind": kind, "experts": _log_int(rng, 4, 256), "hidden": hidden, "inter": inter,
                "group": rng.choice((64, 128)), "layout": layout,
                "zeros": layout == "awq" or rng.random() < 0.6,
                "bf16_scales": layout == "wna16" and rng.random() < 0.5}
    if kind == "hr":
        return {"kind": kind, "examples": _log_int(rng, 1, 640), "hidden": 2048, "experts": 256,
                "layers": 40, "width": rng.choice((128, 256, 512)), "window": rng.choice((1, 4, 8)),
                "top_k": rng.choice((8, 16, 32))}
    return {"kind": kind, "tokens": _log_int(rng, 1, 16), "hidden": 2048, "experts": 256,
            "layers": rng.choice((8, 20, 40)), "width": rng.choice((512, 1024)),
            "top_k": rng.choice((8, 16, 32))}


# ------------------------------------------------------------------------------ inputs
def _gen(seed: int, salt: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1009 + salt)
    return g


def _randn(shape, g: torch.Generator, scale: float = 1.0) -> torch.Tensor:
    return (torch.randn(shape, generator=g, device="cuda") * scale).to(torch.bfloat16)


def _moe_layers(case: dict, seed: int) -> list[synth.SyntheticLayer]:
    """The synthetic layers of the package (uniform int4 weights and zero points, fp16 scales,
    Zipf-skewed routing); layer l of seed s takes the package's seeds of layer 64 s + l."""
    return [synth.make_layer(64 * (int(seed) % (1 << 20)) + l, num_experts=case["experts"],
                             hidden=case["hidden"], intermediate=case["inter"], zipf=True,
                             shared=case["shared"], group=case["group"], device="cuda")
            for l in range(case["layers"])]


def _given_routing(case: dict, layer: synth.SyntheticLayer, x: torch.Tensor):
    """A caller's routing: top-k of its own softmax, renormalised."""
    logits = x.float() @ layer.router_w.float().T + layer.logit_bias
    w, ids = torch.softmax(logits, dim=-1).topk(case["top_k"], dim=-1)
    return ids.to(torch.int32), (w / w.sum(dim=-1, keepdim=True)).contiguous()


def _graph(fn):
    """fn captured in a graph after one eager call, and fn's outputs in the graph's memory."""
    fn()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = fn()
    return g, out


def _inputs(case: dict, seed: int) -> dict:
    kind, H = case["kind"], case["hidden"]
    g = _gen(seed, 7)
    if kind in ("step", "decode", "routed", "layer"):
        T, L = case["tokens"], case["layers"]
        s = {"layers": _moe_layers(case, seed)}
        if kind == "step":
            s["res"], s["add"] = _randn((T, H), g), _randn((T, H), g)
            s["norm_w"] = [_randn((H,), g, 0.1) for _ in range(L)]
        else:
            s["x"] = [_randn((T, H), g) for _ in range(L)]
        if kind == "routed":
            s["routing"] = [_given_routing(case, ly, x) for ly, x in zip(s["layers"], s["x"])]
        return s
    if kind in ("dequant", "awq"):
        E, N, G = case["experts"], case["inter"], case["group"]
        p = synth.make_projection(E, H, N, g, "cuda", G)
        if kind == "dequant":
            gi = None
            if case["g_idx"]:  # act-order: a permutation of the group of each input row
                k = torch.arange(H, device="cuda")
                gi = (k[torch.randperm(H, generator=g, device="cuda")] // G).to(torch.int32)
                gi = gi.expand(E, H).contiguous()
            return {"qweight": p.qweight, "qzeros": p.qzeros, "scales": p.scales, "g_idx": gi}
        if case["layout"] == "wna16":
            # bytes [E, N, K/2], zero points [E, N/2, K/G], scales [E, N, K/G]
            scales = p.scales.transpose(1, 2).contiguous()
            return {"qweight": p.qweight.transpose(1, 2).contiguous().view(torch.uint8),
                    "qzeros": (torch.randint(0, 256, (E, N // 2, H // G), dtype=torch.uint8,
                                             generator=g, device="cuda")
                               if case["zeros"] else None),
                    # the bf16 scales of such checkpoints are exact in fp16
                    "scales": scales.bfloat16() if case["bf16_scales"] else scales}
        shape = (E, H, N // 8)
        return {"qweight": synth._rand_u32_as_i32(shape, g, "cuda"), "qzeros": p.qzeros,
                "scales": p.scales}
    L, W, E = case["layers"], case["width"], case["experts"]
    if kind == "hr":
        n = case["examples"]
        model = HiddenResidualExpertPredictor(
            hidden_size=H, num_experts=E, num_layers=L, future_window=case["window"], width=W,
            seed=int(seed), device="cuda")
        return {"model": model, "x": _randn((n, H), g),
                "layer_ids": torch.arange(n, device="cuda", dtype=torch.int32) % L,
                "prior": torch.randn((n, case["window"], E), generator=g, device="cuda")}
    return {"x": _randn((case["tokens"], H), g), "w1": _randn((L, W, H), g, 0.02),
            "w2": _randn((L, E, W), g, 0.03)}


def prepare(case: dict, seed: int) -> dict:
    s = {"case": case, **_inputs(case, seed)}
    kind, k = case["kind"], case.get("top_k")
    if kind == "step":
        def step():
            res, add, outs = s["res"], s["add"], []
            for ly, nw in zip(s["layers"], s["norm_w"]):
                add, res, _ = ops.norm_layer(res, ly.router_w, ly.experts, nw, add=add, top_k=k,
                                             logit_bias=ly.logit_bias, shared=ly.shared,
                                             shared_gate_w=ly.shared_gate_w)
                outs.append(add)
            return {"out": outs, "res": res}
        s["graph"], s["outs"] = _graph(step)
    elif kind in ("decode", "layer"):
        s["blocks"] = [MoeBlock(ly.experts, ly.router_w, shared_expert=ly.shared,
                                shared_expert_gate_weight=ly.shared_gate_w, top_k=k,
                                logit_bias=ly.logit_bias) for ly in s["layers"]]
        if kind == "decode":
            s["graph"], s["outs"] = _graph(
                lambda: [b(x) for b, x in zip(s["blocks"], s["x"])])
    elif kind == "routed":
        s["graph"], s["outs"] = _graph(
            lambda: [ops.fused_experts(x, ids, w, ly.experts)
                     for ly, x, (ids, w) in zip(s["layers"], s["x"], s["routing"])])
    return s


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if "graph" in state:
        state["graph"].replay()
        return state["outs"]
    if kind == "layer":
        return [b(x) for b, x in zip(state["blocks"], state["x"])]
    if kind == "dequant":
        return ops.dequantize(state["qweight"], state["qzeros"], state["scales"], state["g_idx"],
                              group_size=case["group"], linear_weight=case["linear"],
                              dtype=getattr(torch, case["dtype"]))
    if kind == "awq":
        st = awq_to_gptq(state["qweight"], state["qzeros"], state["scales"],
                         layout=case["layout"], in_features=case["hidden"],
                         group_size=case["group"])
        return {"qweight": st.qweight, "qzeros": st.qzeros, "scales": st.scales}
    if kind == "hr":
        ids, logits = state["model"].predict_topk(state["x"], layer_ids=state["layer_ids"],
                                                  k=case["top_k"], prior=state["prior"],
                                                  return_logits=True)
        return {"ids": ids, "logits": logits}
    return ops.predictor_topk(state["x"], state["w1"], state["w2"], case["top_k"])


# ------------------------------------------------------------------------------ work
def _distinct(case: dict) -> float:
    """Expected distinct routed experts of a layer: a draw of the skewed router's logits (x . w has
    a standard deviation of 0.02 sqrt(hidden))."""
    g = torch.Generator().manual_seed(5)
    T, E = case["tokens"], case["experts"]
    logits = torch.randn((T, E), generator=g) * (0.02 * math.sqrt(case["hidden"]))
    ids = (logits + synth.zipf_logit_bias(E, seed=5)).topk(case["top_k"], dim=-1).indices
    return float(ids.unique().numel())


def work(case: dict) -> dict:
    kind, H = case["kind"], case["hidden"]
    if kind in ("step", "decode", "routed", "layer"):
        T, E, I, k = case["tokens"], case["experts"], case["inter"], case["top_k"]
        sh = int(case["shared"])
        expert = synth.expert_bytes(H, I, case["group"])
        b = (_distinct(case) + sh) * expert + 2 * T * H * 2
        f = 2 * T * (k + sh) * 3 * H * I
        if kind != "routed":
            b += (E + sh) * H * 2
            f += 2 * T * (E + sh) * H
        else:
            b += T * k * 8
        if kind == "step":
            b += 3 * T * H * 2 + H * 2
        return {"bytes": case["layers"] * b, "flops": case["layers"] * f}
    if kind in ("dequant", "awq"):
        E, N, G = case["experts"], case["inter"], case["group"]
        packed = E * (H * N // 2)
        zeros, scales = E * (H // G) * (N // 2), E * (H // G) * N * 2
        if kind == "dequant":
            size = 4 if case["dtype"] == "float32" else 2
            idx = E * H * 4 if case["g_idx"] else 0
            return {"bytes": packed + zeros + scales + idx + E * H * N * size,
                    "flops": 2 * E * H * N}
        return {"bytes": 2 * (packed + scales) + zeros * (2 if case["zeros"] else 1), "flops": 0}
    L, W, E = case["layers"], case["width"], case["experts"]
    if kind == "hr":
        n, F = case["examples"], case["window"]
        return {"bytes": n * H * 2 + W * H * 2 + E * W * 2 + 2 * n * F * E * 4
                + n * F * case["top_k"] * 4,
                "flops": 2 * n * W * H + 2 * n * F * E * W}
    T = case["tokens"]
    return {"bytes": L * (W * H + E * W) * 2 + T * H * 2 + L * T * case["top_k"] * 4,
            "flops": 2 * T * L * (W * H + E * W)}


def tolerance(case: dict):
    kind = case["kind"]
    if kind in ("dequant", "awq", "heads"):
        return "exact"  # moved bits, or one rounding of an exact product; expert ids
    if kind == "hr":
        # fp32 sums of bf16 products; a last-bit change of an activation moves a logit
        return {"rel": 2e-3, "max": 5e-2, "differ": 5e-3}
    if kind == "step":
        # a bf16 rounding in one layer travels through the norms and routers of the later ones
        return {"rel": 3e-2, "max": 5e-1}
    # bf16 outputs and bf16 activations between the two products; the kernels hold the weights
    # either unrounded or rounded to bf16
    return {"rel": 1e-2, "max": 1e-1}


# ------------------------------------------------------------------------------ 64 bits
def _nibbles(words: torch.Tensor, dim: int) -> torch.Tensor:
    """The eight nibbles of each int32 word along `dim`, low nibble first."""
    v = torch.stack([(words >> (4 * j)) & 0xF for j in range(8)], dim=dim + 1)
    shape = list(words.shape)
    shape[dim] *= 8
    return v.reshape(shape)


def _dense(qweight, qzeros, scales, group: int, g_idx=None) -> torch.Tensor:
    """[K, N] in 64 bits: (q - z) * s."""
    q, z = _nibbles(qweight, 0).double(), _nibbles(qzeros, 1).double()
    g = (torch.arange(q.shape[0], device=q.device) // group) if g_idx is None else g_idx.long()
    return (q - z[g]) * scales.double()[g]


def _expert(experts, e: int, x: torch.Tensor) -> torch.Tensor:
    w = [_dense(p.qweight[e], p.qzeros[e], p.scales[e], experts.group_size)
         for p in (experts.gate, experts.up, experts.down)]
    return (torch.nn.functional.silu(x @ w[0]) * (x @ w[1])) @ w[2]


def _moe_exact(layer, x: torch.Tensor, top_k: int, routing=None) -> torch.Tensor:
    x = x.double()
    if routing is None:
        logits = x @ layer.router_w.double().T + layer.logit_bias.double()
        v, ids = logits.topk(top_k, dim=-1)
        w = torch.softmax(v, dim=-1)
    else:
        ids, w = routing[0].long(), routing[1].double()
    out = torch.zeros_like(x)
    for e in ids.unique().tolist():
        t, slot = (ids == e).nonzero(as_tuple=True)
        out.index_add_(0, t, w[t, slot, None] * _expert(layer.experts, e, x[t]))
    if layer.shared is not None:
        gate = torch.sigmoid(x @ layer.shared_gate_w.double().reshape(-1, 1))
        out += gate * _expert(layer.shared, 0, x)
    return out


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "heads":
        return None  # expert ids
    s = _inputs(case, seed)
    if kind == "step":
        # the first layer's input is rounded as the residual stream is; the later layers' inputs
        # carry the roundings before them
        res = (s["res"].float() + s["add"].float()).to(torch.bfloat16)
        r = res.double()
        x = r * torch.rsqrt(r.square().mean(dim=-1, keepdim=True) + 1e-6)
        x = (x * (1 + s["norm_w"][0].double())).to(torch.bfloat16)
        first = _moe_exact(s["layers"][0], x, case["top_k"])
        return {"out": [first] + [None] * (case["layers"] - 1), "res": None}
    if kind in ("decode", "layer"):
        return [_moe_exact(ly, x, case["top_k"]) for ly, x in zip(s["layers"], s["x"])]
    if kind == "routed":
        return [_moe_exact(ly, x, case["top_k"], r)
                for ly, x, r in zip(s["layers"], s["x"], s["routing"])]
    if kind == "dequant":
        out = torch.stack([
            _dense(s["qweight"][e], s["qzeros"][e], s["scales"][e], case["group"],
                   None if s["g_idx"] is None else s["g_idx"][e])
            for e in range(case["experts"])])
        return out.transpose(1, 2).contiguous() if case["linear"] else out
    if kind == "awq":
        # integers have no 64-bit value of their own: the scales only
        sc = s["scales"].double()
        return {"qweight": None, "qzeros": None,
                "scales": sc.transpose(1, 2).contiguous() if case["layout"] == "wna16" else sc}
    m, F = s["model"], torch.nn.functional
    d = lambda t: t.double()  # noqa: E731
    a = F.silu(d(s["x"]) @ d(m.enc_w).T + d(m.enc_b))
    c = F.layer_norm(a, (case["width"],), d(m.ln_w), d(m.ln_b), m.ln_eps)
    c = (c + d(m.layer_emb)[s["layer_ids"].long()])[:, None, :] + d(m.delta_emb)[None]
    return {"ids": None, "logits": d(s["prior"]) + F.silu(c) @ d(m.cls_w).T + d(m.cls_b)}
