"""The work that programs on this framework do, as cases that can be timed.

Each case is one pass through a public entry point:
  layer   HomeSeekMoEEngine._forward_ffn: the router (or a hash layer's token
          table), the routed FP4 experts and the FP8 shared expert of one layer
  routed  FusedMoEFFN.forward_table: the routed experts with given ids, E8M0
          or fp32 scales, fp32 results beside the bf16 ones
  loader  FusedMoEFFN.forward: the same through the caller's expert loader
  shared  SharedExpertFFN.forward: one expert of bf16 weights
  logits  ops.lm_head_accept: logits, argmax and draft acceptance
  verify  HomeSeekMoEEngine._mtp_verify_batched: one verify of a small stack
Sizes are those of MoEConfig (hidden 4096, expert 2048, 256 experts, top 6,
vocabulary 129,280) and, among the drawn ones, smaller generic ones.
"""
import math

import numpy as np
import torch

import __graft_entry__

__graft_entry__.package()

from home_seek_amd import ops, synthetic  # noqa: E402
from home_seek_amd.engine import HomeSeekMoEEngine  # noqa: E402
from home_seek_amd.expert_store import HbmExpertStore  # noqa: E402
from home_seek_amd.fused_moe import FusedMoEFFN, SharedExpertFFN  # noqa: E402
from home_seek_amd.model_config import MoEConfig  # noqa: E402
from home_seek_amd.stack import build_stack  # noqa: E402

DEVICE = "cuda"
VOCAB = 129280
LIMIT = 10.0
SCALING = 1.5
BF16 = torch.bfloat16


def _layer(name, batch, t, d=4096, i=2048, experts=256, k=6, hashed=False):
    return {"name": name, "kind": "layer", "batch": batch, "t": t, "d": d, "i": i, "experts": experts, "k": k,
            "hashed": hashed}


def listed():
    return [
        _layer("layer_1", 1, 1),          # one token of one sequence: plain decode, latency bound
        _layer("layer_3", 1, 3),          # verify of a token and two drafts
        _layer("layer_8", 8, 1),          # eight sequences decoding together
        _layer("layer_32", 32, 1),        # a larger batch of sequences, or a short question
        _layer("layer_509", 1, 509),      # a prompt of ragged length
        _layer("layer_4096", 1, 4096),    # a long prompt (or a chunk of one)
        # prefill with a skewed popularity of the experts, fp32 results asked for
        {"name": "routed_zipf_512", "kind": "routed", "m": 512, "d": 4096, "i": 2048, "experts": 256, "k": 6,
         "zipf": 1.1, "scales": "e8m0"},
        # an engine that keeps its experts itself and hands them over one by one, with fp32 scales
        {"name": "loader_f32_24", "kind": "loader", "m": 24, "d": 4096, "i": 2048, "experts": 256, "k": 6, "zipf": 0.0,
         "scales": "f32"},
        # the shared expert alone, dequantised to bf16 by the engine, over a ragged prompt
        {"name": "shared_bf16_500", "kind": "shared", "m": 500, "d": 4096, "i": 2048},
        # the head after plain decode, and after a verify of four drafts
        {"name": "logits_1", "kind": "logits", "t": 1, "d": 4096, "vocab": VOCAB},
        {"name": "logits_5", "kind": "logits", "t": 5, "d": 4096, "vocab": VOCAB},
        # a whole verify: embedding, hash-routed and routed layers with their norms, head, acceptance
        {"name": "verify_2_drafts", "kind": "verify", "layers": 4, "hash": 2, "drafts": 2, "d": 4096, "i": 2048,
         "experts": 256, "k": 6, "vocab": VOCAB},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("layer", "layer", "layer", "routed", "routed", "loader", "shared", "logits", "verify"))
    d = rng.choice((1024, 2048, 4096, 4096))
    i = rng.choice((512, 1024, 1536, 2048, 2048))
    experts = rng.choice((64, 128, 160, 256, 256))
    k = rng.choice((4, 6, 6, 8))
    if kind == "layer":
        t = _log_int(rng, 1, 2700)
        batch = rng.choice((1, 1, t)) if t <= 64 else 1
        return {"kind": kind, "batch": batch, "t": t // batch, "d": d, "i": i, "experts": experts, "k": k,
                "hashed": rng.random() < 0.2}
    if kind == "routed":
        return {"kind": kind, "m": _log_int(rng, 1, 2700), "d": d, "i": i, "experts": experts, "k": k,
                "zipf": round(rng.uniform(0.0, 1.3), 2), "scales": rng.choice(("e8m0", "e8m0", "f32"))}
    if kind == "loader":
        return {"kind": kind, "m": _log_int(rng, 1, 300), "d": d, "i": i, "experts": experts, "k": k,
                "zipf": round(rng.uniform(0.0, 1.3), 2), "scales": rng.choice(("e8m0", "f32"))}
    if kind == "shared":
        return {"kind": kind, "m": _log_int(rng, 1, 4096), "d": d, "i": i}
    if kind == "logits":
        return {"kind": kind, "t": rng.randint(1, 8), "d": rng.choice((2048, 4096, 4096)),
                "vocab": _log_int(rng, 30000, VOCAB)}
    return {"kind": kind, "layers": rng.randint(1, 4), "hash": rng.randint(0, 2), "drafts": rng.randint(1, 4), "d": d,
            "i": i, "experts": rng.choice((64, 128)), "k": k, "vocab": _log_int(rng, 30000, VOCAB)}


# ---------------------------------------------------------------- inputs

def _routing(case, seed):
    """Given ids and weights, the popularity of the experts falling as 1/rank^zipf."""
    idx, w = synthetic.zipf_routing(seed, case["m"], case["experts"], case["k"], case["zipf"], SCALING)
    return torch.from_numpy(idx).to(DEVICE), torch.from_numpy(w).to(DEVICE)


def _store(case, seed, with_shared):
    store = HbmExpertStore(1, case["experts"], case["d"], case["i"], DEVICE, with_shared=with_shared)
    store.fill_synthetic(seed)
    return store


def _f32_entry(views):
    w1, s1, w3, s3, w2, s2 = views
    return w1, s1.to(torch.float32), w3, s3.to(torch.float32), w2, s2.to(torch.float32)


def _normal(seed, sub, shape, std):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed * 64 + sub)
    return (torch.randn(shape, generator=g, device=DEVICE) * std).to(BF16)


def _hash_ids(case, seed, n):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed * 64 + 9)
    return torch.randint(0, VOCAB, (1, n), generator=g, device=DEVICE)


def _prepare_layer(case, seed):
    cfg = MoEConfig(num_hidden_layers=1, hidden_size=case["d"], moe_intermediate_size=case["i"],
                    n_routed_experts=case["experts"], num_experts_per_tok=case["k"],
                    num_hash_layers=1 if case["hashed"] else 0)
    gate, bias = synthetic.router_weights(seed, 0, case["experts"], case["d"], DEVICE)
    lw = {"ffn.gate.weight": gate, "ffn.gate.bias": bias}
    ids = None
    m = case["batch"] * case["t"]
    if case["hashed"]:
        base = torch.empty(VOCAB, dtype=torch.int64, device=DEVICE)
        ops.gen_index(synthetic.key(seed, 3), base, case["experts"])
        step = torch.arange(case["k"], dtype=torch.int64, device=DEVICE) * 7
        lw["ffn.gate.tid2eid"] = (base[:, None] + step[None, :]) % case["experts"]
        ids = _hash_ids(case, seed, m).reshape(case["batch"], case["t"])
    engine = HomeSeekMoEEngine(cfg, _store(case, seed, True), {0: lw})
    engine.store.table(0)
    engine.store.shared_entry(0)
    x = _normal(seed, 1, (case["batch"], case["t"], case["d"]), 1.0)
    return {"kind": "layer", "engine": engine, "lw": lw, "x": x, "ids": ids}


def _prepare_routed(case, seed):
    store = _store(case, seed, False)
    idx, w = _routing(case, seed)
    ffn = FusedMoEFFN(case["experts"], case["i"], case["d"], LIMIT)
    state = {"kind": "routed", "ffn": ffn, "store": store, "idx": idx, "w": w,
             "x": _normal(seed, 1, (case["m"], case["d"]), 1.0),
             "out_f32": torch.empty(case["m"], case["d"], dtype=torch.float32, device=DEVICE)}
    if case["scales"] == "f32":
        state["entries"] = [_f32_entry(store.expert_views(0, e)) for e in range(case["experts"])]
        state["table"] = ops.expert_table(state["entries"], torch.device(DEVICE))
        state["scale_kind"] = ops.SCALE_F32
    else:
        state["table"] = store.table(0)
        state["scale_kind"] = ops.SCALE_E8M0
    return state


def _prepare_loader(case, seed):
    store = _store(case, seed, False)
    idx, w = _routing(case, seed)
    views = [store.expert_views(0, e) for e in range(case["experts"])]
    if case["scales"] == "f32":
        views = [_f32_entry(v) for v in views]
    return {"kind": "loader", "ffn": FusedMoEFFN(case["experts"], case["i"], case["d"], LIMIT), "store": store,
            "load": lambda layer, eid: views[eid], "views": views, "idx": idx, "w": w,
            "x": _normal(seed, 1, (case["m"], case["d"]), 1.0)}


def _prepare_shared(case, seed):
    d, i = case["d"], case["i"]
    return {"kind": "shared", "ffn": SharedExpertFFN(d, i, LIMIT), "x": _normal(seed, 1, (1, case["m"], d), 1.0),
            "w1": _normal(seed, 2, (i, d), 0.02), "w3": _normal(seed, 3, (i, d), 0.02),
            "w2": _normal(seed, 4, (d, i), 0.02)}


def _prepare_logits(case, seed):
    state = {"kind": "logits", "h": _normal(seed, 1, (case["t"], case["d"]), 1.0),
             "head": _normal(seed, 2, (case["vocab"], case["d"]), 0.02), "ids": None}
    if case["t"] > 1:  # the verified row: a token and its drafts
        g = torch.Generator(device=DEVICE)
        g.manual_seed(seed * 64 + 5)
        state["ids"] = torch.randint(0, case["vocab"], (case["t"],), generator=g, device=DEVICE)
    return state


def _prepare_verify(case, seed):
    engine = build_stack(seed, case["layers"], case["experts"], case["d"], case["i"], case["vocab"], case["k"],
                         case["hash"], DEVICE)
    for layer in range(case["layers"]):
        engine.store.table(layer)
        engine.store.shared_entry(layer)
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed * 64 + 6)
    ids = torch.randint(0, case["vocab"], (1, 1 + case["drafts"]), generator=g, device=DEVICE)
    return {"kind": "verify", "engine": engine, "main": ids[:, :1].contiguous(), "drafts": ids[:, 1:].contiguous()}


def prepare(case, seed):
    """What the program holds before the call: experts and their address tables on the GPU, inputs, routing."""
    make = {"layer": _prepare_layer, "routed": _prepare_routed, "loader": _prepare_loader, "shared": _prepare_shared,
            "logits": _prepare_logits, "verify": _prepare_verify}
    return make[case["kind"]](case, seed)


# ---------------------------------------------------------------- the pass

def run(state):
    kind = state["kind"]
    if kind == "layer":
        return state["engine"]._forward_ffn(state["x"], state["lw"], 0, state["ids"])[0]
    if kind == "routed":
        out = state["ffn"].forward_table(state["x"], state["idx"], state["w"], state["table"], state["scale_kind"], None,
                                         out_f32=state["out_f32"])
        return {"out": out, "out_f32": state["out_f32"]}
    if kind == "loader":
        return state["ffn"].forward(state["x"], state["idx"], state["w"], state["load"], 0)
    if kind == "shared":
        return state["ffn"].forward(state["x"], state["w1"], state["w3"], state["w2"])
    if kind == "logits":
        logits, pred, result = ops.lm_head_accept(state["h"], state["head"], state["ids"])
        return {"logits": logits, "pred": pred, "result": result}
    n_accept, bonus = state["engine"]._mtp_verify_batched(state["drafts"], 0.0, state["main"])
    return {"n_accept": n_accept, "bonus_logits": bonus}


# ---------------------------------------------------------------- what a pass cannot do without

def _touched(m, experts, k, zipf=0.0):
    """Experts that m tokens of k distinct ids each select, on average."""
    p = np.arange(1, experts + 1, dtype=np.float64) ** -zipf
    if zipf == 0.0:
        return experts * (1.0 - (1.0 - k / experts) ** m)
    rng = np.random.Generator(np.random.PCG64(1))
    n = min(m, 2048)
    picks = np.argsort(-(np.log(p)[None, :] + rng.gumbel(size=(n, experts))), axis=1)[:, :k]
    share = np.bincount(picks.reshape(-1), minlength=experts) / n
    return float(np.sum(1.0 - (1.0 - np.minimum(share, 1.0)) ** m))


def _expert_bytes(d, i, scale_bytes):
    return 3 * d * i / 2 + 3 * d * i / 32 * scale_bytes


def _layer_work(m, d, i, experts, k, hashed):
    nbytes = (_touched(m, experts, k) * _expert_bytes(d, i, 1) + 3 * d * i + 4 * 3 * d * i / 128 ** 2 + m * 2 * d * 2)
    flops = m * (k + 1) * 6 * d * i
    if not hashed:
        nbytes += experts * (2 * d + 4)
        flops += 2 * m * experts * d
    return nbytes, flops


def work(case):
    kind, d = case["kind"], case["d"]
    if kind == "layer":
        nbytes, flops = _layer_work(case["batch"] * case["t"], d, case["i"], case["experts"], case["k"],
                                    case["hashed"])
    elif kind in ("routed", "loader"):
        m, i, k = case["m"], case["i"], case["k"]
        nbytes = (_touched(m, case["experts"], k, case["zipf"]) * _expert_bytes(d, i, 4 if case["scales"] == "f32" else 1)
                  + m * k * 12 + m * d * (8 if kind == "routed" else 4))
        flops = m * k * 6 * d * i
    elif kind == "shared":
        nbytes = 3 * d * case["i"] * 2 + case["m"] * d * 4
        flops = case["m"] * 6 * d * case["i"]
    elif kind == "logits":
        nbytes = 2 * d * case["vocab"] + case["t"] * 2 * (d + case["vocab"])
        flops = 2 * case["t"] * d * case["vocab"]
    else:
        t = 1 + case["drafts"]
        nbytes, flops = 2 * d * case["vocab"] + 2 * case["vocab"], 2 * t * d * case["vocab"]
        for layer in range(case["layers"]):
            b, f = _layer_work(t, d, case["i"], case["experts"], case["k"], layer < case["hash"])
            nbytes, flops = nbytes + b, flops + f
    return {"bytes": float(nbytes), "flops": float(flops)}


def tolerance(case):
    kind = case["kind"]
    if kind == "verify":
        # bf16 residual adds and norms between the layers carry one rounding of a layer on through the rest
        return {"rel": 0.02, "max": 0.1, "differ": 0.0}
    if kind == "logits":
        # each logit is the correctly rounded bf16 of the exact sum: only a near-tie of the rounding can differ
        return {"rel": 1e-4, "max": 0.008, "differ": 0.0}
    # results rounded to bf16 from fp32 sums
    return {"rel": 0.007, "max": 0.016}


# ---------------------------------------------------------------- 64 bits

_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _fp4(data, scale):
    """The bf16 weights that FP4 codes and their scales stand for, in 64 bits."""
    b = data.view(torch.uint8).to(torch.int64)
    lut = torch.tensor(_E2M1, dtype=torch.float64, device=b.device)
    v = torch.stack((lut[b & 15], lut[b >> 4]), dim=-1).reshape(b.shape[0], -1, 32)
    s = scale.to(torch.float32).to(torch.float64)
    return (v * s[:, :, None]).reshape(b.shape[0], -1).to(BF16).double()


def _fp8(data, scale):
    v = data.to(torch.float32)
    s = scale.repeat_interleave(128, 0)[: v.shape[0]].repeat_interleave(128, 1)[:, : v.shape[1]]
    return (v * s).to(BF16).double()


def _swiglu(x, w1, w3, w2):
    g, u = (x @ w1.T).clamp(max=LIMIT), (x @ w3.T).clamp(-LIMIT, LIMIT)
    return (g * torch.sigmoid(g) * u) @ w2.T


def _experts(x, idx, w, views):
    """sum_j w[t, j] FFN_{idx[t, j]}(x[t]); views(e): the 6 FP4 tensors of expert e."""
    out = torch.zeros_like(x)
    for e in torch.unique(idx).tolist():
        t, j = torch.nonzero(idx == e, as_tuple=True)
        w1, s1, w3, s3, w2, s2 = views(e)
        y = _swiglu(x[t], _fp4(w1, s1), _fp4(w3, s3), _fp4(w2, s2))
        out.index_add_(0, t, y * w[t, j].double()[:, None])
    return out


def _route(x, lw, k):
    """The router's definition: bf16 logits (rounded before and after the bias), sqrt(softplus), stable top k."""
    logits = (x @ lw["ffn.gate.weight"].double().T).to(BF16) + lw["ffn.gate.bias"].to(BF16)
    scores = torch.nn.functional.softplus(logits.double()).sqrt()
    idx = torch.sort(scores, dim=1, descending=True, stable=True).indices[:, :k]
    w = torch.gather(scores, 1, idx)
    return idx, w / w.sum(dim=1, keepdim=True) * SCALING


def _exact_layer(engine, lw, layer, x, ids, hashed, k):
    """[M, D] in 64 bits of the layer's FFN on hidden rows x [M, D]."""
    x = x.double()
    if hashed:
        idx = lw["ffn.gate.tid2eid"][ids.reshape(-1)]
        w = torch.full(idx.shape, 1.0 / k, dtype=torch.float64, device=x.device)
    else:
        idx, w = _route(x, lw, k)
    w1, s1, w3, s3, w2, s2 = engine.store.shared_views(layer)
    out = _experts(x, idx, w, lambda e: engine.store.expert_views(layer, e))
    return out + _swiglu(x, _fp8(w1, s1), _fp8(w3, s3), _fp8(w2, s2))


def _norm(h, weight):
    h = h.double()
    return (h * torch.rsqrt(h.square().mean(dim=-1, keepdim=True) + 1e-6) * weight.double()).to(BF16)


def exact(case, seed):
    state = prepare(case, seed)
    kind = case["kind"]
    if kind == "layer":
        x = state["x"]
        out = _exact_layer(state["engine"], state["lw"], 0, x.reshape(-1, case["d"]), state["ids"], case["hashed"],
                           case["k"])
        return out.reshape(x.shape)
    if kind in ("routed", "loader"):
        views = state.get("entries") or state.get("views")
        out = _experts(state["x"].double(), state["idx"], state["w"],
                       lambda e: views[e] if views else state["store"].expert_views(0, e))
        return {"out": out, "out_f32": out} if kind == "routed" else out
    if kind == "shared":
        return _swiglu(state["x"].double(), state["w1"].double(), state["w3"].double(), state["w2"].double())
    if kind == "logits":
        return {"logits": _head(state["h"], state["head"]), "pred": None, "result": None}
    engine, ids = state["engine"], torch.cat((state["main"], state["drafts"]), dim=1).reshape(-1)
    h = engine.embed[ids]
    for layer in range(case["layers"]):  # the residual stream is bf16 between the layers
        lw = engine._layer_weights[layer]
        h = h + lw["attn.residual"]
        f = _exact_layer(engine, lw, layer, _norm(h, lw["ffn_norm.weight"]), ids, layer < case["hash"], case["k"])
        h = h + f.to(BF16)
    logits = _head(_norm(h, engine.norm_weight), engine.lm_head)
    pred = logits.to(BF16).argmax(dim=1)
    n = 0
    while n < case["drafts"] and int(pred[n]) == int(ids[n + 1]):
        n += 1
    return {"n_accept": None, "bonus_logits": logits[n:n + 1]}


def _head(h, head):
    h = h.double()
    return torch.cat([h @ part.double().T for part in head.split(16384)], dim=1)
