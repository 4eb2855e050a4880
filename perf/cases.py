"""Performance cases of the FP8 block-scale MoE layer and of the activation
quantiser in front of it, through the package's public entry points.

A case's kind is
  * "layer": one call of `run` (or `run_noalloc`) for T tokens on one
    expert-parallel rank (32 of 256 experts), as a serving engine makes it once
    per MoE layer and step.  `offset` is the rank's first expert, `hot` the
    number of this rank's experts whose routing bias is raised by 2.0 (every
    token then selects them, as in the skewed benchmark configuration), `rsf`
    the routed scaling factor;
  * "quantize": one call of `quantize_hidden`, which makes the layer's e4m3
    rows and block scales out of bf16 hidden rows.

Inputs come from the package's seeded GPU generator (the benchmark's
distributions); weights and buffers are what a serving program keeps.
"""
import importlib
import math

import torch

pkg = importlib.import_module("mlsys-contest-syfi-fully-agent_amd")

H, I, E_LOCAL, E_GLOBAL, TOP_K, BLOCK = 7168, 2048, 32, 256, 8, 128
MAX_T = 14107  # the largest token count of the contest's dataset
MAX_T_HOT = 8192  # the largest with hot experts (the benchmark's skewed configuration)
HOT_LOCAL = (0, 8, 16, 24)  # rank-local ids of the hot experts


def _layer(name, T, offset=0, hot=0, rsf=2.5, noalloc=False):
    return {"name": name, "kind": "layer", "T": T, "offset": offset, "hot": hot, "rsf": rsf, "noalloc": noalloc}


def listed():
    return [
        # one token being decoded, its rank holding two experts that the router favours
        _layer("decode_t1", 1, hot=2),
        # a small decode batch through the call that needs no workspace (graph capture, tight loops)
        _layer("decode_t7_noalloc", 7, offset=96, noalloc=True),
        # a decode batch, or the last chunk of a short prompt
        _layer("small_t64", 64, offset=32),
        # a decode batch over hot experts, with a ragged count
        _layer("hot_t51", 51, hot=4),
        # a mid-size batch with a ragged count, scaling factor of another model configuration
        _layer("mid_t333", 333, offset=224, rsf=1.0),
        # one prefill chunk
        _layer("prefill_t1024", 1024),
        # a prefill chunk with hot experts, ragged
        _layer("hot_t1451", 1451, offset=64, hot=4),
        # several prompts in one batch
        _layer("prefill_t4096", 4096, offset=128),
        # the skewed benchmark configuration: the most work of all
        _layer("skewed_t8192", 8192, hot=4),
        # the longest batch of the dataset, uniform routing
        _layer("prefill_t14107", MAX_T, offset=32),
        # the quantiser of a prefill chunk and of the longest batches
        {"name": "quantize_t1023", "kind": "quantize", "T": 1023},
        {"name": "quantize_t8192", "kind": "quantize", "T": 8192},
    ]


def draw(rng):
    if rng.random() < 0.15:
        return {"kind": "quantize", "T": int(round(math.exp(rng.uniform(math.log(64), math.log(MAX_T)))))}
    hot = rng.choice([0, 0, 0, 2, 3, 4])
    T = max(1, int(round(math.exp(rng.uniform(0.0, math.log(MAX_T_HOT if hot else MAX_T))))))
    if T < 16 and not hot:
        hot = 2  # a single token of uniform routing often selects no expert of the rank
    offset = 32 * rng.randrange(8) if rng.random() < 0.8 else rng.randrange(225)
    noalloc = T <= 64 and rng.random() < 0.3
    c = _layer("", T, offset, hot, rng.choice([2.5, 2.5, 1.0]), noalloc)
    del c["name"]
    return c


def prepare(case, seed):
    dev = torch.device("cuda")
    T = case["T"]
    if case["kind"] == "quantize":
        g = torch.Generator(device=dev).manual_seed(int(seed))
        x = torch.randn((T, H), generator=g, device=dev, dtype=torch.float32).to(torch.bfloat16)
        return {"case": case, "x": x, "q": torch.empty((T, H), dtype=torch.float8_e4m3fn, device=dev),
                "scale": torch.empty((H // BLOCK, T), dtype=torch.float32, device=dev)}
    hot = tuple(case["offset"] + h for h in HOT_LOCAL[: case["hot"]])
    cfg = pkg.synth.Config("case", T, case["offset"], int(seed), hot, 2.0 if hot else 0.0, case["rsf"])
    return {"case": case, "args": pkg.synth.inputs(cfg, dev),
            "out": torch.empty((T, H), dtype=torch.bfloat16, device=dev)}


def run(state):
    case = state["case"]
    if case["kind"] == "quantize":
        return pkg.quantize_hidden(state["x"], state["q"], state["scale"])
    call = pkg.run_noalloc if case["noalloc"] else pkg.run
    return call(*state["args"], case["offset"], case["rsf"], state["out"])


def _select(score, bias):
    """The definition's selection: top 2 sums of 8 groups, 4 groups, 8 experts."""
    T = score.shape[0]
    groups = (score + bias).view(T, 8, 32)
    best = groups.topk(2, dim=2).values.sum(2).topk(4, dim=1).indices
    keep = torch.zeros((T, 8), dtype=torch.bool, device=score.device).scatter_(1, best, True)
    masked = groups.masked_fill(~keep[:, :, None], float("-inf")).view(T, E_GLOBAL)
    return masked.topk(TOP_K, dim=1).indices


def work(case):
    """Pairs and active experts of the case's routing, averaged over draws of
    logits and bias from the generator's distributions."""
    T = case["T"]
    if case["kind"] == "quantize":
        return {"bytes": T * (3 * H + 4 * (H // BLOCK)), "flops": 0}
    pairs = experts = 0.0
    draws = max(2, min(64, 4096 // T))
    for seed in range(draws):
        g = torch.Generator().manual_seed(seed)
        logits = torch.randn((T, E_GLOBAL), generator=g)
        bias = 0.1 * torch.randn((E_GLOBAL,), generator=g)
        for h in HOT_LOCAL[: case["hot"]]:
            bias[case["offset"] + h] += 2.0
        local = _select(torch.sigmoid(logits), bias) - case["offset"]
        local = local[(local >= 0) & (local < E_LOCAL)]
        pairs += local.numel() / draws
        experts += local.unique().numel() / draws
    per_expert = 3 * I * H + 4 * 3 * (I // BLOCK) * (H // BLOCK)
    per_token = H + 4 * (H // BLOCK) + 4 * E_GLOBAL + 2 * H
    return {"bytes": experts * per_expert + T * per_token + 2 * E_GLOBAL, "flops": pairs * 3 * 2 * I * H}


def tolerance(case):
    if case["kind"] == "quantize":
        return "exact"
    # bf16 outputs: against 64 bits the layer is 1.7e-3 off in the 2-norm and
    # at most one half unit in the last place (2^-8 of the value) in any element
    return {"rel": 7e-3, "max": 1.6e-2}


def exact(case, seed):
    state = prepare(case, seed)
    if case["kind"] == "quantize":
        x = state["x"].double().view(-1, H // BLOCK, BLOCK)
        amax = x.abs().amax(2)
        s = torch.where(amax > 0, amax / 448.0, torch.ones_like(amax))
        # a code is the rounding of the 32-bit quotient by the stored 32-bit
        # scale (its ties are frequent and would all be broken in 64 bits)
        y = (x / s.float().double()[:, :, None]).float().double().clamp(-448.0, 448.0)
        step = torch.exp2(torch.floor(torch.log2(y.abs().clamp_min(2.0 ** -6))) - 3)
        return torch.round(y / step).mul(step).view(-1, H), s.t().contiguous()
    logits, bias, hs, hs_scale, w13, w13s, w2, w2s = state["args"]
    T = case["T"]
    # selection in 32 bits, as the definition states it; the weights in 64
    score = torch.sigmoid(logits.double())
    ids = _select(score.float(), bias.float())
    w = score.gather(1, ids)
    w = w / (w.sum(1, keepdim=True) + 1e-20) * case["rsf"]
    a_all = (hs.float().view(T, H // BLOCK, BLOCK).double() * hs_scale.t().double()[:, :, None]).view(T, H)
    out = torch.zeros((T, H), dtype=torch.float64, device=logits.device)

    def wide(q, s):
        q = q.float().double().view(s.shape[0], BLOCK, s.shape[1], BLOCK)
        return (q * s.double()[:, None, :, None]).view(s.shape[0] * BLOCK, s.shape[1] * BLOCK)

    for e in range(E_LOCAL):
        tok, pick = torch.where(ids == case["offset"] + e)
        if tok.numel():
            g = a_all[tok] @ wide(w13[e], w13s[e]).t()
            up = g[:, I:]
            c = up * torch.sigmoid(up) * g[:, :I]
            out.index_add_(0, tok, (c @ wide(w2[e], w2s[e]).t()) * w[tok, pick][:, None])
    return out
