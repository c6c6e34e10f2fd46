"""Performance cases of the fused-MoE operator: what a serving or prefill program runs.

A case is one pass over `layers` MoE layers of an expert-parallel rank (32 of 256
experts), each with its own weights, routing and tokens, through the package's public
entry points: `kernel.kernel` on FP8 activations, with `quantize_fp8_blockwise` before it
where the program holds bf16 hidden states (`bf16`), or the quantizer alone (`cols`).
Decode cases walk several layers, as a decode step does, so that the weights of a call are
not still in the last-level cache from the pass before.

  listed()            the cases
  draw(rng)           one more case of the same ranges
  prepare(case, seed) inputs, weights and output buffers on the GPU, from the seed alone
  run(state)          one pass, returning the outputs
  work(case)          bytes and operations a pass cannot do without
  tolerance(case)     how far two correct implementations may differ
  exact(case, seed)   the outputs in 64 bits, by plain torch
"""
import importlib
import math

import torch

_PKG = "flash-infer-bench-starter-kit_amd"
kernel = importlib.import_module(_PKG + ".kernel")
workloads = importlib.import_module(_PKG + ".workloads")

H, I, BLK, N_GLOBAL, N_LOCAL, TOP_K = 7168, 2048, 128, 256, 32, 8
FACTOR = 2.5


def _moe(T, offset=0, layers=1, hot=False, bf16=False):
    """tokens, first expert of the rank, layers of the pass, four hot local experts,
    activations given in bf16 (the pass quantises them)."""
    return {"T": T, "offset": offset, "layers": layers, "hot": hot, "bf16": bf16}


def _quant(rows, cols, fp32):
    return {"rows": rows, "cols": cols, "fp32": fp32}


def listed():
    cases = {
        # one interactive sequence: the smallest call, two launches, latency counts
        "decode_t1": _moe(1, 0, layers=8),
        # a small decode batch (the smallest benchmark configuration's size)
        "decode_t8": _moe(8, 32, layers=4),
        # a ragged decode batch between the powers of two, on the last rank
        "decode_t27": _moe(27, 224, layers=2),
        # a full decode batch (the headline benchmark configuration's size)
        "decode_t64": _moe(64, 0, layers=1),
        # a large decode batch, or decode with draft tokens, odd count
        "decode_t157": _moe(157, 128),
        # a prefill chunk from bf16 hidden states: the quantizer, then the operator
        "chunk_t509_bf16": _moe(509, 96, bf16=True),
        # a prefill chunk on another rank (benchmark configuration)
        "prefill_t1024_off64": _moe(1024, 64),
        # a prefill of an odd length
        "prefill_t2731": _moe(2731, 160),
        # skewed routing: four hot experts on this rank (benchmark configuration)
        "skew_t4096": _moe(4096, 0, hot=True),
        # a long prefill (benchmark configuration)
        "prefill_t8192": _moe(8192, 0),
        # the longest prefill: a sequence length of the operator's data set
        "prefill_t14107": _moe(14107, 32),
        # the activation quantizer alone, as the layer before the operator calls it
        "quantize_bf16_4093": _quant(4093, H, False),
    }
    return [dict(c, name=n) for n, c in cases.items()]


def draw(rng):
    """Sizes spread over their logarithm; a skewed case stays at or below 4096 tokens."""
    def size(lo, hi):
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    if rng.random() < 0.2:
        return _quant(size(1, 14107), rng.choice((1536, 2048, 4096, 5120, H, H)), rng.random() < 0.4)
    hot = rng.random() < 0.15
    T = size(256, 4096) if hot else size(1, 14107)
    layers = 8 if T <= 2 else 4 if T <= 12 else 2 if T <= 40 else 1
    return _moe(T, 32 * rng.randrange(8), layers, hot, rng.random() < 0.3)


def _config(case, seed, layer):
    hot = (3, 11, 19, 27) if case["hot"] else ()
    return workloads.Config("case", case["T"], case["offset"], hot, FACTOR, seed=1000 * seed + 16 + layer)


def _hidden(shape, seed, dtype):
    """Hidden states after a normalisation: N(0, 1)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(7919 * seed + 5)
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def prepare(case, seed):
    if "cols" in case:
        return {"x": _hidden((case["rows"], case["cols"]), seed, torch.float32 if case["fp32"] else torch.bfloat16)}
    layers = []
    for i in range(case["layers"]):
        d = workloads.make_inputs(_config(case, seed, i), device="cuda")
        x = _hidden((case["T"], H), 64 * seed + i, torch.bfloat16) if case["bf16"] else None
        layers.append((x, workloads.as_args(d)))
    return {"layers": layers}


def run(state):
    if "x" in state:
        return kernel.quantize_fp8_blockwise(state["x"])
    for x, args in state["layers"]:
        if x is not None:
            args[2], args[3] = kernel.quantize_fp8_blockwise(x)
        kernel.kernel(*args)
    return [args[10] for _, args in state["layers"]]


def _topk8(logits, bias):
    """The routing rule (DeepSeek no-aux, 8 groups, best 4): ids [T, 8] and the sigmoids.
    The selection is made on fp32 values, as the rule has it, ties to the lower index."""
    s = torch.sigmoid(logits.double()).float()
    sb = s + bias.float()
    T = s.shape[0]
    g = sb.view(T, 8, 32)
    top2 = torch.sort(g, dim=2, descending=True, stable=True).values[:, :, :2]
    gscore = top2[:, :, 0] + top2[:, :, 1]
    gid = torch.sort(gscore, dim=1, descending=True, stable=True).indices[:, :4]
    keep = torch.zeros(T, 8, dtype=torch.bool, device=s.device)
    keep.scatter_(1, gid, True)
    masked = torch.where(keep[:, :, None], g, torch.full_like(g, float("-inf"))).view(T, N_GLOBAL)
    return torch.sort(masked, dim=1, descending=True, stable=True).indices[:, :TOP_K], s


def work(case):
    if "cols" in case:
        n = case["rows"] * case["cols"]
        return {"bytes": n * ((4 if case["fp32"] else 2) + 1) + n // BLK * 4, "flops": 2 * n}
    # the routed rows and active experts of a typical routing of these sizes
    total = {"bytes": 0, "flops": 0}
    for i in range(case["layers"]):
        cfg = _config(case, 0, i)
        ids, _ = _topk8(*workloads.make_routing_inputs(cfg))
        w = workloads.algorithmic_work(ids, case["offset"], case["T"])
        total["bytes"] += w["bytes"] + (case["T"] * (2 * H + H + H // BLK * 4) if case["bf16"] else 0)
        total["flops"] += w["flops"]
    return total


def tolerance(case):
    if "cols" in case:
        return "exact"      # codes and scales are defined bit for bit
    # against exact() the bf16 rounding of the output alone shows as 1.7e-3, with the
    # intermediate in 8 bits more as 1.8e-3
    return {"rel": 7e-3, "max": 0.05}


def _quantized(x):
    """Codes and scales by the quantizer's rule, in torch's own fp32."""
    T, C = x.shape
    xf = x.float().view(T, C // BLK, BLK)
    amax = xf.abs().amax(dim=2)
    # a tensor divisor: torch divides by a number as a product with its reciprocal
    scale = torch.where(amax > 0, amax / torch.full_like(amax, 448.0), torch.ones_like(amax))
    q = (xf * (1.0 / scale)[:, :, None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return q.view(T, C), scale.t().contiguous()


def _dequant_weight(q, s):
    return (q.double().view(q.shape[0] // BLK, BLK, q.shape[1] // BLK, BLK) * s.double()[:, None, :, None]).view(q.shape)


def exact(case, seed):
    state = prepare(case, seed)
    if "cols" in case:
        x = state["x"].double().view(case["rows"], case["cols"] // BLK, BLK)
        scale = x.abs().amax(dim=2) / 448.0
        return (x / scale[:, :, None]).view(case["rows"], case["cols"]), scale.t().contiguous()
    outs = []
    for x, args in state["layers"]:
        logits, bias, hs, hs_scale, w1, s1, w2, s2, offset, factor, _ = args
        if x is not None:
            hs, hs_scale = _quantized(x)
        ids, s = _topk8(logits, bias)
        w = torch.gather(s, 1, ids).double()
        w = w / (w.sum(dim=1, keepdim=True) + 1e-20) * factor
        T = case["T"]
        a = (hs.double().view(T, H // BLK, BLK) * hs_scale.double().t()[:, :, None]).view(T, H)
        out = torch.zeros(T, H, dtype=torch.float64, device="cuda")
        for e in range(N_LOCAL):
            tok, slot = (ids == offset + e).nonzero(as_tuple=True)
            if tok.numel() == 0:
                continue
            h = a[tok] @ _dequant_weight(w1[e], s1[e]).t()
            c = torch.nn.functional.silu(h[:, I:]) * h[:, :I]
            o = c @ _dequant_weight(w2[e], s2[e]).t()
            out.index_add_(0, tok, o * w[tok, slot][:, None])
        outs.append(out)
    return outs
