"""The work this package is timed on: quantised linear layers, MoE blocks and weight dequantisation,
called the way a serving engine calls them (layer methods with loaded weights, one call per layer
and step, eager on the current stream).

A case is one of
  op = "linears": the AWQ linear layers of one decoder layer, each through AWQLinearMethod.apply on
       its own activations ("layers" = "KxN,KxN,...", a "+b" behind a layer gives it a bias);
  op = "moe": one fused MoE block through AWQMoEMethod.apply;
  op = "dequantize": the weight matrices of "layers" through awq_dequantize.

Weights and zero points are uniform int4, scales uniform in [0.001, 0.02], activations and router
logits N(0, 1): the distributions of workloads.py.
"""
import torch

import server_benchmark_amd as sba

# Layers of one decoder layer: qkv, o, gate_up, down.
DENSE_72B = "8192x10240+b,8192x8192,8192x59136,29568x8192"      # Qwen2.5-72B (workloads.QWEN25_72B_LAYERS)
DENSE_7B = "3584x4608+b,3584x3584,3584x37888,18944x3584"        # a 7B-class model
DENSE_5K = "5120x7168,5120x5120,5120x27648,13824x5120"          # 5120-wide models
MOE_ATTENTION = "2048x5120,4096x2048"                           # qkv and o of Qwen3-30B-A3B

# hidden, inter, experts, top-k
QWEN3_MOE = (2048, 768, 128, 8)
MOE_SHAPES = (QWEN3_MOE, QWEN3_MOE, QWEN3_MOE, (2048, 1408, 64, 6), (5120, 1024, 64, 4), (4096, 14336, 8, 2))


def _linears(name, layers, rows, group=128):
    return {"name": name, "op": "linears", "layers": layers, "rows": rows, "group": group}


def _moe(name, shape, rows, group=128, scoring="softmax"):
    return {"name": name, "op": "moe", "hidden": shape[0], "inter": shape[1], "experts": shape[2], "topk": shape[3],
            "rows": rows, "group": group, "scoring": scoring}


def listed():
    return [
        # attention projections of the MoE model for a single user's next token: the smallest calls
        _linears("moe_attention_m1", MOE_ATTENTION, 1),
        # one decoder layer, single user (the serving load at concurrency 1)
        _linears("dense72b_m1", DENSE_72B, 1),
        # ... a small batch of users
        _linears("dense72b_m16", DENSE_72B, 16),
        # ... the decode batch of the serving driver (decoder.run_serving_load)
        _linears("dense72b_m64", DENSE_72B, 64),
        # ... the load generator's concurrency on one GPU (400 requests decoding together)
        _linears("dense72b_m400", DENSE_72B, 400),
        # one request's 1000-token prompt on a small model quantised with 64-row groups
        _linears("dense7b_m1000_g64", DENSE_7B, 1000, group=64),
        # prefill with the token budget full (8192 tokens per step)
        _linears("dense72b_m8192", DENSE_72B, 8192),
        # the MoE block: single user, decode batch of the serving driver, the load generator's
        # concurrency, prefill with the token budget full
        _moe("moe_t1", QWEN3_MOE, 1),
        _moe("moe_t64", QWEN3_MOE, 64),
        _moe("moe_t400", QWEN3_MOE, 400),
        _moe("moe_t8192", QWEN3_MOE, 8192),
        # weights handed to a library GEMM (an engine that only rebinds awq_dequantize)
        {"name": "dequantize_72b", "op": "dequantize", "layers": DENSE_72B, "group": 128},
    ]


def draw(rng):
    """One more case: rows over 1 .. 8192 (log-uniform, any integer), layers of the models above or a
    single layer of any size, group sizes 128, 64 and 32."""
    rows = min(8192, max(1, round(2.0 ** rng.uniform(0.0, 13.0))))
    kind = rng.random()
    if kind < 0.45:
        layers = rng.choice((DENSE_72B, DENSE_7B, DENSE_5K, MOE_ATTENTION))
        c = _linears("", layers, rows, group=rng.choice((128, 128, 128, 64, 32)))
    elif kind < 0.6:
        # one layer, sizes of tensor-parallel shards and smaller models among them
        k = 128 * max(4, round(2.0 ** rng.uniform(2.0, 7.85)))
        n = 32 * max(16, round(2.0 ** rng.uniform(4.0, 10.85)))
        c = _linears("", "%dx%d%s" % (k, n, rng.choice(("", "+b"))), rows, group=rng.choice((128, 128, 64, 32)))
    elif kind < 0.92:
        shape = rng.choice(MOE_SHAPES)
        c = _moe("", shape, rows, group=rng.choice((128, 128, 64)), scoring=rng.choice(("softmax", "softmax", "sigmoid")))
    else:
        k = 128 * round(2.0 ** rng.uniform(3.0, 7.85))
        n = 32 * round(2.0 ** rng.uniform(5.0, 10.85))
        c = {"op": "dequantize", "layers": "%dx%d" % (k, n), "group": rng.choice((128, 64, 32))}
    c.pop("name", None)
    return c


def _shapes(case):
    out = []
    for item in case["layers"].split(","):
        dims, _, bias = item.partition("+")
        k, n = dims.split("x")
        out.append((int(k), int(n), bool(bias)))
    return out


def _rand_awq(k, n, group, gen, lead=()):
    dev = gen.device
    qw = torch.randint(-2 ** 31, 2 ** 31, (*lead, k, n // 8), dtype=torch.int32, device=dev, generator=gen)
    qz = torch.randint(-2 ** 31, 2 ** 31, (*lead, k // group, n // 8), dtype=torch.int32, device=dev, generator=gen)
    sc = (torch.rand((*lead, k // group, n), device=dev, generator=gen) * 0.019 + 0.001).half()
    return qw, sc, qz


def prepare(case, seed):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(seed)
    group = case["group"]
    config = sba.AWQConfig(weight_bits=4, group_size=group, zero_point=True)
    if case["op"] == "dequantize":
        return {"op": "dequantize", "weights": [_rand_awq(k, n, group, gen) for k, n, _ in _shapes(case)]}
    if case["op"] == "linears":
        method, calls = sba.AWQLinearMethod(config), []
        for k, n, has_bias in _shapes(case):
            layer = torch.nn.Module()
            method.create_weights(layer, k, [n], k, n, torch.float16, device=dev)
            layer.qweight.data, layer.scales.data, layer.qzeros.data = _rand_awq(k, n, group, gen)
            method.process_weights_after_loading(layer)
            bias = torch.randn(n, device=dev, generator=gen).half() if has_bias else None
            calls.append((layer, torch.randn((case["rows"], k), device=dev, generator=gen).half(), bias))
        return {"op": "linears", "method": method, "calls": calls}
    method, layer = sba.AWQMoEMethod(config), torch.nn.Module()
    hidden, inter, experts, rows = case["hidden"], case["inter"], case["experts"], case["rows"]
    method.create_weights(layer, experts, hidden, inter, torch.float16, device=dev)
    layer.w13_qweight.data, layer.w13_scales.data, layer.w13_qzeros.data = _rand_awq(hidden, 2 * inter, group, gen, (experts,))
    layer.w2_qweight.data, layer.w2_scales.data, layer.w2_qzeros.data = _rand_awq(inter, hidden, group, gen, (experts,))
    method.process_weights_after_loading(layer)
    sigmoid = case["scoring"] == "sigmoid"
    return {"op": "moe", "method": method, "layer": layer, "topk": case["topk"], "scoring": case["scoring"],
            "x": torch.randn((rows, hidden), device=dev, generator=gen).half(),
            "logits": torch.randn((rows, experts), device=dev, generator=gen),
            "bias": torch.randn(experts, device=dev, generator=gen) * 0.1 if sigmoid else None}


def run(state):
    if state["op"] == "linears":
        return [state["method"].apply(layer, x, bias) for layer, x, bias in state["calls"]]
    if state["op"] == "moe":
        return state["method"].apply(state["layer"], state["x"], state["logits"], state["topk"], True,
                                     scoring_func=state["scoring"], e_score_correction_bias=state["bias"])
    return [sba.awq_dequantize(*w) for w in state["weights"]]


def _weight_bytes(k, n, group):
    return k * n // 2 + (k // group) * (2 * n + n // 2)


def work(case):
    if case["op"] == "linears":
        m = case["rows"]
        return {"bytes": sum(_weight_bytes(k, n, case["group"]) + 2 * m * (k + n) + 2 * n * b for k, n, b in _shapes(case)),
                "flops": sum(2 * m * k * n for k, n, _ in _shapes(case))}
    if case["op"] == "dequantize":
        return {"bytes": sum(_weight_bytes(k, n, case["group"]) + 2 * k * n for k, n, _ in _shapes(case)), "flops": 0}
    hidden, inter, experts, m = case["hidden"], case["inter"], case["experts"], case["rows"]
    # experts that at least one of the tokens picks, on average
    touched = experts * (1.0 - (1.0 - case["topk"] / experts) ** m)
    per_expert = _weight_bytes(hidden, 2 * inter, case["group"]) + _weight_bytes(inter, hidden, case["group"])
    return {"bytes": int(touched * per_expert) + 4 * m * hidden + 4 * m * experts,
            "flops": 2 * m * case["topk"] * 3 * hidden * inter}


def tolerance(case):
    """Largest differences seen against the same pass on exact weights with float64 sums (relative
    2-norm / single value over the result's rms): linears 3.5e-4 / 1.25e-3 (2.1e-4 of it the fp16
    rounding of the result), MoE block 6.6e-4 / 3.1e-3 (activations and slot results are rounded to
    fp16 on the way).  About four times that.  Dequantised weights are exact by definition."""
    if case["op"] == "dequantize":
        return "exact"
    return {"rel": 1.2e-3, "max": 5e-3} if case["op"] == "linears" else {"rel": 2.6e-3, "max": 1.2e-2}


def _unpack(words):
    shifts = torch.tensor([0, 16, 4, 20, 8, 24, 12, 28], dtype=torch.int32, device=words.device)   # AWQ nibble order
    return ((words[..., None] >> shifts) & 15).flatten(-2)


def _weights(qw, sc, qz, k0=0, k1=None):
    """Rows k0 .. k1 of (w - z) * s in float64 (qw [K, N / 8], sc [K / G, N], qz [K / G, N / 8])."""
    k1 = qw.shape[0] if k1 is None else k1
    g = torch.arange(k0, k1, device=qw.device) // (qw.shape[0] // sc.shape[0])
    return (_unpack(qw[k0:k1]) - _unpack(qz)[g]).double() * sc.double()[g]


def _matmul64(x, qw, sc, qz):
    """x (float64) times the exact weights, a few thousand weight rows at a time."""
    step = max(128, 2 ** 27 // sc.shape[1])
    out = torch.zeros((x.shape[0], sc.shape[1]), dtype=torch.float64, device=x.device)
    for k0 in range(0, qw.shape[0], step):
        k1 = min(k0 + step, qw.shape[0])
        out += x[:, k0:k1] @ _weights(qw, sc, qz, k0, k1)
    return out


def exact(case, seed):
    """The pass on exact weights with float64 sums and no rounding on the way."""
    state = prepare(case, seed)
    if state["op"] == "dequantize":
        return [torch.cat([_weights(*w, k0, min(k0 + 4096, w[0].shape[0])).half() for k0 in range(0, w[0].shape[0], 4096)])
                for w in state["weights"]]
    if state["op"] == "linears":
        return [_matmul64(x.double(), layer.qweight, layer.scales, layer.qzeros) + (0.0 if bias is None else bias.double())
                for layer, x, bias in state["calls"]]
    layer, x, logits, topk = state["layer"], state["x"].double(), state["logits"].double(), state["topk"]
    if state["scoring"] == "sigmoid":
        score = torch.sigmoid(logits)
        chosen = torch.topk(score + state["bias"].double(), topk, dim=-1).indices
    else:
        score = torch.softmax(logits, dim=-1)
        chosen = torch.topk(score, topk, dim=-1).indices
    weight = score.gather(1, chosen)
    weight = weight / weight.sum(dim=-1, keepdim=True)
    out = torch.zeros_like(x)
    for e in range(logits.shape[1]):
        token, slot = torch.nonzero(chosen == e, as_tuple=True)
        if token.numel() == 0:
            continue
        h = _matmul64(x[token], layer.w13_qweight[e], layer.w13_scales[e], layer.w13_qzeros[e])
        gate, up = h.chunk(2, dim=-1)
        o = _matmul64(torch.nn.functional.silu(gate) * up, layer.w2_qweight[e], layer.w2_scales[e], layer.w2_qzeros[e])
        out.index_add_(0, token, o * weight[token, slot, None])
    return out
