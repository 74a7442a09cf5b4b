"""Cases that stand for what this library is used for: decoding with INT4 AWQ weights on one GPU.

  gemv      one projection called on its own, launch by launch (the layer API, tests, a model under development)
  layers    the seven projections of several decoder layers, replayed from a HIP graph (what bench.py measures)
  dense     one BF16 GEMV (lm_head), launch by launch
  step      a whole decode step of one sequence, from a HIP graph or launch by launch
  batch     a whole decode step of several sequences together, from a HIP graph

Sizes are those of mykuiperllama_amd.synth and mykuiperllama_amd.decode, or generic.
"""
import math

import torch

from mykuiperllama_amd import capi, decode, synth

_PROJECTIONS = ("q", "k", "v", "o", "gate", "up", "down")


def listed():
    small = {"hidden": 1024, "inter": 3072, "n_q": 16, "n_kv": 8}
    eight = {"hidden": 4096, "inter": 12288, "n_q": 32, "n_kv": 8}
    thirty = {"hidden": 5120, "inter": 25600, "n_q": 64, "n_kv": 8}
    return [
        # the smallest call: the Qwen3-0.6B query projection of one token, where launch and host cost are all there is
        {"name": "gemv-1024x2048-1row", "kind": "gemv", "rows": 1, "k": 1024, "n": 2048, "group": 128},
        # an ordinary call at sizes nobody tuned: groups of 32, a column count that is no multiple of sixteen
        {"name": "gemv-ragged-6rows", "kind": "gemv", "rows": 6, "k": 5472, "n": 9000, "group": 32},
        # the benchmark's seven Qwen3-8B projections at one token; four layers, so that the weights are cold
        dict(eight, name="layers-8b-1row", kind="layers", rows=1, layers=4, group=128),
        # the same with as many tokens as the entry point takes (sixteen sequences decoded together)
        dict(eight, name="layers-8b-16rows", kind="layers", rows=16, layers=4, group=128),
        # lm_head of the 8B model for one token
        {"name": "dense-lm-head-1row", "kind": "dense", "rows": 1, "k": 4096, "n": 151936},
        # lm_head of the 32B-shaped model for an odd number of sequences
        {"name": "dense-lm-head-11rows", "kind": "dense", "rows": 11, "k": 5120, "n": 151936},
        # a small model driven launch by launch from Python: the step of someone who does not capture a graph
        dict(small, name="step-small-eager", kind="step", layers=28, vocab=151936, ctx=700, positions=1024, graph=False),
        # the headline: one token of Qwen3-8B at context 4096
        dict(eight, name="step-8b-ctx4096", kind="step", layers=36, vocab=151936, ctx=4096, positions=4224, graph=True),
        # one token of the 32B-shaped model at context 8192, the largest weights
        dict(thirty, name="step-32b-ctx8192", kind="step", layers=64, vocab=151936, ctx=8192, positions=8320, graph=True),
        # a quarter of the 8B layers at a long context: the KV cache outweighs the weights
        dict(eight, name="step-8b-long", kind="step", layers=9, vocab=151936, ctx=40001, positions=40960, graph=True),
        # a few sequences together, of unequal length
        dict(eight, name="batch-8b-3", kind="batch", layers=36, vocab=151936, ctx=2050, positions=2304, rows=3),
        # as many sequences as the library takes
        dict(eight, name="batch-8b-16", kind="batch", layers=36, vocab=151936, ctx=4096, positions=4224, rows=16),
    ]


def _log(rng, low, high, step=1):
    """A multiple of `step` in [low, high], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return min(high // step * step, max(-(-low // step) * step, int(round(v / step)) * step))


def _model_sizes(rng):
    n_kv = rng.choice((2, 4, 8))
    return {"hidden": _log(rng, 1024, 5120, 128), "inter": _log(rng, 2048, 25600, 128),
            "n_q": n_kv * rng.choice((1, 2, 4, 5, 8)), "n_kv": n_kv}


def draw(rng):
    kind = rng.choice(("gemv", "layers", "dense", "step", "batch"))
    rows = 1 if rng.random() < 0.3 else rng.randint(2, 16)
    if kind == "gemv":
        group = rng.choice((32, 64, 128))
        return {"kind": kind, "rows": rows, "k": _log(rng, 512, 25600, group), "n": _log(rng, 512, 25600, 8), "group": group}
    if kind == "layers":
        return dict(_model_sizes(rng), kind=kind, rows=rows, layers=rng.randint(1, 6), group=rng.choice((64, 128)))
    if kind == "dense":
        return {"kind": kind, "rows": rows, "k": _log(rng, 768, 8192, 8), "n": _log(rng, 4000, 151936)}
    ctx = _log(rng, 16, 16384 if kind == "step" else 4096)
    case = dict(_model_sizes(rng), kind=kind, layers=rng.randint(2, 24), vocab=_log(rng, 8000, 151936, 8), ctx=ctx,
                positions=ctx + rng.randint(1, 600))
    if kind == "step":
        return dict(case, graph=rng.random() < 0.7)
    return dict(case, rows=rng.randint(2, 16))


def _shapes(c):
    """(K, N) of the seven projections of a decoder layer."""
    q, kv = c["n_q"] * 128, c["n_kv"] * 128
    return dict(zip(_PROJECTIONS, ((c["hidden"], q), (c["hidden"], kv), (c["hidden"], kv), (q, c["hidden"]),
                                   (c["hidden"], c["inter"]), (c["hidden"], c["inter"]), (c["inter"], c["hidden"]))))


def _codes(shape, gen):
    return torch.randint(-2**31, 2**31, shape, dtype=torch.int32, device="cuda", generator=gen)


def _normal(shape, gen, std=1.0):
    return torch.randn(shape, dtype=torch.bfloat16, device="cuda", generator=gen).mul_(std)


def _projection(K, N, group, gen):
    """Packed weights as the benchmark draws them: uniform codes and zero points, scales U(0.001, 0.02)."""
    scales = torch.rand((K // group, N), device="cuda", generator=gen).mul_(0.019).add_(0.001).half()
    return _codes((K, N // 8), gen), scales, _codes((K // group, N // 8), gen)


def _model_projection(K, N, gen, gain=1.0):
    """The same, scaled so that the product keeps the activations' magnitude (times `gain`)."""
    qweight, scales, qzeros = _projection(K, N, 128, gen)
    return qweight, scales.float().mul_(gain / (0.0105 * 6.6 * math.sqrt(K))).half(), qzeros


def _model(c, gen):
    """Random weights of a trained model's proportions: what a layer adds to the residual stream is small beside the
    stream itself (1 / sqrt(2 layers)), so a rounding in one layer is not blown up by the ones behind it."""
    cfg = decode.ModelConfig(layers=c["layers"], hidden=c["hidden"], intermediate=c["inter"], n_q=c["n_q"],
                             n_kv=c["n_kv"], vocab=c["vocab"])
    into_stream = 1.0 / math.sqrt(2 * c["layers"])
    layers = []
    for _ in range(c["layers"]):
        layer = {"qkv": _model_projection(cfg.hidden, cfg.qkv_out, gen),
                 "o": _model_projection(cfg.n_q * 128, cfg.hidden, gen, into_stream),
                 "gateup": _model_projection(cfg.hidden, 2 * cfg.intermediate, gen),
                 "down": _model_projection(cfg.intermediate, cfg.hidden, gen, into_stream)}
        for name, n in (("in_norm", cfg.hidden), ("post_norm", cfg.hidden), ("q_norm", 128), ("k_norm", 128)):
            layer[name] = _normal((n,), gen, 0.05).add_(1)
        layers.append(layer)
    weights = {"layers": layers, "embed": _normal((cfg.vocab, cfg.hidden), gen),
               "lm_head": _normal((cfg.vocab, cfg.hidden), gen, 0.02), "final_norm": _normal((cfg.hidden,), gen, 0.05).add_(1)}
    return decode.DecodeModel(cfg, c["positions"], weights=weights)


def _captured(launch):
    """`launch` as a HIP graph, after one pass outside it."""
    launch()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        launch()
    return graph


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind = case["kind"]
    if kind == "gemv":
        M, K, N = case["rows"], case["k"], case["n"]
        return {"case": case, "x": _normal((M, K), gen), "w": _projection(K, N, case["group"], gen),
                "y": torch.empty((M, N), dtype=torch.bfloat16, device="cuda"), "ws": capi.make_workspace(M, K, N)}
    if kind == "dense":
        M, K, N = case["rows"], case["k"], case["n"]
        return {"case": case, "x": _normal((M, K), gen), "w": _normal((N, K), gen, 0.02),
                "y": torch.empty((M, N), dtype=torch.bfloat16, device="cuda")}
    if kind == "layers":
        M, shapes = case["rows"], _shapes(case)
        x = {K: _normal((M, K), gen) for K, _ in shapes.values()}
        weights = [{name: _projection(K, N, case["group"], gen) for name, (K, N) in shapes.items()}
                   for _ in range(case["layers"])]
        ys = [{name: torch.empty((M, N), dtype=torch.bfloat16, device="cuda") for name, (_, N) in shapes.items()}
              for _ in range(case["layers"])]
        ws = capi.make_workspace(M, max(K for K, _ in shapes.values()), max(N for _, N in shapes.values()))

        def launch():
            for layer, y in zip(weights, ys):
                for name, (K, _) in shapes.items():
                    capi.gemv_awq_bf16(x[K], *layer[name], y[name], case["group"], ws)

        return {"case": case, "graph": _captured(launch), "keep": (x, weights, ws), "out": ys}

    # a model with a filled KV cache, about to decode the token behind it
    model = _model(case, gen)
    rng = torch.Generator().manual_seed(seed)
    if kind == "batch":
        model = decode.BatchDecodeModel(model, case["rows"])
        lengths = [max(1, case["ctx"] - 5 * b) for b in range(case["rows"])]
        tokens = torch.randint(0, case["vocab"], (case["rows"],), generator=rng).tolist()
    else:
        lengths, tokens = case["ctx"], int(torch.randint(0, case["vocab"], (1,), generator=rng))
    model.prefill_cache_random(lengths, seed=seed)
    model.set_input(tokens, lengths)
    if case.get("graph", True):
        return {"case": case, "graph": _captured(model.step), "model": model}
    return {"case": case, "model": model}


def run(state):
    kind = state["case"]["kind"]
    if kind == "gemv":
        capi.gemv_awq_bf16(state["x"], *state["w"], state["y"], state["case"]["group"], state["ws"])
        return state["y"]
    if kind == "dense":
        capi.gemv_bf16(state["x"], state["w"], state["y"])
        return state["y"]
    if kind == "layers":
        state["graph"].replay()
        return state["out"]
    model = state["model"]
    if "graph" in state:
        state["graph"].replay()
    else:
        model.step()
    # the logits, the residual stream, and the caches of the last layers (the step wrote a row of each)
    return {"logits": model.logits, "x": model.x, "k": model.k_cache[-8:], "v": model.v_cache[-8:]}


def work(case):
    kind, rows = case["kind"], case.get("rows", 1)
    if kind == "gemv":
        return {"bytes": synth.awq_gemv_bytes(rows, case["k"], case["n"], case["group"]),
                "flops": 2 * rows * case["k"] * case["n"]}
    if kind == "dense":
        return {"bytes": synth.bf16_gemv_bytes(rows, case["k"], case["n"]), "flops": 2 * rows * case["k"] * case["n"]}
    shapes = _shapes(case).values()
    weights = sum(K * N for K, N in shapes)
    if kind == "layers":
        return {"bytes": case["layers"] * sum(synth.awq_gemv_bytes(rows, K, N, case["group"]) for K, N in shapes),
                "flops": 2 * rows * case["layers"] * weights}
    # packed weights and lm_head once, every sequence's cache rows once, embedding rows and logits
    positions = sum(max(1, case["ctx"] - 5 * b) + 1 for b in range(rows))
    packed = sum(synth.awq_gemv_bytes(0, K, N, 128) for K, N in shapes)
    cache = positions * case["n_kv"] * 128 * 2 * 2
    head = case["vocab"] * case["hidden"]
    return {"bytes": case["layers"] * (packed + cache) + 2 * head + 2 * rows * (case["hidden"] + case["vocab"]),
            "flops": 2 * rows * (case["layers"] * weights + head) + case["layers"] * 4 * positions * case["n_q"] * 128}


def tolerance(case):
    # one GEMV: products of bf16 numbers added in fp32, one rounding to bf16 (2^-9), whose flips are what differs;
    # a step carries such flips through its layers
    return {"rel": 2e-3} if case["kind"] in ("gemv", "dense", "layers") else {"rel": 1e-2}
