"""The work that users of this package have it do, as cases to be timed: five kinds of call, each through the
package's public entry points.

  round_trip   MSECompressor.compress, then MSECompressor.decompress (to float32), one tensor: a script that studies one
               layer's keys, or a compressor used on its own
  layer        TurboQuantV3.compress_kv, then decompress_kv, keys and values of one layer with a window of recent
               tokens left as they are: prefill of a layer, and its cache handed back to the model
  cache        every layer's keys and values in one launch per code width and direction (JobList): a whole cache
               parked and brought back
  update       one decode step of V3Cache.update on every layer: the new token joins the window, the oldest one is
               compressed, the full-length keys and values come back
  attend       one decode step of V3Cache.append + V3Cache.attend on every layer: attention from the packed store
  v2           TurboQuantCompressorV2.compress, then asymmetric_attention_scores, keys of one layer

Decode steps move their cache on by a token, as they do in use: the histories are long, or the steps many layers deep,
so that a timed run adds little to them.
"""
import math

import torch

import turboquant_amd as tq

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
DEVICE = "cuda"


def listed():
    return [
        # the smallest call: 8192 float32 keys at 4 bits there and back; latency and launches count
        {"name": "round_trip 8k f32", "kind": "round_trip", "dtype": "f32", "batch": 1, "heads": 8, "tokens": 1024, "dim": 128, "bits": 4},
        # float32 states of an ordinary prompt, four sequences, a token count that fills no tile evenly
        {"name": "round_trip 131k f32", "kind": "round_trip", "dtype": "f32", "batch": 4, "heads": 8, "tokens": 4099, "dim": 128, "bits": 4},
        # one layer of a long bf16 prompt (8 KV heads), K4/V2 with the default window
        {"name": "layer 32k bf16", "kind": "layer", "dtype": "bf16", "batch": 1, "heads": 8, "tokens": 32768, "dim": 128, "key_bits": 4, "value_bits": 2, "window": 128},
        # one layer of a batch of eight fp16 prompts (2 KV heads), K6/V4: the widths recommended for generation
        {"name": "layer 8x4k f16", "kind": "layer", "dtype": "f16", "batch": 8, "heads": 2, "tokens": 4096, "dim": 128, "key_bits": 6, "value_bits": 4, "window": 128},
        # 256-wide heads
        {"name": "layer d256", "kind": "layer", "dtype": "bf16", "batch": 1, "heads": 8, "tokens": 16384, "dim": 256, "key_bits": 4, "value_bits": 2, "window": 128},
        # 80-wide heads (no multiple of 32), two prompts of an odd length
        {"name": "layer d80", "kind": "layer", "dtype": "f16", "batch": 2, "heads": 16, "tokens": 6001, "dim": 80, "key_bits": 4, "value_bits": 4, "window": 128},
        # the headline workload: 32 layers x 8 KV heads x 32768 tokens, bf16, K4/V2, first and last four layers at 8 bits
        {"name": "cache 32k", "kind": "cache", "dtype": "bf16", "layers": 32, "batch": 1, "heads": 8, "tokens": 32768, "dim": 128, "key_bits": 4, "value_bits": 2, "protected": 4},
        # decode of sixteen sequences through a model's own attention: the whole history de-quantised for every token
        {"name": "update 16x16k", "kind": "update", "dtype": "bf16", "layers": 8, "batch": 16, "heads": 8, "tokens": 16384, "dim": 128, "key_bits": 4, "value_bits": 2, "window": 128},
        # decode from the packed store: many sequences, where the packed bytes count ...
        {"name": "attend 64x16k", "kind": "attend", "dtype": "bf16", "layers": 8, "batch": 64, "heads": 8, "q_heads": 32, "tokens": 16384, "dim": 128, "key_bits": 4, "value_bits": 2, "window": 128},
        # ... and one long sequence, where launches do
        {"name": "attend 1x32k", "kind": "attend", "dtype": "bf16", "layers": 32, "batch": 1, "heads": 8, "q_heads": 32, "tokens": 32768, "dim": 128, "key_bits": 4, "value_bits": 2, "window": 128},
        # the same step of a model with 64-wide heads, K6/V4
        {"name": "attend d64", "kind": "attend", "dtype": "f16", "layers": 16, "batch": 4, "heads": 8, "q_heads": 32, "tokens": 6000, "dim": 64, "key_bits": 6, "value_bits": 4, "window": 128},
        # V2 keys (2-bit codes and one sign bit), one layer, one query token per head
        {"name": "v2 32k", "kind": "v2", "dtype": "bf16", "batch": 1, "heads": 8, "tokens": 32768, "dim": 128, "bits": 3, "queries": 1},
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, evenly over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges that the listed ones stand for."""
    kind = rng.choice(("round_trip", "layer", "layer", "cache", "update", "attend", "attend", "v2"))
    half = rng.choice(("bf16", "bf16", "f16"))
    key_bits, value_bits = rng.choice(((4, 2), (4, 2), (4, 4), (6, 4), (8, 4), (3, 2), (8, 8)))
    batch, heads = rng.choice((1, 1, 2, 4, 8, 16)), rng.choice((1, 2, 4, 8, 8, 16))
    rows = batch * heads
    if kind == "round_trip":
        return {"kind": kind, "dtype": rng.choice(("f32", half)), "batch": batch, "heads": heads, "tokens": max(1, _spread(rng, 1 << 9, 1 << 18) // rows),
                "dim": rng.choice((64, 128, 128, 256)), "bits": rng.choice((2, 3, 4, 4, 6, 8))}
    if kind == "layer":
        window = rng.choice((0, 64, 128, 128))
        return {"kind": kind, "dtype": half, "batch": batch, "heads": heads, "tokens": window + max(1, _spread(rng, 1 << 11, 1 << 19) // rows),
                "dim": rng.choice((64, 80, 96, 128, 128, 128, 256)), "key_bits": key_bits, "value_bits": value_bits, "window": window}
    if kind == "cache":
        layers = rng.choice((16, 24, 28, 32, 36))
        return {"kind": kind, "dtype": half, "layers": layers, "batch": 1, "heads": heads, "tokens": max(64, _spread(rng, 1 << 13, 1 << 18) // heads),
                "dim": rng.choice((64, 80, 96, 128, 128, 128)), "key_bits": key_bits, "value_bits": value_bits, "protected": rng.choice((0, 2, 4))}
    heads = min(heads, 8)
    rows = batch * heads
    if kind == "update":
        return {"kind": kind, "dtype": half, "layers": rng.choice((16, 24, 32)), "batch": batch, "heads": heads, "tokens": max(1024, _spread(rng, 1 << 14, 1 << 19) // rows),
                "dim": rng.choice((64, 96, 128, 128, 128)), "key_bits": key_bits, "value_bits": value_bits, "window": 128}
    if kind == "attend":
        dim = rng.choice((64, 96, 128, 128, 128, 256))
        return {"kind": kind, "dtype": half, "layers": rng.choice((16, 24, 32)), "batch": batch, "heads": heads, "q_heads": heads * rng.choice((1, 2, 4, 4, 7, 8)),
                "tokens": max(1024, _spread(rng, 1 << 14, 1 << (20 if dim <= 128 else 19)) // rows), "dim": dim, "key_bits": key_bits, "value_bits": value_bits, "window": 128}
    return {"kind": kind, "dtype": half, "batch": batch, "heads": heads, "tokens": max(1, _spread(rng, 1 << 11, 1 << 19) // rows), "dim": 128,
            "bits": rng.choice((2, 3, 3, 4)), "queries": rng.choice((1, 1, 2, 5))}


def _states(g, shape, dtype):
    """Keys or values: N(0,1) with log-normal channel scales (a few outlier channels) and token norms spread over a factor of four."""
    x = torch.randn(shape, generator=g, device=DEVICE, dtype=torch.float32)
    x *= torch.exp(torch.randn(shape[-1], generator=g, device=DEVICE))
    x *= 0.5 + 1.5 * torch.rand(shape[:-1] + (1,), generator=g, device=DEVICE)
    return x.to(dtype)


def _width(dim, bits):
    return -(-dim // (8 // bits))


def prepare(case, seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    c, dtype = case, DTYPES[case["dtype"]]
    shape = (c["batch"], c["heads"], c["tokens"], c["dim"])
    if c["kind"] == "round_trip":
        return {"kind": "round_trip", "comp": tq.MSECompressor(c["dim"], c["bits"], seed=42, device=DEVICE), "x": _states(g, shape, dtype)}
    if c["kind"] == "layer":
        comp = tq.TurboQuantV3(c["dim"], key_bits=c["key_bits"], value_bits=c["value_bits"], residual_window=c["window"], layer_idx=8, device=DEVICE)
        return {"kind": "layer", "comp": comp, "k": _states(g, shape, dtype), "v": _states(g, shape, dtype)}
    if c["kind"] == "cache":
        return _prepare_cache(c, g, shape, dtype)
    if c["kind"] == "v2":
        return {"kind": "v2", "comp": tq.TurboQuantCompressorV2(c["dim"], c["bits"], seed=42, device=DEVICE), "x": _states(g, shape, dtype),
                "q": _states(g, (c["batch"], c["heads"], c["queries"], c["dim"]), dtype)}
    # decode: a prefilled cache, and the new token (and query) of the step
    cache = tq.V3Cache(key_bits=c["key_bits"], value_bits=c["value_bits"], residual_window=c["window"], n_layers=c["layers"], capacity=c["tokens"] + 4096)
    history = shape[:2] + (c["tokens"] + c["window"], c["dim"])
    for layer in range(c["layers"]):
        cache.append(_states(g, history, dtype), _states(g, history, dtype), layer)
    token = shape[:2] + (1, c["dim"])
    state = {"kind": c["kind"], "cache": cache, "layers": c["layers"], "k": [_states(g, token, dtype) for _ in range(c["layers"])],
             "v": [_states(g, token, dtype) for _ in range(c["layers"])]}
    if c["kind"] == "attend":
        # queries of unit channels: logits of the size that attention layers see
        state["q"] = [torch.randn((c["batch"], c["q_heads"], 1, c["dim"]), generator=g, device=DEVICE).to(dtype) for _ in range(c["layers"])]
    return state


def _prepare_cache(c, g, shape, dtype):
    """Per code width one job list per direction; packed buffers and de-quantised tensors of a width lie in one allocation each."""
    by_bits = {}
    for layer in range(c["layers"]):
        comp = tq.TurboQuantV3(c["dim"], key_bits=c["key_bits"], value_bits=c["value_bits"], residual_window=0, layer_idx=layer, n_layers=c["layers"],
                               protected_layers=c["protected"], device=DEVICE)
        for one in (comp.key_compressor, comp.val_compressor):
            by_bits.setdefault(one.bits, []).append((one, _states(g, shape, dtype)))
    groups = {}
    for bits, members in by_bits.items():
        n, device = len(members), members[0][1].device
        idx = torch.empty((n,) + shape[:3] + (_width(c["dim"], bits),), dtype=torch.uint8, device=DEVICE)
        norms = torch.empty((n,) + shape[:3], dtype=torch.float16, device=DEVICE)
        out = torch.empty((n,) + shape, dtype=dtype, device=DEVICE)
        jobs = [{"states": x, "idx_bytes": idx[i], "vec_norms": norms[i], "table": one.table(), "bits": bits} for i, (one, x) in enumerate(members)]
        back = [dict(j, states=out[i]) for i, j in enumerate(jobs)]
        groups[bits] = {"compress": tq._native.JobList(jobs, device), "decompress": tq._native.JobList(back, device), "idx": idx, "norms": norms, "out": out}
    return {"kind": "cache", "groups": groups}


def run(state):
    kind = state["kind"]
    if kind == "round_trip":
        packed = state["comp"].compress(state["x"])
        return packed, state["comp"].decompress(packed)
    if kind == "layer":
        k, v = state["comp"].compress_kv(state["k"], state["v"])
        return k["compressed"], v["compressed"], state["comp"].decompress_kv(k, v)
    if kind == "cache":
        groups = [state["groups"][bits] for bits in sorted(state["groups"])]
        for group in groups:
            group["compress"].compress()
        for group in groups:
            group["decompress"].decompress()
        return [(group["idx"], group["norms"], group["out"]) for group in groups]
    if kind == "v2":
        packed = state["comp"].compress(state["x"])
        return packed, state["comp"].asymmetric_attention_scores(state["q"], packed)
    cache, out = state["cache"], []
    for layer in range(state["layers"]):
        if kind == "update":
            out.append(cache.update(state["k"][layer], state["v"][layer], layer))
        else:
            cache.append(state["k"][layer], state["v"][layer], layer)
            out.append(cache.attend(state["q"][layer], layer))
    return out


def work(case):
    """Every tensor of a pass crosses memory once: states in, packed form out, packed form in, de-quantised tensor (or scores) out.
    The rotation of a vector is counted once per direction, attention as its two products."""
    c, dim = case, case["dim"]
    elem = 4 if c["dtype"] == "f32" else 2
    rotation = 2.0 * dim * dim
    rows = c["batch"] * c["heads"]
    packed = lambda bits: _width(dim, bits) + 2  # noqa: E731
    if c["kind"] == "round_trip":
        n = rows * c["tokens"]
        return {"bytes": n * (dim * elem + 2 * packed(c["bits"]) + dim * 4), "flops": n * 2 * rotation}
    if c["kind"] == "layer":
        n, window = rows * (c["tokens"] - c["window"]), rows * c["window"]
        return {"bytes": n * (4 * dim * elem + 2 * (packed(c["key_bits"]) + packed(c["value_bits"]))) + window * 4 * dim * elem, "flops": n * 4 * rotation}
    if c["kind"] == "cache":
        # a layer is protected if it lies among the first or last `protected` ones
        wide = min(2 * c["protected"], c["layers"])
        widths = [8, 8] * wide + [c["key_bits"], c["value_bits"]] * (c["layers"] - wide)
        n = rows * c["tokens"]
        return {"bytes": sum(n * (2 * dim * elem + 2 * packed(b)) for b in widths), "flops": len(widths) * n * 2 * rotation}
    if c["kind"] == "v2":
        n, mse_bits = rows * c["tokens"], max(c["bits"] - 1, 1)
        stored = packed(mse_bits) + -(-dim // 8) + 2
        q = rows * c["queries"]
        return {"bytes": n * (dim * elem + 2 * stored + 4 * c["queries"]) + q * dim * elem, "flops": n * (2 * rotation + 4.0 * dim * c["queries"])}
    both = packed(c["key_bits"]) + packed(c["value_bits"])
    one_token = rows * (2 * dim * elem + both)          # the new token read, the leaving one written packed
    window = rows * c["window"] * 2 * dim * elem
    if c["kind"] == "update":
        out = rows * (c["tokens"] + c["window"] + 1) * 2 * dim * elem
        return {"bytes": c["layers"] * (rows * c["tokens"] * both + out + window + one_token), "flops": c["layers"] * rows * c["tokens"] * 2 * rotation}
    queries = c["batch"] * c["q_heads"]
    return {"bytes": c["layers"] * (rows * c["tokens"] * both + window + one_token + 2 * queries * dim * elem),
            "flops": c["layers"] * queries * (c["tokens"] + c["window"]) * 4.0 * dim}


def tolerance(case):
    """About four times what the path differs by from itself in float64 on the same inputs.  A coordinate within the rounding
    of a decision boundary falls to either side of it: up to 8e-5 of the bytes differ (8-bit codes of bf16 vectors; 1.2e-4 of the
    sign bytes of v2), and one such code moves single elements of its de-quantised vector by up to half their size (2-bit
    codes), the tensor as a whole by no more than its rounding: 0.4-0.5e-3 in float32 and float16, 0.9-2.0e-3 in bfloat16.
    Attention: 0.7-1.0e-3 in float16, 1.7-2.4e-3 in bfloat16, single elements 1.5e-2; v2 scores 2.4e-3."""
    if case["kind"] == "attend":
        return {"rel": 4e-3 if case["dtype"] == "f16" else 8e-3, "max": 0.06}
    return {"rel": 8e-3 if case["dtype"] == "bf16" or case["kind"] == "v2" else 2e-3, "max": 0.9, "differ": 5e-4}
