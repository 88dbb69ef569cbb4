"""What a user of this framework has it do, as a list of measurable cases: the quantized linear layer over its range
of rows, widths, shapes and activation types (``QLinear.init`` and ``layer(x)``), the repacking of a GPTQ checkpoint
tensor (``convert_params``), and a Llama-shaped model around them (decode step and prefill).

A case is a dict of plain values; ``prepare`` makes what a program holds before the call, ``run`` is one pass through
the public entry points, ``work`` what the pass cannot do without, ``exact`` the results in 64 bits, ``tolerance`` how far another correct
implementation's results may be off.
"""
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "qfactory-ae_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(1, _PACKAGE)
os.environ.setdefault("QFACTORY_CACHE_DIR", os.path.join(_PACKAGE, "jit_cache"))
os.environ.setdefault("QFACTORY_LOG_LEVEL", "WARNING")

from qfactory import QLinear  # noqa: E402
from qfactory.convert import convert_params  # noqa: E402

NO_SEARCH = {"enable_transform": False, "enable_schedule": False, "enable_lower": False}

# The model cases: the Llama-2-7B layer of decode_llama.py.  Eight layers and the output projection are 0.9 GB of
# packed weights, several times the Infinity Cache, so a layer's cost is that of the full 32.
MODEL_LAYERS, HIDDEN, HEADS, MLP, VOCAB, MAX_LEN = 8, 4096, 32, 11008, 32000, 256


def _linear(name, M, N, K, nbits=4, gs=128, sym=False, dtype="fp16"):
    case = {"kind": "linear", "M": M, "N": N, "K": K, "nbits": nbits, "gs": gs, "sym": sym, "dtype": dtype}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one token through an attention output projection: the smallest call, all launch and latency
        _linear("linear 1x4096x4096 w4", 1, 4096, 4096),
        # one token through the down projection of a 70B-sized layer: the longest rows, a plain read of the weights
        _linear("linear 1x28672x8192 w4", 1, 8192, 28672),
        # a few sequences (or the candidates of speculative decoding) against 2-bit weights in short groups
        _linear("linear 4x8192x8192 w2", 4, 8192, 8192, nbits=2, gs=64, sym=True),
        # sixteen sequences through a 7B down projection: the ordinary batched decode call
        _linear("linear 16x11008x4096 w4", 16, 4096, 11008),
        # sixty-four sequences through a 7B gate+up projection: the largest ordinary decode batch
        _linear("linear 64x4096x22016 w4", 64, 22016, 4096),
        # a server's mixed batch (decode rows and a chunk of a prompt), bf16 activations, a 70B-sized qkv projection
        _linear("linear 200x8192x10240 w4 bf16", 200, 10240, 8192, dtype="bf16"),
        # a prompt of odd length through 8-bit symmetric weights
        _linear("linear 333x8192x8192 w8", 333, 8192, 8192, nbits=8, sym=True),
        # prefill of 64 prompts of 128 tokens through a 7B qkv projection: the largest call
        _linear("linear 8192x4096x12288 w4", 8192, 12288, 4096),
        # loading a layer: GPTQ tensors (int32 fields, fp16 scales, zero-points) to the packed layout, on the device
        {"name": "convert 4096x22016 w4", "kind": "convert", "N": 22016, "K": 4096, "nbits": 4, "gs": 128, "sym": False},
        # one decode step as the decode loop runs it (one HIP-graph replay): a single sequence, and a batch of 64
        {"name": "decode batch 1", "kind": "decode", "batch": 1, "pos": 190},
        {"name": "decode batch 64", "kind": "decode", "batch": 64, "pos": 190},
        # the prompt of eight sequences of 128 tokens
        {"name": "prefill 8x128", "kind": "prefill", "batch": 8, "tokens": 128},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """Another case of the same ranges: rows, columns, depth and batch spread over their logarithms."""
    kind = rng.choices(["linear", "plain", "convert", "decode", "prefill"], [14, 1, 2, 2, 2])[0]
    if kind == "decode":
        return {"kind": "decode", "batch": _log_int(rng, 1, 96), "pos": rng.randint(16, MAX_LEN - 1)}
    if kind == "prefill":
        tokens = rng.randint(17, MAX_LEN)
        return {"kind": "prefill", "batch": max(1, _log_int(rng, 32, 1024) // tokens), "tokens": tokens}
    nbits = rng.choices([4, 8, 2, 3], [6, 2, 1, 1])[0]
    gs = rng.choices([128, 64, 32], [7, 2, 1])[0]
    sym = rng.random() < 0.4
    # hidden sizes are multiples of 256 (and whole bytes of zero-points: of four groups at 2 bits); output columns any number
    unit = max(256, 4 * gs) if nbits == 2 else 256
    while True:
        K = max(1, _log_int(rng, 1024, 28672) // unit) * unit
        N = _log_int(rng, 1024, 57344)
        N = N if rng.random() < 0.2 else max(64, N // 64 * 64)
        if N * K <= 57344 * 8192:
            break
    if kind == "convert":
        return {"kind": "convert", "N": N, "K": K, "nbits": nbits, "gs": gs, "sym": sym}
    if kind == "plain":
        return _linear(None, rng.randint(1, 4), N, K, nbits, -1, True)
    M = _log_int(rng, 1, 8192)
    M = min(M, max(1, 8192 * 12288 * 4096 // (N * K)))
    return _linear(None, M, N, K, nbits, gs, sym, "bf16" if rng.random() < 0.25 else "fp16")


def _gptq_tensors(case, gen):
    """GPTQ-orientation tensors: fields in a bell around the zero-point, positive scales, zero-points near the middle."""
    K, N, nbits, gs = case["K"], case["N"], case["nbits"], case["gs"]
    top, half = 2 ** nbits - 1, 2 ** (nbits - 1)
    weight = torch.empty(K, N, dtype=torch.int32, device="cuda")
    for k in range(0, K, 1024):                                  # in pieces: the float draws of a large layer would be 2 GB
        rows = torch.randn(min(1024, K - k), N, device="cuda", generator=gen)
        weight[k:k + rows.shape[0]] = rows.mul_(2 ** nbits / 5.0).add_(half).round_().clamp_(0, top).to(torch.int32)
    if gs == -1:
        return weight, None, None
    scale = (torch.rand(K // gs, N, device="cuda", generator=gen) * 0.019 + 0.001).to(torch.float16)
    zero = None
    if not case["sym"]:
        zero = torch.randint(max(0, half - 3), min(top, half + 2) + 1, (K // gs, N), dtype=torch.int32, device="cuda", generator=gen)
    return weight, scale, zero


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] == "linear":
        dtype = torch.bfloat16 if case["dtype"] == "bf16" else torch.float16
        weight, scale, zero = _gptq_tensors(case, gen)
        layer = QLinear.init(case["M"], case["K"], case["N"], case["nbits"], weight, case["gs"], scale, zero,
                             compile_flags=NO_SEARCH)
        x = torch.randn(case["M"], case["K"], device="cuda", generator=gen).to(dtype)
        if dtype is torch.bfloat16:
            layer.func_for(case["M"], dtype)                     # the bf16 specialisation is compiled where a server warms up
        return {"kind": "linear", "layer": layer, "x": x}
    if case["kind"] == "convert":
        weight, scale, zero = _gptq_tensors(case, gen)
        return {"kind": "convert", "args": {"K": case["K"], "N": case["N"], "NBITS": case["nbits"], "GS": case["gs"]},
                "params": (weight, scale, zero)}

    import decode_llama
    shape = decode_llama.LlamaShape(layers=MODEL_LAYERS, hidden=HIDDEN, heads=HEADS, mlp=MLP, vocab=VOCAB, max_len=MAX_LEN)
    batch = case["batch"]
    model = decode_llama.QuantLlama(shape, batch, seed)
    if case["kind"] == "prefill":
        tokens = torch.randint(0, VOCAB, (batch, case["tokens"]), device="cuda", generator=gen)
        pos = torch.arange(case["tokens"], device="cuda")
        model.prefill(tokens, pos)                               # first use of the prompt's row count: compiled here
        return {"kind": "prefill", "model": model, "tokens": tokens, "pos": pos}
    for cache in (model.k_cache, model.v_cache):
        for layer in cache:
            layer[:, :, :case["pos"]] = torch.randn(batch, HEADS, case["pos"], HIDDEN // HEADS, device="cuda", generator=gen)
    tok = torch.randint(0, VOCAB, (batch, 1), device="cuda", generator=gen)
    pos = torch.full((1,), case["pos"], dtype=torch.int64, device="cuda")
    model.decode_step(tok, pos)                                  # compiled and warmed up outside the capture
    torch.cuda.synchronize()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
        logits = model.decode_step(tok, pos)
    torch.cuda.current_stream().wait_stream(side)
    return {"kind": "decode", "model": model, "graph": graph, "tok": tok, "pos": pos, "logits": logits}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "convert":
        return convert_params(state["args"], state["params"])
    model = state["model"]
    if kind == "prefill":
        logits = model.prefill(state["tokens"], state["pos"])
    else:
        state["graph"].replay()
        logits = state["logits"]
    return {"logits": logits, "k": model.k_cache, "v": model.v_cache}


def _linear_work(M, N, K, nbits, gs, sym):
    """The layer's packed tensors once, the activations once, the output once."""
    weights = N * K * nbits // 8
    if gs != -1:
        groups = N * (K // gs)
        weights += groups * 2 + (0 if sym else groups * (4 if nbits == 3 else nbits) // 8)
    return weights + 2 * M * (K + N), 2 * M * N * K


def work(case):
    if case["kind"] == "linear":
        nbytes, flops = _linear_work(case["M"], case["N"], case["K"], case["nbits"], case["gs"], case["sym"])
        return {"bytes": nbytes, "flops": flops}
    if case["kind"] == "convert":
        N, K, nbits, groups = case["N"], case["K"], case["nbits"], case["N"] * (case["K"] // case["gs"])
        packed = N * K * nbits // 8 + groups * 2 + (0 if case["sym"] else groups * (4 if nbits == 3 else nbits) // 8)
        return {"bytes": 4 * K * N + 2 * groups + (0 if case["sym"] else 4 * groups) + packed, "flops": 0}
    rows = case["batch"] * case.get("tokens", 1)
    nbytes = flops = 0
    for N, K in ((3 * HIDDEN, HIDDEN), (HIDDEN, HIDDEN), (2 * MLP, HIDDEN), (HIDDEN, MLP)):
        weights, ops = _linear_work(0, N, K, 4, 128, False)[0], 2 * rows * N * K
        nbytes, flops = nbytes + weights, flops + ops
    if case["kind"] == "decode":                                 # the cached keys and values, and every head's scores and sums
        nbytes += 2 * 2 * case["batch"] * HIDDEN * case["pos"]
        flops += 4 * case["batch"] * HIDDEN * case["pos"]
    else:                                                        # the new keys and values are written; causal scores and sums
        nbytes += 2 * 2 * rows * HIDDEN
        flops += 2 * rows * HIDDEN * case["tokens"]
    head = _linear_work(case["batch"], VOCAB, HIDDEN, 4, 128, False)
    return {"bytes": MODEL_LAYERS * nbytes + head[0], "flops": MODEL_LAYERS * flops + head[1]}


def tolerance(case):
    if case["kind"] == "convert":
        return "exact"
    if case["kind"] == "linear":
        if case["dtype"] == "bf16":
            # one rounding to bf16: 1.7e-3 and 4e-3 measured against sums in 64 bits
            return {"rel": 4e-3, "max": 2e-2}
        # one rounding to fp16, and to fp16 of every weight or not: 2.8e-4 and 1.3e-3 measured against sums in 64 bits
        return {"rel": 1e-3, "max": 5e-3}
    # eight layers of fp16 roundings between the linears: 8.5e-4 and 6e-3 measured against the same model with
    # PyTorch operations there
    return {"rel": 4e-3, "max": 3e-2}


def _exact_linear(x, q, zero, scale, gs):
    """``x @ ((q - zero) * scale)`` in 64 bits: q (K, N), zero and scale (K / gs, N)."""
    w = q.to(torch.float64)
    if scale is not None:
        w = ((w.reshape(-1, gs, q.shape[1]) - zero.to(torch.float64)[:, None]) * scale.to(torch.float64)[:, None]).reshape(q.shape)
    return x @ w


def _packed_fields(t):
    """The sixteen values of a byte pair's four-bit fields, in the order of the elements: (rows, bytes) -> (rows, 2 * bytes).
    In a word the even elements fill the low half, the odd ones the high half."""
    b = t.view(torch.uint8).reshape(t.shape[0], -1, 4)
    nibbles = torch.stack((b & 15, b >> 4), dim=-1).reshape(t.shape[0], -1, 2, 4)
    return nibbles.transpose(2, 3).reshape(t.shape[0], -1)


def _exact_model(case, seed):
    """Logits and caches of the model cases in 64 bits: the same random packed tensors, plain matrix products, no fp16 between the steps."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    batch, hd, f64 = case["batch"], HIDDEN // HEADS, torch.float64
    weights = torch.Generator(device="cuda").manual_seed(seed)
    embed = (torch.randn(VOCAB, HIDDEN, device="cuda", generator=weights) * 0.5).to(torch.float16)

    def linear(K, N):
        w = torch.randint(-128, 128, (N, K // 2), dtype=torch.int8, device="cuda", generator=weights)
        z = torch.randint(-128, 128, (N, K // 256), dtype=torch.int8, device="cuda", generator=weights).view(torch.uint8)
        s = ((torch.rand(N, K // 128, device="cuda", generator=weights) + 0.5) * (0.5 / (16 * 0.41 * K ** 0.5))).to(torch.float16)
        zero = torch.stack((z & 15, z >> 4), dim=-1).reshape(N, K // 128)
        return lambda x: _exact_linear(x, _packed_fields(w).T, zero.T, s.T, 128)

    layers = [[linear(HIDDEN, 3 * HIDDEN), linear(HIDDEN, HIDDEN), linear(HIDDEN, 2 * MLP), linear(MLP, HIDDEN)] for _ in range(MODEL_LAYERS)]
    head = linear(HIDDEN, VOCAB)
    k_cache = torch.zeros(MODEL_LAYERS, batch, HEADS, MAX_LEN, hd, dtype=f64, device="cuda")
    v_cache = torch.zeros_like(k_cache)
    if case["kind"] == "prefill":
        tokens = torch.randint(0, VOCAB, (batch, case["tokens"]), device="cuda", generator=gen)
        pos = torch.arange(case["tokens"], device="cuda")
    else:
        for cache in (k_cache, v_cache):
            for layer in cache:
                layer[:, :, :case["pos"]] = torch.randn(batch, HEADS, case["pos"], hd, device="cuda", generator=gen).to(torch.float16)
        tokens = torch.randint(0, VOCAB, (batch, 1), device="cuda", generator=gen)
        pos = torch.full((1,), case["pos"], dtype=torch.int64, device="cuda")
    T = tokens.shape[1]
    angle = pos.to(f64)[:, None] / 10000.0 ** (torch.arange(0, hd, 2, device="cuda", dtype=f64) / hd)[None]
    cos, sin = angle.cos(), angle.sin()
    hidden = (torch.arange(MAX_LEN, device="cuda")[None] > pos[:, None])[None, None]

    def norm(x):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5)

    def rope(x):
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack((a * cos - b * sin, a * sin + b * cos), dim=-1).flatten(-2)

    x = embed[tokens].to(f64).reshape(batch * T, HIDDEN)
    for li, (qkv, o, gate_up, down) in enumerate(layers):
        q, k, v = qkv(norm(x)).reshape(batch, T, 3, HEADS, hd).permute(2, 0, 3, 1, 4)
        k_cache[li][:, :, pos], v_cache[li][:, :, pos] = rope(k), v
        scores = (rope(q) @ k_cache[li].transpose(-1, -2).contiguous()) * hd ** -0.5
        att = scores.masked_fill(hidden, float("-inf")).softmax(-1) @ v_cache[li]
        x = x + o(att.transpose(1, 2).reshape(batch * T, HIDDEN))
        gate, up = gate_up(norm(x)).split(MLP, dim=1)
        x = x + down(gate / (1 + torch.exp(-gate)) * up)
    return {"logits": head(norm(x.reshape(batch, T, HIDDEN)[:, -1])), "k": k_cache, "v": v_cache}


def exact(case, seed):
    """What ``run`` returns for these inputs, in 64 bits and without this repository's kernels."""
    if case["kind"] in ("decode", "prefill"):
        return _exact_model(case, seed)
    if case["kind"] == "convert":
        return None                                              # packed bytes: compared bit for bit
    gen = torch.Generator(device="cuda").manual_seed(seed)
    weight, scale, zero = _gptq_tensors(case, gen)
    x = torch.randn(case["M"], case["K"], device="cuda", generator=gen).to(torch.bfloat16 if case["dtype"] == "bf16" else torch.float16)
    top = 2 ** case["nbits"] - 1
    if scale is not None:                                        # GPTQ stores the zero-point less one; the packed form clamps the sum
        zero = torch.full_like(scale, (top + 1) // 2) if zero is None else (zero + 1).clamp(max=top)
    return _exact_linear(x.to(torch.float64), weight, zero, scale, case["gs"])
