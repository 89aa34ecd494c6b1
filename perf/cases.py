"""Performance cases: the work that users of this library give it, through its public entry points.

Four kinds of case, each with sizes from this repository's configurations, benchmark and tests or generic ones:

* linears   the quantized linears of one transformer layer through Matrix::mulBatched, call by call, as a graph engine that
            runs op by op issues them (decode at 1 token, batched decode at 2..16, prompts beyond)
* decode    DecodeModel::run: n greedy tokens of a batch-1 model from a given position
* sample    DecodeModel::reset / step / logits, one token at a time with the pick on the host, as a caller with a sampler of
            its own does (the reference copies the logits back for every token)
* prompt    DecodeModel::prefill: T tokens at once, from an empty cache or behind earlier turns
* quantize  a BF16 weight to FP8 or FP4 on the device and back to BF16 (loading an unquantized model; its dequantized copy)

Weights are normal values of the spread that trained weights have, activations are unit normal.  The models are random but
well behaved: the norm weights keep the projections at unit spread and a layer's MLP contribution small against the residual
stream, and row t + 1 of the head is parallel to the embedding of token t (tied heads: row t), so that the next token stands
clear of all others as a trained model's mostly does and greedy decoding does not hang on the last bit of a logit.
"""
import importlib
import math

import numpy as np
import torch

pkg = importlib.import_module("cccc-lite_amd")
HALF, BF16, E4M3, E5M2, FP4 = 2, 3, 4, 5, 6

# weight format -> (type, codes quantized on the device with a per-tensor or per-block scale, spread of the weights: an FP4 block
# scale is amax / 6 as an E4M3 number, whose smallest step is 0.002)
FORMATS = {"e5m2": (E5M2, False, 0.02), "e5m2_scaled": (E5M2, True, 0.02), "e4m3_scaled": (E4M3, True, 0.02), "fp4": (FP4, True, 0.03)}

MODEL_8B_QK = dict(layers=36, hidden=4096, n_q=32, n_kv=8, inter=12288, vocab=151936, qk_norm=True, tied=False)      # the Qwen3-8B shape
MODEL_8B = dict(layers=32, hidden=4096, n_q=32, n_kv=8, inter=14336, vocab=128256, qk_norm=False, tied=False)        # the Llama-3.1-8B shape
MODEL_SMALL = dict(layers=12, hidden=1024, n_q=16, n_kv=8, inter=3072, vocab=32000, qk_norm=True, tied=True)
MODEL_LONG = dict(layers=8, hidden=4096, n_q=32, n_kv=8, inter=12288, vocab=151936, qk_norm=True, tied=False)


def listed():
    return [
        # one token through a layer of the 8B model, op by op on the file layout: the smallest calls, where latency counts
        dict(name="linears_e5m2_1_token", kind="linears", weight="e5m2", act="bf16", tiled=False, tokens=1, hidden=4096, kv=1024, inter=12288),
        # four sequences decoded together on block-scaled FP4 weights
        dict(name="linears_fp4_4_tokens", kind="linears", weight="fp4", act="bf16", tiled=True, tokens=4, hidden=4096, kv=1024, inter=14336),
        # sixteen sequences decoded together (the largest batch the matrix-vector kernels take), tiled copies as the loader makes them
        dict(name="linears_e5m2_16_tokens", kind="linears", weight="e5m2", act="bf16", tiled=True, tokens=16, hidden=4096, kv=1024, inter=12288),
        # a ragged prompt through one layer of a HALF graph, weights quantized on load with a per-tensor scale
        dict(name="linears_half_301_tokens", kind="linears", weight="e4m3_scaled", act="half", tiled=True, tokens=301, hidden=4096, kv=1024, inter=12288),
        # greedy generation at the context the benchmark is quoted on
        dict(name="decode_8b_e5m2_at_4096", kind="decode", weight="e5m2", pos=4064, steps=32, exact=False, **MODEL_8B_QK),
        # greedy generation of a short chat answer on FP4 weights
        dict(name="decode_8b_fp4_at_640", kind="decode", weight="fp4", pos=640, steps=32, exact=False, **MODEL_8B),
        # a small model with tied embeddings, sampled on the host, every rounding point of the reference kept
        dict(name="sample_small_at_300", kind="sample", weight="e4m3_scaled", pos=300, steps=4, exact=True, **MODEL_SMALL),
        # generation behind a long document: the attention over the cache weighs as much as the weights
        dict(name="decode_long_at_32000", kind="decode", weight="e5m2_scaled", pos=32000, steps=8, exact=False, **MODEL_LONG),
        # a full prompt piece on a model that keeps tiled copies for its prompts
        dict(name="prompt_8b_e5m2_2048", kind="prompt", weight="e5m2", pos=0, tokens=2048, repack=True, **MODEL_8B_QK),
        # a short question on the layout a batch-1 model keeps
        dict(name="prompt_8b_e5m2_100", kind="prompt", weight="e5m2", pos=0, tokens=100, repack=False, **MODEL_8B_QK),
        # the next turn of a conversation: 512 tokens behind 3000 on FP4 weights
        dict(name="prompt_8b_fp4_512_at_3000", kind="prompt", weight="fp4", pos=3000, tokens=512, repack=True, **MODEL_8B),
        # loading an unquantized MLP weight as FP4
        dict(name="quantize_fp4_mlp", kind="quantize", weight="fp4", n_out=12288, K=4096),
    ]


def _log(rng, lo, hi, step=1):
    """lo..hi in multiples of step, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    weight = rng.choice(sorted(FORMATS))
    kind = rng.choice(["linears", "linears", "linears", "decode", "decode", "sample", "prompt", "prompt", "quantize"])
    if kind == "quantize":
        return dict(kind=kind, weight=weight, n_out=_log(rng, 256, 16384), K=_log(rng, 256, 16384, 32))
    if kind == "linears":
        act = "half" if weight != "fp4" and rng.random() < 0.2 else "bf16"
        tiled = weight == "fp4" or rng.random() < 0.6
        step = rng.choice([64, 128, 128, 256])
        hidden = _log(rng, 512, 8192, step)
        return dict(kind=kind, weight=weight, act=act, tiled=tiled, tokens=_log(rng, 1, 2048), hidden=hidden,
                    kv=max(128, hidden // rng.choice([1, 2, 4, 8]) // 128 * 128), inter=_log(rng, 1024, 16384, step))
    n_kv, ratio = rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 4])
    hidden = _log(rng, 1024, 4096, 128)
    model = dict(layers=rng.randint(1, 8), hidden=hidden, n_q=n_kv * ratio, n_kv=n_kv, inter=_log(rng, 1024, 14336, 128),
                 vocab=_log(rng, 2000, 152000), qk_norm=rng.random() < 0.5, tied=rng.random() < 0.3)
    pos = _log(rng, 16, 16000)
    if kind == "prompt":
        return dict(kind=kind, weight=weight, pos=0 if rng.random() < 0.6 else pos, tokens=_log(rng, 2, 2048), repack=rng.random() < 0.5, **model)
    return dict(kind=kind, weight=weight, pos=pos, steps=_log(rng, 1, 32) if kind == "decode" else rng.randint(1, 4), exact=rng.random() < 0.3, **model)


class _Memory:
    """Device memory of the library as a torch tensor; `owner` stays alive as long as a tensor on the memory does."""

    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (ptr, False), "version": 2}


def _bytes_at(ptr, n, owner):
    return torch.as_tensor(_Memory(ptr, (n,), "|u1", owner), device="cuda")


def _16bit_at(ptr, shape, owner, dtype=torch.bfloat16):
    return torch.as_tensor(_Memory(ptr, shape, "<i2", owner), device="cuda").view(dtype)


def _normal(gen, *shape, std=1.0, dtype=torch.bfloat16):
    return torch.randn(*shape, device="cuda", generator=gen).mul_(std).to(dtype)


def _host():
    host = pkg.host_api.host()
    host.init(0)
    return host


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = {"linears": _prepare_linears, "quantize": _prepare_quantize}.get(case["kind"], _prepare_model)(case, gen, seed)
    torch.cuda.synchronize()
    return state


def run(state):
    return {"linears": _run_linears, "quantize": _run_quantize, "decode": _run_decode, "sample": _run_sample, "prompt": _run_prompt}[state["kind"]](state)


# ---- the linears of one layer

def _layer_shapes(case):
    h, kv, inter = case["hidden"], case["kv"], case["inter"]
    return [("q", h, h), ("k", h, kv), ("v", h, kv), ("o", h, h), ("gate", h, inter), ("up", h, inter), ("down", inter, h)]       # (name, K, n_out)


def _prepare_linears(case, gen, seed):
    host = _host()
    w_type, scaled, spread = FORMATS[case["weight"]]
    act, act_dtype = (HALF, torch.float16) if case["act"] == "half" else (BF16, torch.bfloat16)
    T = case["tokens"]
    x = {}
    for K in {case["hidden"], case["inter"]}:
        x[K] = host.matrix(K, T, 1, 1, act)
        _16bit_at(x[K].data_ptr, (T, K), x[K], act_dtype).copy_(_normal(gen, T, K, dtype=act_dtype))
    calls, outputs = [], {}
    host.set_repack(case["tiled"])
    try:
        for name, K, n_out in _layer_shapes(case):
            values = _normal(gen, n_out, K, std=spread)
            W = host.matrix(K, n_out, 1, 1, BF16 if scaled else w_type)
            if scaled:
                _16bit_at(W.data_ptr, (n_out, K), W).copy_(values)
                torch.cuda.synchronize()
                W.quantize(w_type)
            else:
                _bytes_at(W.data_ptr, n_out * K, W).copy_(values.to(torch.float8_e5m2).view(torch.uint8).view(-1))
                torch.cuda.synchronize()
                if case["tiled"]:
                    W.prepare_tiled()
            Y = host.matrix(n_out, T, 1, 1, act)
            calls.append((W, x[K], Y))
            outputs[name] = _16bit_at(Y.data_ptr, (T, n_out), Y, act_dtype)
    finally:
        host.set_repack(True)
    return dict(kind="linears", calls=calls, outputs=outputs)


def _run_linears(state):
    for W, X, Y in state["calls"]:
        if pkg.host_api.mul_batched(W, X, Y, ta=1, tb=0) != 0:
            raise RuntimeError("linear failed")
    return state["outputs"]


# ---- quantizing a weight on the device and reading it back (the calls Matrix::quantizeWeights makes)

def _prepare_quantize(case, gen, seed):
    n = case["n_out"] * case["K"]
    codes = torch.empty((n + 1) // 2 if case["weight"] == "fp4" else n, dtype=torch.uint8, device="cuda")
    return dict(kind="quantize", type=FORMATS[case["weight"]][0], n=n, w=_normal(gen, n, std=FORMATS[case["weight"]][2]), f=torch.empty(n, device="cuda"), codes=codes,
                scales=torch.empty((n + 15) // 16, dtype=torch.uint8, device="cuda"), amax=torch.empty(1, device="cuda"),
                back=torch.empty(n, dtype=torch.bfloat16, device="cuda"))


def _run_quantize(s):
    lib, n, to = pkg.library(), s["n"], s["type"]
    w, f, codes, scales, amax, back = (s[k].data_ptr() for k in ("w", "f", "codes", "scales", "amax", "back"))
    rc = lib.convert(w, BF16, f, 0, n)
    if to == FP4:
        rc |= lib.float_to_fp4_blockscale(f, codes, scales, n, 16)
        rc |= lib.fp4_blockscale_to_bf16(codes, scales, back, n, 16)
        out = dict(codes=s["codes"], scales=s["scales"], back=s["back"])
    else:
        top = 448.0 if to == E4M3 else 57344.0
        rc |= lib.absmax(f, 0, n, amax)
        a = float(s["amax"])                              # the per-tensor scale is an argument of the conversions that follow
        rc |= lib.convert(f, 0, codes, to, n, top / a)
        rc |= lib.convert(codes, to, back, BF16, n, a / top)
        out = dict(codes=s["codes"], amax=s["amax"], back=s["back"])
    if rc != 0:
        raise RuntimeError("conversion failed")
    return out


# ---- whole models

def _prepare_model(case, gen, seed):
    host = _host()
    c = {k: case[k] for k in ("layers", "hidden", "n_q", "n_kv", "inter", "vocab")}
    w_type, scaled, spread = FORMATS[case["weight"]]
    t_kv = case["pos"] + case.get("steps", 0) + case.get("tokens", 0)
    model = pkg.host_api.DecodeModel(host, c["layers"], c["hidden"], c["n_q"], c["n_kv"], 128, c["inter"], c["vocab"], t_kv,
                                     theta=1e6 if case["qk_norm"] else 5e5)
    model.set_qk_norm(case["qk_norm"])
    model.set_tied_lm_head(case["tied"])
    model.set_exact_attention(case.get("exact", False))
    model.set_repack_linears(case.get("repack", False))

    def put(layer, name, values):                         # [n_out][K] BF16 values of a linear
        if scaled:
            torch.cuda.synchronize()
            model.quantize_linear(layer, name, values.data_ptr(), w_type)
        else:
            _bytes_at(model.tensor_ptr(layer, name), values.numel(), model).copy_(values.to(torch.float8_e5m2).view(torch.uint8).view(-1))
            if case.get("repack", False) or name == "lm_head":
                torch.cuda.synchronize()
                model.prepare_tiled(layer, name)

    def plain(layer, name, values):
        _16bit_at(model.tensor_ptr(layer, name), (values.numel(),), model).copy_(values.view(-1))

    h, inter, q_out, kv_out = c["hidden"], c["inter"], c["n_q"] * 128, c["n_kv"] * 128
    # projections of unit spread; gate and up smaller, so that down's output has the spread (2 layers)^-1/2 (silu(g) u is about
    # g u / 2 there)
    attn_gain = 1.0 / (spread * math.sqrt(h))
    ffn_gain = attn_gain * math.sqrt(2.0 / (spread * math.sqrt(inter)) / math.sqrt(2.0 * c["layers"]))
    gains = {"rms_attn": (h, attn_gain), "rms_ffn": (h, ffn_gain)}
    if case["qk_norm"]:
        gains.update(q_norm=(128, 1.0), k_norm=(128, 1.0))
    shapes = {"wq": (q_out, h), "wk": (kv_out, h), "wv": (kv_out, h), "wo": (h, q_out), "w_gate": (inter, h), "w_up": (inter, h), "w_down": (h, inter)}
    for layer in range(c["layers"]):
        for name, (n_out, K) in shapes.items():
            put(layer, name, _normal(gen, n_out, K, std=spread))
        for name, (n, gain) in gains.items():
            plain(layer, name, _normal(gen, n, std=0.1, dtype=torch.float32).add_(1.0).mul_(gain).to(torch.bfloat16))
        for is_v in (False, True):
            if case["pos"]:                               # the context so far
                _16bit_at(model.kv_ptr(layer, is_v), (c["n_kv"], t_kv, 128), model)[:, :case["pos"]].copy_(_normal(gen, c["n_kv"], case["pos"], 128))
    plain(0, "rms_final", _normal(gen, h, std=0.1, dtype=torch.float32).add_(1.0).to(torch.bfloat16))
    emb = _normal(gen, c["vocab"], h)
    plain(0, "emb", emb)
    if not case["tied"]:
        put(0, "lm_head", emb.roll(1, 0).mul_(spread))
    last = c["layers"] - 1
    caches = {("v" if is_v else "k"): _16bit_at(model.kv_ptr(last, is_v), (c["n_kv"], t_kv, 128), model) for is_v in (False, True)}
    rng = np.random.default_rng(seed)
    tokens = [int(t) for t in rng.integers(0, c["vocab"], case.get("tokens", 1 if case["kind"] == "decode" else case.get("steps", 1)))]
    torch.cuda.synchronize()
    return dict(kind=case["kind"], model=model, tokens=tokens, pos=case["pos"], steps=case.get("steps", 0), caches=caches)


def _logits(model):
    return torch.from_numpy(model.logits().view(np.int16)).view(torch.bfloat16)


def _run_decode(s):
    model = s["model"]
    model.reset(s["tokens"][0], s["pos"])
    model.run(s["steps"], True)
    return dict(token=model.token, logits=_logits(model), **s["caches"])


def _run_sample(s):
    model, logits = s["model"], []
    for i, token in enumerate(s["tokens"]):               # the tokens a sampler on the host came up with
        model.reset(token, s["pos"] + i)
        model.step()
        logits.append(_logits(model))
    return dict(logits=logits, **s["caches"])


def _run_prompt(s):
    token = s["model"].prefill(s["tokens"], s["pos"])
    return dict(token=token, logits=_logits(s["model"]), **s["caches"])


# ---- what one pass cannot do without

def _weight_bytes(weight, n):
    return n // 2 + n // 16 if weight == "fp4" else n


def work(case):
    if case["kind"] == "quantize":
        n = case["n_out"] * case["K"]
        return {"bytes": 4 * n + 2 * _weight_bytes(case["weight"], n), "flops": 0}
    if case["kind"] == "linears":
        T = case["tokens"]
        n = sum(K * n_out for _, K, n_out in _layer_shapes(case))
        x = 2 * T * (case["hidden"] + case["inter"])
        return {"bytes": _weight_bytes(case["weight"], n) + x + sum(2 * T * n_out for _, _, n_out in _layer_shapes(case)), "flops": 2.0 * T * n}
    h, q_out, kv_out = case["hidden"], case["n_q"] * 128, case["n_kv"] * 128
    per_layer = h * (q_out + 2 * kv_out) + q_out * h + 3 * h * case["inter"]
    layers = _weight_bytes(case["weight"], per_layer) * case["layers"]
    head = 2 * h * case["vocab"] if case["tied"] else _weight_bytes(case["weight"], h * case["vocab"])
    small = case["layers"] * 4 * h + 2 * h + 2 * case["vocab"]
    if case["kind"] == "prompt":
        T, P = case["tokens"], case["pos"]
        pairs = T * P + T * (T + 1) / 2.0
        return {"bytes": layers + head + small + 2 * T * h + case["layers"] * 4 * kv_out * (P + T),
                "flops": 2.0 * T * per_layer * case["layers"] + 4.0 * q_out * case["layers"] * pairs + 2.0 * h * case["vocab"]}
    S = case["steps"]
    seen = sum(case["pos"] + i + 1 for i in range(S))
    return {"bytes": S * (layers + head + small + 2 * h) + case["layers"] * 4 * kv_out * seen,
            "flops": S * 2.0 * (per_layer * case["layers"] + h * case["vocab"]) + 4.0 * q_out * case["layers"] * seen}


def tolerance(case):
    """Measured: the linears on tiled copies against the file layout (other kernels, other FP32 sums) differ by up to 4e-5, a
    BF16 step at the worst value; models between prompt and step-by-step (other sums, probabilities rounded or not) by up to
    1.6e-2, 0.08 at the worst value, and no tolerance goes beyond 3e-2."""
    if case["kind"] == "quantize":
        return "exact"
    if case["kind"] == "linears":
        return {"rel": 5e-4, "max": 0.02}
    return {"rel": 0.03, "max": 0.2}
