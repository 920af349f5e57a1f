"""Performance cases of this package: what a user of it has it do, through its public entry points.

Kinds of work
  int4    one weight-only int4 linear layer on device tensors (PackedInt4Weight.matmul): the MatMulNBits node of an
          exported LLM, from one decode row to a long prompt
  int8    one int8 linear layer on device tensors (PackedI8B.matmul / matmul_requant): MatMulInteger and QLinearMatMul
  dql     DynamicQuantizeLinear -> MatMulInteger on f32 carriers, the pair a dynamically quantised ONNX graph runs
  between the operators between the MatMuls of an LLM graph on f32 tensors: RMSNorm and GroupQueryAttention
  decode  greedy decoding of a resident decoder: reset, n steps, tokens and last logits back
  prefill the prompt phase of the same decoder, first token and logits back
  generate the sampling loop with its default settings (temperature 1, top-k 50, top-p 0.9)

Decoders carry random layers.  Embedding and LM head are made so that every token predicts one successor by a clear
margin, as a trained model's next token mostly does: picks then do not hang on the last bit of two equal logits, while
most of every other logit comes from the layers.
"""
import math

import numpy as np
import torch

from yscv_amd import kernels as K
from yscv_amd import onnx_ops as O
from yscv_amd.decoder import Decoder

TORCH_DTYPE = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
ITEM = {"f32": 4, "f16": 2, "bf16": 2}

# the two decoder shapes of bench.py: the 7B-shape model of the headline, and the small model the reference publishes
# its own figures on (head width 64, eight query heads per kv head, vocabulary 151936)
MODELS = {
    "7b": dict(n_layers=32, d_model=4096, n_heads=32, n_kv_heads=8, head_dim=128, d_ff=14336, vocab=32000, group_size=32,
               rope_theta=10000.0, rms_eps=1e-5),
    "24l": dict(n_layers=24, d_model=1024, n_heads=16, n_kv_heads=2, head_dim=64, d_ff=2816, vocab=151936, group_size=32,
                rope_theta=1000000.0, rms_eps=1e-6),
}


def int4(name, m, n, k, group, act, scales, zero_points=False):
    return {"name": name, "kind": "int4", "m": m, "n": n, "k": k, "group": group, "act": act, "scales": scales,
            "zero_points": zero_points}


def listed():
    return [
        # one projection of a 7B layer for one token in f32, as a runner with f32 tensors calls it: the smallest call,
        # launch and host time count
        int4("int4_gemv_f32", 1, 4096, 4096, 32, "f32", "f32"),
        # LM head of a 128k vocabulary for a batch of 16 sequences: the weight stream
        int4("int4_lm_head_m16_bf16", 16, 128256, 4096, 32, "bf16", "f16"),
        # a short prompt through a layer whose sizes fit no tile: odd rows and columns, k a multiple of the group only
        int4("int4_ragged_m77_f16", 77, 3001, 2880, 64, "f16", "f16"),
        # gate or up projection of a 2048-token prompt, asymmetric weights of 128-groups: matrix cores
        int4("int4_prefill_2048_bf16", 2048, 14336, 4096, 128, "bf16", "f16", True),
        # MatMulInteger of a 512-row activation with a uint8 zero point
        {"name": "int8_m512_i32", "kind": "int8", "m": 512, "n": 4096, "k": 4096, "requant": False},
        # QLinearMatMul of a 197-token image encoder (odd rows): GEMM with the requantising epilogue
        {"name": "int8_requant_m197", "kind": "int8", "m": 197, "n": 3072, "k": 768, "requant": True},
        # a dynamically quantised encoder layer, 128 tokens
        {"name": "dql_m128", "kind": "dql", "m": 128, "n": 4096, "k": 1024},
        # norm and attention of a 512-token prompt between the MatMuls, 7B head layout
        {"name": "norm_gqa_512", "kind": "between", "batch": 1, "sq": 512, "sk": 512, "heads": 32, "kv_heads": 8, "head_dim": 128},
        # chat decoding for one user: 16 greedy tokens at 2048 cached positions
        {"name": "decode_7b_b1", "kind": "decode", "model": "7b", "batch": 1, "ctx": 2048, "steps": 16, "kv": "f16"},
        # serving a full batch of 16 sequences
        {"name": "decode_7b_b16", "kind": "decode", "model": "7b", "batch": 16, "ctx": 2048, "steps": 8, "kv": "f16"},
        # a long prompt through the whole model: the largest call
        {"name": "prefill_7b_2048", "kind": "prefill", "model": "7b", "tokens": 2048, "kv": "f16"},
        # llm-bench's own run: a 43-token prompt, 16 sampled tokens
        {"name": "generate_24l_p43", "kind": "generate", "model": "24l", "tokens": 43, "steps": 16, "kv": "f16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["int4", "int4", "int4", "int8", "int8", "dql", "between", "decode", "prefill", "generate"])
    if kind == "int4":
        group = rng.choice([32, 64, 128])
        scales = rng.choice(["f16", "f16", "f32"])
        act = "f32" if scales == "f32" else rng.choice(["f32", "f16", "bf16"])
        m = _log_int(rng, 1, 2048) if scales == "f16" else _log_int(rng, 1, 128)
        k = group * max(1, _log_int(rng, 512, 14336) // group)
        n = _log_int(rng, 256, min(128256, 4096 * 128256 // k, 2048 * 4096 * 14336 // (m * k)))
        return {"kind": "int4", "m": m, "n": n, "k": k, "group": group, "act": act, "scales": scales,
                "zero_points": scales == "f16" and rng.random() < 0.3}
    if kind == "int8":
        m, k, n = _log_int(rng, 1, 2048), _log_int(rng, 256, 8192), _log_int(rng, 256, 8192)
        if rng.random() < 0.75:  # layer widths are mostly multiples of 64
            k, n = max(64, k // 64 * 64), max(64, n // 64 * 64)
        return {"kind": "int8", "m": m, "n": n, "k": k, "requant": rng.random() < 0.5}
    if kind == "dql":
        return {"kind": "dql", "m": _log_int(rng, 1, 1024), "n": 64 * _log_int(rng, 4, 128), "k": 64 * _log_int(rng, 4, 128)}
    if kind == "between":
        kv_heads = rng.choice([2, 8])
        sk = _log_int(rng, 32, 2048)
        sq = 1 if rng.random() < 0.25 else max(1, min(sk, _log_int(rng, 16, 1024)))
        return {"kind": "between", "batch": rng.choice([1, 1, 2, 4]), "sq": sq, "sk": sk, "heads": kv_heads * rng.choice([1, 4]),
                "kv_heads": kv_heads, "head_dim": rng.choice([64, 128])}
    model = rng.choice(["7b", "24l"])
    if kind == "decode":
        kv = "i8" if model == "7b" and rng.random() < 0.25 else "f16"
        return {"kind": "decode", "model": model, "batch": rng.choice([1, 1, 2, 3, 4, 8, 11, 16]), "ctx": _log_int(rng, 64, 2048),
                "steps": rng.randint(4, 16) if model == "24l" else rng.randint(4, 8), "kv": kv}
    if kind == "prefill":
        return {"kind": "prefill", "model": model, "tokens": _log_int(rng, 9, 2048), "kv": "f16"}
    return {"kind": "generate", "model": model, "tokens": _log_int(rng, 9, 512), "steps": rng.randint(6, 16), "kv": "f16"}


# ---- inputs ------------------------------------------------------------------------------------------------------------
def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _int4_weight(g, n, k, group, scales, zero_points):
    b = torch.randint(0, 256, (n * k // 2,), generator=g, device="cuda", dtype=torch.uint8)
    sc = torch.rand(n * (k // group), generator=g, device="cuda") * 0.015 + 0.005
    zp = None
    if zero_points:
        zp = torch.randint(6, 11, (2, n * ((k // group + 1) // 2)), generator=g, device="cuda", dtype=torch.uint8)
        zp = (zp[0] | (zp[1] << 4)).cpu().numpy()
    sc = sc.to(TORCH_DTYPE[scales]).cpu().numpy()
    return K.PackedInt4Weight(b.cpu().numpy(), sc, group, n, k, zero_points=zp, nibble_format=K.NIBBLE_UNSIGNED)


def _decoder(case, seed):
    cfg = dict(MODELS[case["model"]])
    last = case.get("ctx", case.get("tokens", 0)) + case.get("steps", 1)
    cfg.update(max_batch=case.get("batch", 1), max_ctx=(last + 127) // 128 * 128, max_steps=64)
    layers, d, vocab, group = cfg["n_layers"], cfg["d_model"], cfg["vocab"], cfg["group_size"]
    dec = Decoder(kv_dtype=case["kv"], **cfg)
    dec.init_random(seed=seed, nibbles=(1, 15))
    g = _rng(seed)
    emb = torch.randn(vocab, d, generator=g, device="cuda")
    # row of the successor of token t: noise plus t's own embedding row
    succ = torch.randperm(vocab, generator=g, device="cuda")
    q = torch.empty(vocab, d, device="cuda", dtype=torch.uint8)
    q[succ] = (torch.randn(vocab, d, generator=g, device="cuda") * 2.0 + emb * 2.5 + 8.0).round_().clamp_(1, 15).to(torch.uint8)
    packed = (q[:, 0::2] | (q[:, 1::2] << 4)).cpu().numpy()
    scales = (torch.rand(vocab, d // group, generator=g, device="cuda") * 0.005 + 0.01).half().cpu().numpy()
    dec.set_linear(0, "lm_head", packed.reshape(-1), scales.reshape(-1), vocab, d)
    # the layers add about 0.1 sqrt(d_ff) per layer to the residual stream; the embedding is a third of their sum
    dec.set_embedding((emb * (math.sqrt(layers * cfg["d_ff"]) * 0.1)).half().cpu().numpy())
    gain = np.full(d, 0.25, np.float32)  # moderate attention scores and gate values
    for layer in range(layers):
        dec.set_norm(layer, "attn", gain)
        dec.set_norm(layer, "ffn", gain)
    dec.finalize()
    return dec, np.random.default_rng(seed)


def prepare(case, seed):
    kind = case["kind"]
    g = _rng(seed)
    if kind == "int4":
        w = _int4_weight(g, case["n"], case["k"], case["group"], case["scales"], case["zero_points"])
        x = torch.randn(case["m"], case["k"], generator=g, device="cuda").to(TORCH_DTYPE[case["act"]])
        return {"kind": kind, "w": w, "x": x}
    if kind == "int8":
        m, n, k = case["m"], case["n"], case["k"]
        b = torch.randint(-127, 128, (k, n), generator=g, device="cuda", dtype=torch.int8)
        state = {"kind": kind, "b": K.pack_i8_b_for_matmul(b.cpu().numpy(), k, n), "requant": case["requant"],
                 "a": torch.randint(0, 256, (m, k), generator=g, device="cuda", dtype=torch.uint8)}
        if case["requant"]:  # per-column scales that spread the products over the byte range
            state["composite"] = (torch.rand(n, generator=g, device="cuda") * 0.5 + 0.75) * (50.0 / (74.0 * 73.6 * math.sqrt(k)))
        return state
    if kind == "dql":
        m, n, k = case["m"], case["n"], case["k"]
        b = torch.randint(-127, 128, (k, n), generator=g, device="cuda", dtype=torch.int8)
        return {"kind": kind, "b": O.PrepackedI8B(b.float()), "x": torch.randn(m, k, generator=g, device="cuda")}
    if kind == "between":
        b, d = case["batch"], case["head_dim"]
        width = case["heads"] * d
        return {"kind": kind, "heads": case["heads"], "kv_heads": case["kv_heads"],
                "h": torch.randn(b, case["sq"], width, generator=g, device="cuda") * 3.0,
                "gamma": torch.rand(width, generator=g, device="cuda") + 0.5,
                "q": torch.randn(b, case["sq"], width, generator=g, device="cuda"),
                "k": torch.randn(b, case["sk"], case["kv_heads"] * d, generator=g, device="cuda"),
                "v": torch.randn(b, case["sk"], case["kv_heads"] * d, generator=g, device="cuda")}
    dec, rng = _decoder(case, seed)
    vocab = MODELS[case["model"]]["vocab"]
    if kind == "decode":
        dec.fill_kv_random(seed=seed)
        return {"kind": kind, "dec": dec, "ctx": case["ctx"], "steps": case["steps"],
                "tokens": rng.integers(0, vocab, case["batch"]).astype(np.int32)}
    tokens = rng.integers(0, vocab, case["tokens"]).astype(np.int32)
    dec.reset(tokens[:1], 0)  # one sequence: logits() returns as many rows as reset() was given
    return {"kind": kind, "dec": dec, "steps": case.get("steps", 0), "tokens": tokens}


# ---- one pass ----------------------------------------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "int4":
        return state["w"].matmul(state["x"])
    if kind == "int8":
        if state["requant"]:
            return state["b"].matmul_requant(state["a"], 128, state["composite"], 128.0, K.ROUND_HALF_AWAY, 0, 255)
        return state["b"].matmul(state["a"], a_zp=128)
    if kind == "dql":
        return O.exec_dql_matmul_integer(state["x"], state["b"])
    if kind == "between":
        return (O.rms_norm(state["h"], state["gamma"], 1e-5),
                O.exec_grouped_query_attention(state["q"], state["k"], state["v"], state["heads"], state["kv_heads"]))
    dec = state["dec"]
    if kind == "decode":
        dec.reset(state["tokens"], state["ctx"])
        dec.run(state["steps"], auto=True)
        return dec.tokens(0, state["steps"]), dec.logits()
    if kind == "prefill":
        dec.prefill(state["tokens"])
        return dec.tokens(0, 1), dec.logits()
    tokens = dec.generate(state["tokens"], max_tokens=state["steps"])
    return tokens.astype(np.int64), dec.logits()


# ---- what a pass cannot do without -------------------------------------------------------------------------------------
def _model_params(model):
    """(weights of all layers, weights of the LM head, bytes per weight with its share of the fp16 scales)"""
    c = MODELS[model]
    d, hd, ff = c["d_model"], c["head_dim"], c["d_ff"]
    hq, hkv = c["n_heads"] * hd, c["n_kv_heads"] * hd
    return c["n_layers"] * ((hq + 2 * hkv) * d + d * hq + 3 * d * ff), c["vocab"] * d, 0.5 + 2.0 / c["group_size"]


def _decode_work(case, batch, ctx, steps):
    c = MODELS[case["model"]]
    layer_w, head_w, per = _model_params(case["model"])
    kv_row = 2 * c["n_kv_heads"] * c["head_dim"] * (2 if case["kv"] == "f16" else 1)
    positions = steps * ctx + steps * (steps + 1) // 2
    return {"bytes": steps * (layer_w + head_w) * per + batch * c["n_layers"] * positions * kv_row + batch * c["vocab"] * 4,
            "flops": 2.0 * batch * steps * (layer_w + head_w) + 4.0 * batch * c["n_layers"] * c["n_heads"] * c["head_dim"] * positions}


def _prefill_work(case):
    c = MODELS[case["model"]]
    layer_w, head_w, per = _model_params(case["model"])
    t = case["tokens"]
    return {"bytes": (layer_w + head_w) * per + t * c["n_layers"] * 2 * c["n_kv_heads"] * c["head_dim"] * 2 + c["vocab"] * 4,
            "flops": 2.0 * (t * layer_w + head_w) + 2.0 * c["n_layers"] * c["n_heads"] * c["head_dim"] * t * (t + 1)}


def work(case):
    kind = case["kind"]
    if kind == "int4":
        m, n, k, groups = case["m"], case["n"], case["k"], case["k"] // case["group"]
        return {"bytes": n * k // 2 + n * groups * ITEM[case["scales"]] + (n * ((groups + 1) // 2) if case["zero_points"] else 0) +
                m * (k + n) * ITEM[case["act"]], "flops": 2.0 * m * n * k}
    if kind == "int8":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": m * k + n * k + m * n * (1 if case["requant"] else 4) + (4 * n if case["requant"] else 0), "flops": 2.0 * m * n * k}
    if kind == "dql":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * m * k + n * k + 4 * m * n, "flops": 2.0 * m * n * k}
    if kind == "between":
        b, sq, sk, d = case["batch"], case["sq"], case["sk"], case["head_dim"]
        width = case["heads"] * d
        return {"bytes": 4 * (b * sq * width * 4 + 2 * b * sk * case["kv_heads"] * d + width), "flops": 4.0 * b * sq * sk * width + 4.0 * b * sq * width}
    if kind == "decode":
        return _decode_work(case, case["batch"], case["ctx"], case["steps"])
    if kind == "prefill":
        return _prefill_work(case)
    a, b = _prefill_work(case), _decode_work(case, 1, case["tokens"], case["steps"] - 1)
    return {"bytes": a["bytes"] + b["bytes"], "flops": a["flops"] + b["flops"]}


def tolerance(case):
    kind = case["kind"]
    if kind in ("int8", "dql"):
        return "exact"  # whole numbers, in f32 carriers for dql
    if kind == "int4":
        if case["act"] == "bf16":
            return {"rel": 5e-3}
        # f32 activations against f32 scales, and f32 rows up to the batch of a decode step, are computed to f32 precision;
        # else activations or scaled weights are fp16 operands
        exact = case["act"] == "f32" and (case["scales"] == "f32" or case["m"] <= 16)
        return {"rel": 1e-5} if exact else {"rel": 1e-3}
    if kind == "between":
        return {"rel": 1e-3}  # softmax weights and values are fp16 operands
    return {"rel": 1e-2}  # fp16 activations through every layer; tokens are the same
