"""Workloads of a program that serves GPTQ models on one MI355X, for timing.

``listed()`` names the fixed ones, ``draw(rng)`` gives more from the same ranges.  ``prepare`` builds what such
a program holds before the call (weights, caches, inputs, from the seed alone), ``run`` is one pass through the
package's entry points and returns what the pass computes, ``work`` the bytes and operations the pass cannot do
without, ``tolerance`` how far two correct implementations of the same precision may be apart.
"""
import math

import torch

import minit_amd.functional as F
from minit_amd import lib, synthetic
from minit_amd.decode import LlamaDecoder, decode_attention
from minit_amd.hip import memory
from minit_amd.hip.tensor import HIPTensor
from minit_amd.quantize.linear import QLinear
from minit_amd.quantize.tensor import QuantizedTensor

HEAD = 128   # head size of every model shape here


def listed():
    return [
        # one projection for one new token: the smallest product a decode step launches (4096 wide, 4 bit)
        {"name": "linear_row1", "kind": "linear", "rows": 1, "k": 4096, "n": 4096, "bits": 4, "group": 128},
        # the four linears of a 70B layer for one new token: batch-1 decoding, bound by the weights' bytes
        {"name": "layer_70b_row1", "kind": "layer", "rows": 1, "hidden": 8192, "kv": 1024, "ffn": 28672, "bits": 4,
         "group": 128},
        # the same for an 8-bit act-order checkpoint with biases (hidden 5120, MLP 13696), a batch of 16 sequences
        {"name": "layer_8bit_rows16", "kind": "qlayer", "rows": 16, "hidden": 5120, "kv": 5120, "ffn": 13696, "bits": 8,
         "group": 128, "act_order": True},
        # and that checkpoint over a prompt of ordinary, ragged length
        {"name": "layer_8bit_prompt1000", "kind": "qlayer", "rows": 1000, "hidden": 5120, "kv": 5120, "ffn": 13696,
         "bits": 8, "group": 128, "act_order": True},
        # the gated MLP of a 7B model (4096 / 14336) for a large decode batch or a short prompt
        {"name": "mlp_4bit_rows128", "kind": "mlp", "rows": 128, "hidden": 4096, "ffn": 14336, "bits": 4, "group": 128},
        # the gated MLP of a 70B model over a 2048-token prompt: the largest pass
        {"name": "mlp_70b_prompt2048", "kind": "mlp", "rows": 2048, "hidden": 8192, "ffn": 28672, "bits": 4, "group": 128},
        # 8-bit weights and activations, a decode batch of 32
        {"name": "w8a8_rows32", "kind": "w8a8", "rows": 32, "n": 11008, "k": 4096},
        # 8-bit weights and activations over a prompt
        {"name": "w8a8_prompt2048", "kind": "w8a8", "rows": 2048, "n": 11008, "k": 4096},
        # attention of a prompt as the models compose it (rotation, q k^T, causal softmax, p v), 32 heads, ragged length
        {"name": "attention_prompt1500", "kind": "prompt_attention", "heads": 32, "seq": 1500},
        # attention of one new token for 32 sequences of different lengths over an 8192-entry cache
        {"name": "attention_decode32", "kind": "decode_attention", "rows": 32, "q_heads": 64, "kv_heads": 8, "context": 8192},
        # a decoder layer (4096 / 14336, 32 query and 8 KV heads) written operator by operator, two sequences: many small
        # launches behind host code
        {"name": "layer_by_operators", "kind": "operators", "rows": 2, "hidden": 4096, "q_heads": 32, "kv_heads": 8,
         "ffn": 14336, "bits": 4, "group": 128, "context": 1024},
        # the native decode loop: eight layers of the 70B shape and their share of vocabulary, eight sequences, four tokens
        {"name": "decode_loop_batch8", "kind": "decode", "rows": 8, "layers": 8, "hidden": 8192, "q_heads": 64,
         "kv_heads": 8, "ffn": 28672, "vocab": 32000, "bits": 4, "group": 128, "context": 2048, "tokens": 4},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _multiple(rng, low, high, of):
    return max(low, _log_int(rng, low, high) // of * of)


def draw(rng):
    kind = rng.choice(["linear", "linear", "layer", "qlayer", "qlayer", "mlp", "mlp", "w8a8", "w8a8", "prompt_attention",
                       "decode_attention", "operators", "decode"])
    bits, group = rng.choice([4, 4, 8]), rng.choice([128, 128, 64, 32])
    if kind == "linear":
        return {"kind": kind, "rows": _log_int(rng, 1, 2048), "k": _multiple(rng, 1024, 28672, 128),
                "n": _multiple(rng, 1024, 28672, 8), "bits": bits, "group": group}
    if kind == "layer":
        return {"kind": kind, "rows": _log_int(rng, 1, 64), "hidden": _multiple(rng, 2048, 8192, 1024), "kv": 1024,
                "ffn": _multiple(rng, 5632, 28672, 128), "bits": bits, "group": group}
    if kind == "qlayer":
        hidden = _multiple(rng, 2048, 8192, 128)
        return {"kind": kind, "rows": _log_int(rng, 1, 1500), "hidden": hidden, "kv": rng.choice([1024, hidden]),
                "ffn": _multiple(rng, 5632, 22016, 128), "bits": rng.choice([4, 8]), "group": group,
                "act_order": rng.random() < 0.5}
    if kind == "mlp":
        return {"kind": kind, "rows": _log_int(rng, 1, 2048), "hidden": _multiple(rng, 2048, 8192, 128),
                "ffn": _multiple(rng, 5632, 22016, 128), "bits": bits, "group": group}
    if kind == "w8a8":
        return {"kind": kind, "rows": _log_int(rng, 1, 4096), "n": _multiple(rng, 1024, 28672, 8),
                "k": _multiple(rng, 1024, 14336, 64)}
    if kind == "prompt_attention":
        return {"kind": kind, "heads": rng.choice([8, 16, 32, 40]), "seq": _log_int(rng, 32, 2300)}
    if kind == "decode_attention":
        kv = rng.choice([4, 8, 8, 16])
        return {"kind": kind, "rows": _log_int(rng, 1, 48), "q_heads": kv * rng.choice([1, 4, 8]), "kv_heads": kv,
                "context": _multiple(rng, 256, 16384, 64)}
    if kind == "operators":
        kv = rng.choice([8, 8, 16])
        heads = kv * rng.choice([2, 4])
        return {"kind": kind, "rows": _log_int(rng, 1, 16), "hidden": heads * HEAD, "q_heads": heads, "kv_heads": kv,
                "ffn": _multiple(rng, 5632, 22016, 128), "bits": bits, "group": group,
                "context": _multiple(rng, 256, 4096, 64)}
    heads = rng.choice([32, 40, 64])
    return {"kind": kind, "rows": _log_int(rng, 1, 32), "layers": rng.choice([2, 4, 6]), "hidden": heads * HEAD,
            "q_heads": heads, "kv_heads": heads // rng.choice([4, 8]),
            "ffn": _multiple(rng, 8192, 28672, 256), "vocab": 32000, "bits": bits, "group": 128,
            "context": _multiple(rng, 256, 4096, 64), "tokens": rng.choice([2, 4])}


# ---- inputs -------------------------------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, std=1.0, mean=0.0):
    return torch.empty(shape, dtype=torch.float16, device="cuda").normal_(mean, std, generator=g)


def _gptq(g, k, n, bits, group):
    """A checkpoint's tensors: sub-words over their whole range, zero points around its middle, steps that give
    weights of about 1 / sqrt(K), as a trained matrix has."""
    per = 32 // bits
    qweight = torch.randint(-2 ** 31, 2 ** 31, (k // per, n), dtype=torch.int32, device="cuda", generator=g)
    middle = (1 << (bits - 1)) - 1
    zeros = torch.randint(middle - 1, middle + 1, (k // group, n // per, per), dtype=torch.int32, device="cuda", generator=g)
    shift = torch.arange(per, dtype=torch.int32, device="cuda") * bits
    qzeros = (zeros << shift).sum(-1, dtype=torch.int64)
    qzeros = torch.where(qzeros >= 2 ** 31, qzeros - 2 ** 32, qzeros).to(torch.int32)
    step = 1.0 / (math.sqrt(k) * (1 << bits) / math.sqrt(12.0))
    scales = step * (0.7 + 0.6 * torch.rand((k // group, n), device="cuda", generator=g))
    return qweight, qzeros, scales.to(torch.float16)


def _quantized(tensors):
    qweight, qzeros, scales = (HIPTensor.from_torch(t) for t in tensors)
    return QuantizedTensor(qweight, None, qzeros, scales)


class _DeviceArray:
    """The package's device tensor as an array that torch can look at (no copy; keeps the memory alive)."""

    _TYPES = {"float16": "<f2", "float32": "<f4", "int32": "<i4"}

    def __init__(self, tensor):
        self._tensor = tensor
        self.__cuda_array_interface__ = {"shape": tuple(tensor._shape), "typestr": self._TYPES[tensor.dtype],
                                         "data": (tensor.data_ptr, False), "version": 2}


def _view(tensor):
    return torch.as_tensor(_DeviceArray(tensor), device="cuda")


def _workspace(nbytes):
    return torch.zeros(max(int(nbytes), 256), dtype=torch.uint8, device="cuda")


def _layer_shapes(case):
    h, ffn = case["hidden"], case["ffn"]
    return [(h, h + 2 * case["kv"]), (h, h), (h, 2 * ffn), (ffn, h)]


# ---- one linear, and the linears of a layer, over the C interface -------------------------------------------

class _Product:
    """One quantized product on buffers the caller owns."""

    def __init__(self, g, rows, k, n, bits, group):
        self.weight = _gptq(g, k, n, bits, group)
        self.x = _normal(g, (rows, k))
        self.out = torch.empty((rows, n), dtype=torch.float16, device="cuda")
        self.args = (rows, n, k, group, bits)
        self.workspace = _workspace(lib.call("mh_gptq_workspace_bytes", *self.args))

    def __call__(self):
        qweight, qzeros, scales = self.weight
        lib.call("mh_gptq_matmul", None, self.x.data_ptr(), qweight.data_ptr(), qzeros.data_ptr(), scales.data_ptr(), None,
                 self.out.data_ptr(), *self.args, self.workspace.data_ptr(), self.workspace.numel())
        return self.out


def _prepare_linear(case, g):
    return [_Product(g, case["rows"], case["k"], case["n"], case["bits"], case["group"])]


def _prepare_layer(case, g):
    return [_Product(g, case["rows"], k, n, case["bits"], case["group"]) for k, n in _layer_shapes(case)]


def _run_products(state):
    return [product() for product in state]


# ---- the linears of a layer as modules of a checkpoint (bias, act-order) ---------------------------------------

def _prepare_qlayer(case, g):
    modules = []
    for k, n in _layer_shapes(case):
        bias = HIPTensor.from_torch(_normal(g, (n,), 0.1))
        order = None
        if case["act_order"]:   # rows sorted by group at load time, the module gathers its input to match
            order = HIPTensor.from_torch(torch.randperm(k, device="cuda", generator=g).to(torch.int32))
        weight = _quantized(_gptq(g, k, n, case["bits"], case["group"]))
        modules.append((QLinear(weight, bias, order), HIPTensor.from_torch(_normal(g, (1, case["rows"], k)))))
    return modules


def _run_qlayer(state):
    return [_view(module(x)) for module, x in state]


# ---- gated MLP ---------------------------------------------------------------------------------------------------

def _prepare_mlp(case, g):
    rows, hidden, ffn, bits, group = (case[n] for n in ("rows", "hidden", "ffn", "bits", "group"))
    state = {"gate_up": _gptq(g, hidden, 2 * ffn, bits, group), "down": _gptq(g, ffn, hidden, bits, group),
             "x": _normal(g, (rows, hidden)), "out": torch.empty((rows, hidden), dtype=torch.float16, device="cuda"),
             "act": torch.empty((rows, ffn), dtype=torch.float16, device="cuda"),
             "up_args": (rows, 2 * ffn, hidden, group, bits), "down_args": (rows, hidden, ffn, group, bits)}
    nbytes = max(lib.call("mh_gptq_silu_pairs_workspace_bytes", *state["up_args"]),
                 lib.call("mh_gptq_workspace_bytes", *state["down_args"]))
    state["workspace"] = _workspace(nbytes)
    return state


def _run_mlp(s):
    ws = (s["workspace"].data_ptr(), s["workspace"].numel())
    lib.call("mh_gptq_matmul_silu_pairs", None, s["x"].data_ptr(), *(t.data_ptr() for t in s["gate_up"]),
             s["act"].data_ptr(), *s["up_args"], *ws)
    lib.call("mh_gptq_matmul", None, s["act"].data_ptr(), *(t.data_ptr() for t in s["down"]), None, s["out"].data_ptr(),
             *s["down_args"], *ws)
    return s["out"], s["act"]


# ---- 8-bit weights and activations ---------------------------------------------------------------------------------

def _prepare_w8a8(case, g):
    rows, n, k = case["rows"], case["n"], case["k"]

    def int8(shape):   # normal values quantised row by row, as a calibrated model's are
        return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, 32.0, generator=g).round_().clamp_(-127, 127).to(torch.int8)

    scale = 1.0 / (32.0 * 32.0 * math.sqrt(k))
    return {"a": int8((rows, k)), "w": int8((n, k)), "shape": (rows, n, k),
            "sa": 0.5 + torch.rand((rows,), device="cuda", generator=g),
            "sw": scale * (0.5 + torch.rand((n,), device="cuda", generator=g)),
            "out": torch.empty((rows, n), dtype=torch.float16, device="cuda")}


def _run_w8a8(s):
    lib.call("mh_i8_gemm", None, s["a"].data_ptr(), s["w"].data_ptr(), s["sa"].data_ptr(), s["sw"].data_ptr(),
             s["out"].data_ptr(), None, *s["shape"])
    return s["out"]


# ---- attention of a prompt, as the models compose it ------------------------------------------------------------------

def _prepare_prompt_attention(case, g):
    heads, seq = case["heads"], case["seq"]
    cos, sin = synthetic.rope_tables(HEAD, seq, 1e4)
    q, k = (HIPTensor.from_torch(_normal(g, (heads, seq, 1, HEAD))) for _ in range(2))
    return {"q": q, "k": k, "vt": HIPTensor.from_torch(_normal(g, (heads, HEAD, seq))), "heads": heads, "seq": seq,
            "cos": HIPTensor.from_numpy(cos), "sin": HIPTensor.from_numpy(sin)}


def _run_prompt_attention(s):
    heads, seq = s["heads"], s["seq"]
    q = F.rope(s["q"], s["cos"], s["sin"]).reshape((heads, seq, HEAD))
    k = F.rope(s["k"], s["cos"], s["sin"]).reshape((heads, seq, HEAD))
    scores = F.batch_matrix_multiply(q, k)
    probs = HIPTensor.allocate((heads, seq, seq), "float16")
    lib.call("mh_softmax_causal", None, scores.data_ptr, probs.data_ptr, heads, seq, seq, 0, 1.0 / math.sqrt(HEAD),
             lib.DTYPE_CODES["float16"])
    return _view(F.batch_matrix_multiply(probs, s["vt"]))


# ---- attention of one new token per sequence ------------------------------------------------------------------------------

def _caches(g, rows, kv_heads, context):
    k = HIPTensor.from_torch(_normal(g, (rows, kv_heads, context, HEAD)))
    vt = HIPTensor.from_torch(_normal(g, (rows, kv_heads, context // 64, HEAD, 64)))
    # sequences of one batch are at different places: from an eighth of the cache to all of it
    positions = torch.randint(context // 8, context, (rows,), dtype=torch.int32, device="cuda", generator=g)
    return k, vt, positions


def _lengths(case):
    """Visible cache entries over the batch, as expected from the distribution of the positions."""
    return case["rows"] * case["context"] * 9 // 16


def _prepare_decode_attention(case, g):
    k, vt, positions = _caches(g, case["rows"], case["kv_heads"], case["context"])
    return {"q": HIPTensor.from_torch(_normal(g, (case["rows"], case["q_heads"], HEAD))), "k": k, "vt": vt,
            "positions": HIPTensor.from_torch(positions), "context": case["context"]}


def _run_decode_attention(s):
    return _view(decode_attention(s["q"], s["k"], s["vt"], s["positions"], s["context"]))


# ---- a decoder layer operator by operator -------------------------------------------------------------------------------------

def _operator_shapes(case):
    h, q, kv, ffn = case["hidden"], case["q_heads"] * HEAD, case["kv_heads"] * HEAD, case["ffn"]
    return {"q": (h, q), "k": (h, kv), "v": (h, kv), "o": (q, h), "gate": (h, ffn), "up": (h, ffn), "down": (ffn, h)}


def _prepare_operators(case, g):
    rows, hidden, context = case["rows"], case["hidden"], case["context"]
    state = {name: _quantized(_gptq(g, k, n, case["bits"], case["group"])) for name, (k, n) in _operator_shapes(case).items()}
    cache_k, cache_v, positions = _caches(g, rows, case["kv_heads"], context)
    cos, sin = synthetic.rope_tables(HEAD, context, 1e4)
    state.update(x=HIPTensor.from_torch(_normal(g, (rows, 1, hidden))), cache_k=cache_k, cache_v=cache_v,
                 norm1=HIPTensor.from_torch(_normal(g, (hidden,), 0.1, 1.0)),
                 norm2=HIPTensor.from_torch(_normal(g, (hidden,), 0.1, 1.0)),
                 positions=HIPTensor.from_torch(positions), positions2=HIPTensor.from_torch(positions.reshape(rows, 1)),
                 cos=HIPTensor.from_numpy(cos), sin=HIPTensor.from_numpy(sin), rows=rows, context=context,
                 heads=(case["q_heads"], case["kv_heads"]))
    return state


def _run_operators(s):
    rows, (qh, kvh) = s["rows"], s["heads"]
    x = s["x"]
    y = F.rms_norm(x, s["norm1"], 2, 1e-5)
    q = F.rope(F.matrix_multiply(y, s["q"]).reshape((rows, 1, qh, HEAD)), s["cos"], s["sin"], s["positions2"])
    k = F.rope(F.matrix_multiply(y, s["k"]).reshape((rows, 1, kvh, HEAD)), s["cos"], s["sin"], s["positions2"])
    v = F.matrix_multiply(y, s["v"])
    a = decode_attention(q.reshape((rows, qh, HEAD)), s["cache_k"], s["cache_v"], s["positions"], s["context"])
    x = x + F.matrix_multiply(a.reshape((rows, 1, qh * HEAD)), s["o"])
    y = F.rms_norm(x, s["norm2"], 2, 1e-5)
    gate = F.matrix_multiply(y, s["gate"])
    x = x + F.matrix_multiply(gate * F.sigmoid(gate) * F.matrix_multiply(y, s["up"]), s["down"])
    return _view(x), _view(k), _view(v)


# ---- the native decode loop --------------------------------------------------------------------------------------------------

def _prepare_decode(case, seed):
    config = dict(n_layers=case["layers"], hidden=case["hidden"], n_q_heads=case["q_heads"], n_kv_heads=case["kv_heads"],
                  head_dim=HEAD, ffn=case["ffn"], vocab=case["vocab"], group_size=case["group"], bits=case["bits"],
                  rope_theta=5e5, rms_eps=1e-5)
    decoder = LlamaDecoder(config, case["rows"], case["context"] + case["tokens"])
    # steps and zero points that keep the activations finite, as the decode benchmark draws them
    fine = {4: dict(scale_std=0.02 / 16, zero_range=(6, 7)), 8: dict(scale_std=0.02 / 256, zero_range=(126, 127))}[case["bits"]]
    decoder.load_synthetic(seed=seed % 100000, prefill=case["context"], **fine)
    # rows of the head follow the embeddings' (token i is followed by i + 1): the sampled token has a clear margin, as a
    # trained model's mostly has, and with it the sequence does not hang on the last bit of a logit
    memory.synchronize()
    embed = torch.empty((case["vocab"], case["hidden"]), dtype=torch.float16, device="cuda")
    embed.normal_(0.0, 1.0, generator=_generator(seed))
    _view(decoder.embed).copy_(embed)
    _view(decoder.lm_head).copy_(torch.roll(embed, 1, 0) * 0.02)
    memory.synchronize()
    g = torch.Generator()
    g.manual_seed(int(seed))
    tokens = torch.randint(0, case["vocab"], (case["rows"],), generator=g, dtype=torch.int32).numpy()
    positions = torch.randint(case["context"] // 2, case["context"], (case["rows"],), generator=g, dtype=torch.int32).numpy()
    return {"decoder": decoder, "first": tokens, "positions": positions, "tokens": case["tokens"]}


def _run_decode(s):
    tokens, logits = s["decoder"].decode(s["first"], s["positions"], s["tokens"], want_logits=True)
    return tokens, logits


# ---- the table of kinds --------------------------------------------------------------------------------------------------------

_PREPARE = {"linear": _prepare_linear, "layer": _prepare_layer, "qlayer": _prepare_qlayer, "mlp": _prepare_mlp,
            "w8a8": _prepare_w8a8, "prompt_attention": _prepare_prompt_attention,
            "decode_attention": _prepare_decode_attention, "operators": _prepare_operators}
_RUN = {"linear": _run_products, "layer": _run_products, "qlayer": _run_qlayer, "mlp": _run_mlp, "w8a8": _run_w8a8,
        "prompt_attention": _run_prompt_attention, "decode_attention": _run_decode_attention,
        "operators": _run_operators, "decode": _run_decode}


def prepare(case, seed):
    if case["kind"] == "decode":
        state = _prepare_decode(case, seed)
    else:
        state = _PREPARE[case["kind"]](case, _generator(seed))
    return case["kind"], state


def run(state):
    kind, held = state
    return _RUN[kind](held)


def _product_bytes(rows, k, n, bits, group):
    weight = k * n * bits // 8 + (k // group) * n * 2 + (k // group) * (n * bits // 32) * 4
    return weight + rows * (k + n) * 2


def work(case):
    kind = case["kind"]
    if kind == "linear":
        shapes = [(case["k"], case["n"])]
    elif kind in ("layer", "qlayer"):
        shapes = _layer_shapes(case)
    elif kind == "mlp":
        shapes = [(case["hidden"], 2 * case["ffn"]), (case["ffn"], case["hidden"])]
    elif kind == "operators":
        shapes = list(_operator_shapes(case).values())
    elif kind == "decode":
        h, q, kv = case["hidden"], case["q_heads"] * HEAD, case["kv_heads"] * HEAD
        shapes = [(h, q + 2 * kv), (q, h), (h, 2 * case["ffn"]), (case["ffn"], h)]
    if kind == "w8a8":
        rows, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": rows * k + n * k + rows * n * 2 + (rows + n) * 4, "flops": 2.0 * rows * n * k}
    if kind == "prompt_attention":
        heads, seq = case["heads"], case["seq"]
        # the composition's entry points hand the scores and the probabilities to their caller
        return {"bytes": heads * seq * (6 * HEAD + 4 * seq) * 2, "flops": 4.0 * heads * seq * seq * HEAD}
    if kind == "decode_attention":
        return {"bytes": _lengths(case) * case["kv_heads"] * HEAD * 4 + 4 * case["rows"] * case["q_heads"] * HEAD,
                "flops": 4.0 * _lengths(case) * case["q_heads"] * HEAD}
    rows = case["rows"]
    nbytes = sum(_product_bytes(rows, k, n, case["bits"], case["group"]) for k, n in shapes)
    flops = sum(2.0 * rows * k * n for k, n in shapes)
    if kind == "mlp":   # the gate and up halves meet in the first product, its output is half as wide
        nbytes -= rows * case["ffn"] * 2
    if kind == "operators":
        nbytes += _lengths(case) * case["kv_heads"] * HEAD * 4
        flops += 4.0 * _lengths(case) * case["q_heads"] * HEAD
    if kind == "decode":
        visible = rows * case["context"] * 3 // 4
        nbytes = case["layers"] * (nbytes + visible * case["kv_heads"] * HEAD * 4) + case["vocab"] * case["hidden"] * 2
        flops = case["layers"] * (flops + 4.0 * visible * case["q_heads"] * HEAD) + 2.0 * rows * case["vocab"] * case["hidden"]
        nbytes, flops = nbytes * case["tokens"], flops * case["tokens"]
    return {"bytes": nbytes, "flops": flops}


# Largest relative error (2-norm) seen against the path in 64 bits, or, for the decode loop, between the batch and its
# rows decoded alone (other kernels, other order of the sums): a product 2.1e-4 (the rounding of its fp16 result), the
# MLP with its fp16 intermediate 4.4e-4, decode attention 2.7e-4, prompt attention with fp16 scores and probabilities
# 6.3e-4, four tokens through eight layers 6.8e-4; the operators of a layer end in such an MLP.  About four times that
# is stated.
_TOLERANCE = {"linear": 1e-3, "layer": 1e-3, "qlayer": 1e-3, "mlp": 1.8e-3, "prompt_attention": 2.5e-3,
              "decode_attention": 1e-3, "operators": 1.8e-3, "decode": 3e-3}


def tolerance(case):
    if case["kind"] == "w8a8":
        return "exact"   # integer sums and a fixed order of the three roundings behind them
    return {"rel": _TOLERANCE[case["kind"]]}
