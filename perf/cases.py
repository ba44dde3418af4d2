"""The work this library is used for, as cases that can be timed.

Every case goes through the public entry points of the package (the functions of `wechat-tfcc_amd/__init__.py` on
device tensors, `runtime_api.Model` on host arrays).  A case is a dict; its "kind" says which path it stands for:

  dense    a fully connected layer in float32: blas_matmul(x, w[, bias]).  One token or one user's features up to the
           flattened tokens of a large batch; layer widths that are round (hidden sizes) and ones that are not
           (vocabularies, label sets, concatenated features).
  batched  products with a leading batch in float32, as attention written out in separate operations makes them
           (scores, context, a weight shared by the whole batch): blas_matmul on tensors of rank three and four.
  qmatmul  a quantized layer inside a quantized network: uint8 activations, int8 weights, int32 sums, requantized to
           uint8 in the same call; row sums come with the activations, column sums were made once with the weights.
  qlayer   a quantized layer between float32 neighbours, the way a dynamically quantized model runs it: the activations
           are quantized with their own range, their row sums taken, the product is formed and then either dequantized
           to float32 or, for a quantized successor, requantized.
  decode   one decoding step of up to eight sequences over int8 weights with a scale per output channel, the weights
           row-major or packed once.
  encoder  one transformer encoder layer of a converted model, served through Model.run: host arrays in, host arrays
           out, with and without an attention mask.  prepare() loads the model and runs it once, as a server does
           before it takes requests.
  bilstm   a bidirectional LSTM of a converted model (tagging, speech), served the same way.
"""
import importlib
import math

import numpy as np
import torch

tfcc = importlib.import_module("wechat-tfcc_amd")
modelfile = importlib.import_module("wechat-tfcc_amd.modelfile")
runtime_api = importlib.import_module("wechat-tfcc_amd.runtime_api")


def listed():
    return [
        # one request, one token: the smallest call there is, latency only
        {"name": "dense_1x768x768", "kind": "dense", "m": 1, "k": 768, "n": 768, "bias": True},
        # one sentence through the widening layer of a base-sized model
        {"name": "dense_128x768x3072", "kind": "dense", "m": 128, "k": 768, "n": 3072, "bias": True},
        # nothing is a multiple of anything: padded-out features into a label set
        {"name": "dense_ragged_333x1003x517", "kind": "dense", "m": 333, "k": 1003, "n": 517, "bias": True},
        # the largest float32 product of the benchmark
        {"name": "dense_4096x4096x4096", "kind": "dense", "m": 4096, "k": 4096, "n": 4096, "bias": False},
        # attention scores of a batch of sixteen sentences, twelve heads of 64
        {"name": "batched_192x128x64x128", "kind": "batched", "batch": 192, "m": 128, "k": 64, "n": 128, "shared": False},
        # the quantized product the benchmark is quoted on
        {"name": "qmatmul_4096x4096x4096", "kind": "qmatmul", "m": 4096, "k": 4096, "n": 4096, "acc": False, "exact": False},
        # a dynamically quantized widening layer on eight sentences
        {"name": "qlayer_1024x768x3072", "kind": "qlayer", "m": 1024, "k": 768, "n": 3072, "requant": False},
        # the same on a ragged batch and odd widths
        {"name": "qlayer_ragged_77x1001x1237", "kind": "qlayer", "m": 77, "k": 1001, "n": 1237, "requant": False},
        # one decoding step of four sequences
        {"name": "decode_m4_4096x11008", "kind": "decode", "m": 4, "k": 4096, "n": 11008, "packed": False, "exact": False,
         "acc": False},
        # eight sentences of 128 tokens through one layer of a base-sized model
        {"name": "encoder_b8_s128_h768", "kind": "encoder", "batch": 8, "seq": 128, "hidden": 768, "mask": False},
        # one short query, padded: what an online service sees most
        {"name": "encoder_b1_s29_h768_mask", "kind": "encoder", "batch": 1, "seq": 29, "hidden": 768, "mask": True},
        # four utterances of 64 steps, tagged together
        {"name": "bilstm_s64_b4_l512_h512", "kind": "bilstm", "seq": 64, "batch": 4, "length": 512, "hidden": 512},
    ]


# ---- drawn cases -------------------------------------------------------------------------------------------------
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size between lo and hi, even over its logarithm: half of them round, the others as they fall."""
    v = max(lo, min(hi, _log(rng, lo, hi)))
    step = rng.choice([1, 1, 8, 64])
    return max(lo, v // step * step)


def draw(rng):
    kind = rng.choice(["dense", "dense", "dense", "batched", "qmatmul", "qlayer", "qlayer", "decode", "encoder", "encoder",
                       "bilstm"])
    if kind == "dense":
        while True:
            c = {"kind": kind, "m": _size(rng, 1, 4096), "k": _size(rng, 64, 8192), "n": _size(rng, 64, 8192),
                 "bias": rng.random() < 0.75}
            if c["m"] * c["k"] * c["n"] <= 4096 ** 3 // 2 and c["k"] * c["n"] <= 4096 * 4096:
                return c
    if kind == "batched":
        while True:
            c = {"kind": kind, "batch": _log(rng, 2, 384), "m": _size(rng, 8, 512), "k": _size(rng, 16, 512),
                 "n": _size(rng, 16, 512), "shared": rng.random() < 0.25}
            if c["batch"] * (c["m"] * c["k"] + c["k"] * c["n"] + c["m"] * c["n"]) <= 32 << 20:
                return c
    if kind == "qmatmul":
        while True:
            c = {"kind": kind, "m": _size(rng, 1, 4096), "k": _size(rng, 64, 8192), "n": _size(rng, 64, 8192),
                 "acc": rng.random() < 0.25, "exact": rng.random() < 0.5}
            if c["m"] * c["k"] * c["n"] <= 4096 ** 3 // 2:
                return c
    if kind == "qlayer":
        while True:
            c = {"kind": kind, "m": _size(rng, 1, 2048), "k": _size(rng, 64, 4096), "n": _size(rng, 64, 4096),
                 "requant": rng.random() < 0.4}
            if c["m"] * c["k"] * c["n"] <= 1 << 34:
                return c
    if kind == "decode":
        while True:
            c = {"kind": kind, "m": rng.randint(1, 8), "k": _size(rng, 512, 12288), "n": _size(rng, 512, 12288),
                 "packed": rng.random() < 0.3, "exact": rng.random() < 0.5, "acc": rng.random() < 0.25}
            if c["k"] * c["n"] <= 64 << 20:
                return c
    if kind == "encoder":
        while True:
            c = {"kind": kind, "batch": _log(rng, 1, 16), "seq": rng.choice([_log(rng, 8, 512), _size(rng, 16, 512)]),
                 "hidden": rng.choice([256, 512, 768, 768, 1024]), "mask": rng.random() < 0.5}
            if c["batch"] * c["seq"] * c["hidden"] <= 8 * 128 * 768:
                return c
    while True:
        c = {"kind": "bilstm", "seq": _log(rng, 4, 128), "batch": _log(rng, 1, 12), "length": _size(rng, 64, 1024),
             "hidden": _size(rng, 64, 1024)}
        if c["seq"] * c["batch"] * (c["length"] + c["hidden"]) <= 1 << 19:
            return c


# ---- inputs ------------------------------------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, std, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std


def _bytes(g, lo, hi, dtype, *shape):
    return torch.randint(lo, hi + 1, shape, generator=g, device="cuda", dtype=dtype)


def _scalar(v):
    return torch.tensor([v], dtype=torch.float32, device="cuda")


def _prepare_dense(c, seed):
    g = _generator(seed)
    s = {"x": _normal(g, 1.0, c["m"], c["k"]), "w": _normal(g, 0.02, c["k"], c["n"])}
    s["bias"] = _normal(g, 0.02, c["n"]) if c["bias"] else None
    return s


def _run_dense(s):
    return tfcc.blas_matmul(s["x"], s["w"], s["bias"])


def _prepare_batched(c, seed):
    g = _generator(seed)
    b = (c["k"], c["n"]) if c["shared"] else (c["batch"], c["k"], c["n"])
    return {"a": _normal(g, 1.0, c["batch"], c["m"], c["k"]), "b": _normal(g, 1.0, *b)}


def _run_batched(s):
    return tfcc.blas_matmul(s["a"], s["b"])


def _prepare_qmatmul(c, seed):
    g = _generator(seed)
    a = _bytes(g, 0, 255, torch.uint8, c["m"], c["k"])
    b = _bytes(g, -127, 127, torch.int8, c["k"], c["n"])
    # zero point 128 for the activations, symmetric weights, an output range that holds almost every sum
    bound = 5.0 * 74.0 * 74.0 * math.sqrt(c["k"])
    return {"a": a, "b": b, "row": tfcc.reduce_sum(a, True), "col": tfcc.reduce_sum(b, False),
            "range_a": (_scalar(-128.0), _scalar(127.0)), "range_b": (_scalar(-128.0), _scalar(127.0)),
            "range_out": (_scalar(-bound), _scalar(bound)), "acc": c["acc"], "exact": c["exact"]}


def _run_qmatmul(s):
    q, acc, low, high = tfcc.quantization_matmul_requantize(s["a"], s["row"], *s["range_a"], s["b"], s["col"], *s["range_b"],
                                                            *s["range_out"], want_acc=s["acc"], colsum_exact=s["exact"])
    return (q, acc, low, high) if s["acc"] else (q, low, high)


def _prepare_qlayer(c, seed):
    g = _generator(seed)
    w = _bytes(g, -127, 127, torch.int8, c["k"], c["n"])
    step = 0.05 / 127.0
    return {"x": _normal(g, 1.0, c["m"], c["k"]), "w": w, "col": tfcc.reduce_sum(w, False),
            "range_w": (_scalar(-128.0 * step), _scalar(127.0 * step)),
            "range_out": (_scalar(-0.15 * math.sqrt(c["k"])), _scalar(0.15 * math.sqrt(c["k"]))), "requant": c["requant"]}


def _run_qlayer(s):
    q, low, high = tfcc.quantize(s["x"], torch.uint8)
    row = tfcc.reduce_sum(q, True)
    if s["requant"]:
        out, _, low_c, high_c = tfcc.quantization_matmul_requantize(q, row, low, high, s["w"], s["col"], *s["range_w"],
                                                                    *s["range_out"])
        return out, low_c, high_c
    acc, low_c, high_c = tfcc.quantization_matmul(q, row, low, high, s["w"], s["col"], *s["range_w"])
    return tfcc.dequantize(acc, low_c, high_c), acc, low_c, high_c


def _prepare_decode(c, seed):
    g = _generator(seed)
    a = _bytes(g, 0, 255, torch.uint8, c["m"], c["k"])
    b = _bytes(g, -127, 127, torch.int8, c["k"], c["n"])
    s = {"a": a, "row": tfcc.reduce_sum(a, True), "col": tfcc.reduce_sum(b, False), "n": c["n"], "packed": c["packed"],
         "scale_b": torch.rand(c["n"], generator=g, device="cuda", dtype=torch.float32) * 0.009 + 0.001,
         "acc": c["acc"], "exact": c["exact"]}
    s["b"] = tfcc.gemv_pack(b) if c["packed"] else b
    return s


def _run_decode(s):
    if s["packed"]:
        out, acc = tfcc.gemv_dequant_packed(s["a"], s["b"], s["n"], s["row"], s["col"], -128, 0, 0.02, s["scale_b"],
                                            want_acc=s["acc"])
    else:
        out, acc = tfcc.gemv_dequant(s["a"], s["b"], s["row"], s["col"], -128, 0, 0.02, s["scale_b"], want_acc=s["acc"],
                                     colsum_exact=s["exact"])
    return (out, acc) if s["acc"] else out


def _prepare_encoder(c, seed):
    rng = np.random.default_rng(seed)
    weights = modelfile.bert_layer_weights(rng, c["hidden"], 4 * c["hidden"])
    graph = modelfile.bert_encoder_layer(weights, c["batch"], c["seq"], c["hidden"] // 64, with_mask=c["mask"])
    model = runtime_api.Model(modelfile.write_model([graph], graph.name))
    inputs = {"hidden_states": rng.standard_normal((c["batch"], c["seq"], c["hidden"]), dtype=np.float32)}
    if c["mask"]:
        used = rng.integers(max(1, c["seq"] // 2), c["seq"] + 1, c["batch"])
        padded = np.arange(c["seq"])[None, :] >= used[:, None]
        inputs["attention_mask"] = np.where(padded, -10000.0, 0.0).astype(np.float32).reshape(c["batch"], 1, 1, c["seq"])
    model.run(inputs)
    return {"model": model, "inputs": inputs}


def _run_model(s):
    return s["model"].run(s["inputs"])


def _prepare_bilstm(c, seed):
    rng = np.random.default_rng(seed)
    bound = 1.0 / math.sqrt(c["hidden"])

    def weights(*shape):
        return rng.uniform(-bound, bound, shape).astype(np.float32)

    state = np.zeros((2, c["batch"], c["hidden"]), dtype=np.float32)
    g = modelfile.GraphBuilder("tagger")
    ins = [g.input("x", modelfile.FLOAT, [c["seq"], c["batch"], c["length"]]),
           g.constant("input_kernel", weights(2, c["length"], 4 * c["hidden"])),
           g.constant("state_kernel", weights(2, c["hidden"], 4 * c["hidden"])),
           g.constant("bias", weights(2, 4 * c["hidden"])), g.constant("h0", state), g.constant("c0", state)]
    outs = [g.variable(name) for name in ("forward", "backward", "forward_h", "backward_h", "forward_c", "backward_c")]
    g.node("rnn.BidirectionalLSTM", ins, outs, modelfile.f_varint(1, c["hidden"]))
    for o in outs:
        g.output(o)
    model = runtime_api.Model(modelfile.write_model([g], g.name))
    inputs = {"x": rng.standard_normal((c["seq"], c["batch"], c["length"]), dtype=np.float32)}
    model.run(inputs)
    return {"model": model, "inputs": inputs}


_PREPARE = {"dense": _prepare_dense, "batched": _prepare_batched, "qmatmul": _prepare_qmatmul, "qlayer": _prepare_qlayer,
            "decode": _prepare_decode, "encoder": _prepare_encoder, "bilstm": _prepare_bilstm}
_RUN = {"dense": _run_dense, "batched": _run_batched, "qmatmul": _run_qmatmul, "qlayer": _run_qlayer, "decode": _run_decode,
        "encoder": _run_model, "bilstm": _run_model}


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, seed)
    state["run"] = _RUN[case["kind"]]
    return state


def run(state):
    return state["run"](state)


# ---- what a pass cannot do without ---------------------------------------------------------------------------------
def work(case):
    c, kind = case, case["kind"]
    if kind == "dense":
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": 4 * (m * k + k * n + m * n + (n if c["bias"] else 0)), "flops": 2 * m * k * n}
    if kind == "batched":
        m, k, n, b = c["m"], c["k"], c["n"], c["batch"]
        return {"bytes": 4 * (b * m * k + (1 if c["shared"] else b) * k * n + b * m * n), "flops": 2 * b * m * k * n}
    if kind == "qmatmul":
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": m * k + k * n + m * n + 4 * (m + n) + (4 * m * n if c["acc"] else 0), "flops": 2 * m * k * n}
    if kind == "qlayer":
        m, k, n = c["m"], c["k"], c["n"]
        # float32 activations in, weights, and out: a byte, or the int32 sums and the float32 values
        return {"bytes": 4 * m * k + k * n + 4 * n + (m * n if c["requant"] else 8 * m * n), "flops": 2 * m * k * n}
    if kind == "decode":
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": m * k + k * n + 4 * (m + 2 * n) + (8 if c["acc"] else 4) * m * n, "flops": 2 * m * k * n}
    if kind == "encoder":
        rows, h, s = c["batch"] * c["seq"], c["hidden"], c["seq"]
        return {"bytes": 4 * (2 * rows * h + 12 * h * h + 13 * h + (rows if c["mask"] else 0)),
                "flops": 2 * rows * 12 * h * h + 4 * rows * s * h}
    steps, h, length = c["seq"] * c["batch"], c["hidden"], c["length"]
    return {"bytes": 4 * (steps * (length + 2 * h) + 8 * h * (length + h + 1) + 8 * c["batch"] * h),
            "flops": 2 * 2 * steps * 4 * h * (length + h)}


def tolerance(case):
    if case["kind"] in ("qmatmul", "qlayer", "decode"):
        return "exact"  # whole numbers, and floats that are one fixed expression of them
    return {"rel": 1e-5}  # float32 sums in another order
