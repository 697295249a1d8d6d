"""The work that users of this package have it do, as cases for a timing program: the SpMM operator and its plan form,
the drop-in layers and fused blocks of the models, and the conversion of weights to V:N:M and back.

A case is a dict of plain values; `listed()` names the fixed ones, `draw(rng)` gives another of the same ranges,
`prepare` makes what a program holds before the call, `run` is one pass through the public entry points."""
import math

import torch

from venom_amd import bert, gpt3, spatha
from venom_amd import format as vnm_format

# (rows, cols) of the projections of BERT-base, BERT-large, GPT-2-large and a GPT-3-sized block
LAYERS = [(768, 768), (3072, 768), (768, 3072), (1024, 1024), (3072, 1024), (4096, 1024), (1024, 4096), (1280, 1280),
          (3840, 1280), (5120, 1280), (1280, 5120), (12288, 12288), (36864, 12288), (49152, 12288), (12288, 49152)]
FORMATS_M = [4, 7, 8, 10, 16, 20, 32, 40]
DEVICE = "cuda:0"


def listed():
    return [
        # one token of eight sequences through one projection of a BERT-large-sized model: the smallest call, all latency
        {"name": "layer_1024_decode8", "kind": "layer", "rows": 1024, "cols": 1024, "v": 64, "m": 8, "tokens": 8},
        # decoding with the GPT-3 feed-forward matrix: sixteen tokens, the stream of the weights is all that matters
        {"name": "op_gpt3_ffn_decode16", "kind": "op", "rows": 49152, "cols": 12288, "v": 128, "m": 16, "tokens": 16},
        # a batch of sequences on the same matrix, and a prompt: the largest single product
        {"name": "op_gpt3_ffn_256", "kind": "op", "rows": 49152, "cols": 12288, "v": 128, "m": 16, "tokens": 256},
        {"name": "plan_gpt3_ffn_2048", "kind": "plan", "rows": 49152, "cols": 12288, "v": 128, "m": 16, "tokens": 2048,
         "transposed": False, "activation": ""},
        # GPT-2-large's feed-forward matrix with as many tokens as a prompt happens to have (odd)
        {"name": "op_gpt2_ffn_1037", "kind": "op", "rows": 5120, "cols": 1280, "v": 64, "m": 10, "tokens": 1037},
        # the reference's benchmark: its --check shape, and the BERT-large feed-forward matrix over 32 x 512 tokens
        {"name": "plan_1024x4096x4096", "kind": "plan", "rows": 1024, "cols": 4096, "v": 128, "m": 8, "tokens": 4096,
         "transposed": False, "activation": ""},
        {"name": "plan_bert_ffn_up_16384", "kind": "plan", "rows": 4096, "cols": 1024, "v": 64, "m": 8, "tokens": 16384,
         "transposed": False, "activation": ""},
        # the small V of the reference's ablation, at a sparser format
        {"name": "op_v32_4096", "kind": "op", "rows": 1024, "cols": 4096, "v": 32, "m": 16, "tokens": 4096},
        # two encoder layers of BERT-large over 32 x 512 tokens, everything the package fuses switched on
        {"name": "bert_encoder_32x512", "kind": "encoder", "layers": 2, "v": 64, "m": 8, "batch": 32, "seq": 512},
        # GPT-2-large's feed-forward block on one ragged prompt
        {"name": "gpt2_mlp_301", "kind": "mlp", "width": 1280, "v": 128, "m": 16, "tokens": 301, "kernel_act": True},
        # model conversion: magnitude selection and encoding of one fp16 weight, and the way back
        {"name": "convert_4096x1024", "kind": "convert", "rows": 4096, "cols": 1024, "v": 64, "m": 8},
        {"name": "to_dense_1024x4096", "kind": "to_dense", "rows": 1024, "cols": 4096, "v": 128, "m": 16},
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["layer", "op", "op", "plan", "plan", "mlp", "encoder", "convert", "to_dense"])
    v, m = rng.choice([32, 64, 64, 128, 128]), rng.choice(FORMATS_M)
    if kind == "encoder":
        return {"kind": kind, "layers": rng.choice([1, 2]), "v": rng.choice([64, 128]), "m": rng.choice([8, 16, 32]),
                "batch": rng.choice([1, 2, 8, 16, 32]), "seq": rng.randint(5, 512)}
    if kind == "mlp":
        return {"kind": kind, "width": rng.choice([768, 1024, 1280]), "v": rng.choice([64, 128]), "m": m,
                "tokens": _log_uniform(rng, 1, 8192), "kernel_act": rng.random() < 0.5}
    if kind in ("convert", "to_dense"):
        rows, cols = rng.choice([s for s in LAYERS if s[0] * s[1] <= 4096 * 1024])
        return {"kind": kind, "rows": rows, "cols": cols, "v": v, "m": rng.choice([4, 7, 8, 10, 16])}
    rows, cols = rng.choice(LAYERS)
    if kind == "layer" and rows * cols > 5120 * 1280:
        rows, cols = rng.choice([s for s in LAYERS if s[0] * s[1] <= 5120 * 1280])
    # no more multiplications and no larger an output than the largest listed case
    most = min(16384, 49152 * 12288 // 16 * 2048 // (rows * cols // m), 49152 * 2048 // max(rows, cols))
    case = {"kind": kind, "rows": rows, "cols": cols, "v": v, "m": m, "tokens": _log_uniform(rng, 1, most)}
    if rng.random() < 0.5:
        case["tokens"] = max(1, case["tokens"] // 8 * 8)
    if kind == "plan":
        case["transposed"] = rng.random() < 0.4
        case["activation"] = rng.choice(["", "", "gelu", "gelu_tanh"]) if v != 32 else ""
    return case


def _vnm_matrix(case, gen):
    """A V:N:M matrix in the package's storage arrays: per V x m block four columns drawn uniformly, per row two of the
    four, values ~N(0, 0.02)."""
    rows, cols, v, m = case["rows"], case["cols"], case["v"], case["m"]
    geo = vnm_format.geometry(rows, cols, 2, m, v)
    groups = geo.ksp // 2
    columns = torch.zeros((rows // v, groups, 4), dtype=torch.int32, device=DEVICE)
    full = cols // m
    keys = torch.rand((rows // v, full, m), generator=gen, device=DEVICE)
    columns[:, :full] = keys.argsort(-1)[..., :4].sort(-1).values.to(torch.int32)
    if cols % m:
        columns[:, full] = torch.arange(4, dtype=torch.int32, device=DEVICE)
    pairs = torch.tensor([4, 8, 12, 9, 13, 14], dtype=torch.int32, device=DEVICE)      # low position | high position << 2
    metadata = torch.zeros(geo.n_metadata, dtype=torch.int32, device=DEVICE)
    for nibble in range(8):
        metadata |= pairs[torch.randint(6, (geo.n_metadata,), generator=gen, device=DEVICE)] << (4 * nibble)
    values = torch.empty(geo.n_values, dtype=torch.float16, device=DEVICE).normal_(0, 0.02, generator=gen)
    return values, metadata, columns.reshape(-1)


def _normal(shape, std, gen):
    return torch.empty(shape, dtype=torch.float16, device=DEVICE).normal_(0, std, generator=gen)


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    kind = case["kind"]
    with torch.no_grad():
        if kind in ("op", "plan"):
            values, metadata, columns = _vnm_matrix(case, gen)
            state = {"case": case, "rhs": _normal((case["cols"], case["tokens"]), 1.0, gen), "bias": _normal((case["rows"],), 0.02, gen)}
            if kind == "op":
                state.update(values=values, metadata=metadata, columns=columns)
            else:
                state["plan"] = spatha.SpmmPlan(values, metadata, columns, case["rows"], case["cols"], 2, case["m"], case["v"])
            return state
        if kind == "layer":
            linear = torch.nn.Linear(case["cols"], case["rows"], device=DEVICE, dtype=torch.float16)
            linear.weight.normal_(0, 0.02, generator=gen)
            linear.bias.normal_(0, 0.02, generator=gen)
            return {"case": case, "layer": bert.SrnmSpmm(linear, 2, case["m"], case["v"], magnitude=True).eval(),
                    "x": _normal((case["tokens"], case["cols"]), 1.0, gen)}
        if kind == "mlp":
            width = case["width"]
            block = gpt3.build_gpt3_block(width, width // 64, 64, seed=seed).half().to(DEVICE)
            mlp = gpt3.conv1d_to_spmm(block, 2, case["m"], case["v"], magnitude=True)
            bert.fuse_feed_forward(mlp, activation_in_kernel=case["kernel_act"])
            return {"case": case, "mlp": mlp.mlp, "x": _normal((1, case["tokens"], width), 1.0, gen)}
        if kind == "encoder":
            model = bert.build_bert_large(case["layers"], seed=seed).to(DEVICE).half()
            bert.linear_to_spmm(model, 2, case["m"], case["v"], magnitude=True)
            bert.fuse_feed_forward(model, activation_in_kernel=True)
            bert.merge_qkv(model)
            bert.fuse_add_layernorm(model, feature_major=True)
            ids = torch.randint(30522, (case["batch"], case["seq"]), generator=gen, device=DEVICE)
            return {"case": case, "model": model, "ids": ids}
        weight = _normal((case["rows"], case["cols"]), 0.02, gen)
        sparsifier = bert.NMVectorSparsifier(2, case["m"], case["v"], magnitude=True)
        if kind == "convert":
            return {"case": case, "sparsifier": sparsifier, "weight": weight}
        return {"case": case, "matrix": sparsifier(weight).wrapped_tensor}


def run(state):
    case = state["case"]
    kind = case["kind"]
    with torch.no_grad():
        if kind == "op":
            return spatha.spmm(state["metadata"], state["columns"], state["values"], state["rhs"], state["bias"], case["rows"],
                               case["cols"], case["tokens"], case["v"], 2, case["m"])
        if kind == "plan":
            if case["activation"]:
                return state["plan"].run(state["rhs"], bias=state["bias"], transposed_out=case["transposed"],
                                         activation=case["activation"])
            return state["plan"].run(state["rhs"], bias=state["bias"] if case["transposed"] else None, transposed_out=case["transposed"])
        if kind == "layer":
            return state["layer"](state["x"])
        if kind == "mlp":
            return state["mlp"](state["x"])
        if kind == "encoder":
            return state["model"](state["ids"]).last_hidden_state
        if kind == "convert":
            matrix = state["sparsifier"](state["weight"]).wrapped_tensor
            return {"values": matrix.values, "metadata": matrix.metadata, "columns": matrix.columns}
        return state["matrix"].to_dense()


def _matrix_bytes(rows, cols, v, m):
    ksp = (-(-cols // m) * 2 + 15) // 16 * 16
    return 2 * rows * ksp + rows // 2 * (ksp // 8) * 4 + rows // v * (ksp // 2) * 16


def _product(rows, cols, v, m, tokens, act_in=True, act_out=True):
    nonzeros = -(-cols // m) * 2
    moved = _matrix_bytes(rows, cols, v, m) + 2 * rows + 2 * tokens * (cols * act_in + rows * act_out)
    return moved, 2 * rows * nonzeros * tokens


def work(case):
    kind, v, m = case["kind"], case["v"], case["m"]
    if kind in ("op", "plan", "layer"):
        moved, flops = _product(case["rows"], case["cols"], v, m, case["tokens"])
    elif kind == "mlp":
        w = case["width"]
        up, down = _product(4 * w, w, v, m, case["tokens"], act_out=False), _product(w, 4 * w, v, m, case["tokens"], act_in=False)
        moved, flops = up[0] + down[0], up[1] + down[1]
    elif kind == "encoder":
        tokens = case["batch"] * case["seq"]
        shapes = [(3072, 1024), (1024, 1024), (4096, 1024), (1024, 4096)]
        parts = [_product(r, c, v, m, tokens, False, False) for r, c in shapes]
        # the ids and the rows of the embedding that they name in, the last hidden state out; attention's two dense products
        moved = case["layers"] * sum(p[0] for p in parts) + tokens * (8 + 2 * 1024 + 2 * 1024)
        flops = case["layers"] * (sum(p[1] for p in parts) + 4 * tokens * case["seq"] * 1024)
    else:
        rows, cols = case["rows"], case["cols"]
        moved = 2 * rows * cols + _matrix_bytes(rows, cols, v, m)
        # converting: per row of a V x m block and per choice of four columns, the two largest of four and two additions
        flops = math.comb(m, 4) * (cols // m) * rows * 7 if kind == "convert" else 0
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """fp16 operands, fp32 sums, one rounding to fp16 at the end of each product (two with a bias).  Against the same path in
    64 bits (32 for the encoder) the listed products are off by 2.1e-4 to 2.9e-4 (norm) and 4.9e-4 to 9.7e-4 (entry), the
    feed-forward block by 3.8e-4 and 1.7e-3, the encoder by 7.0e-4 and 4.1e-3; four times that is allowed.  Converting and
    decoding move numbers and choose by comparing sums of a fixed order."""
    kind = case["kind"]
    if kind in ("convert", "to_dense"):
        return "exact"
    if kind == "encoder":
        return {"rel": 2.8e-3, "max": 1.6e-2}
    if kind == "mlp":
        return {"rel": 1.5e-3, "max": 7e-3}
    return {"rel": 1.2e-3, "max": 4e-3}
