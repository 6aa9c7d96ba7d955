"""Performance cases of the extreme-classifier layers: what a training run, an evaluation and a serving loop ask of them.

A case names a layer (true FP8, simulated FP8, FP8 with a compensated head, bf16), a call (one training step, the dense
inference logits, the k best labels) and the sizes.  Label counts, chunkings, batches and distributions are those of the
benchmark workloads (elmo_amd/synth.py) and of the shipped dataset configurations; `draw` spreads them over the ranges
these stand for.  Label spaces of up to MODULE_LABELS go through the drop-in modules (elmo_amd.xmc_classifiers), host work
included; larger FP8 layers through the tensor-level calls (elmo_amd.ops), as bench.py does, because the modules
initialise their weights on the CPU.  The bf16 layer initialises on the GPU and always goes through its module.
"""
import math
import types

import numpy as np
import torch

from elmo_amd import ops
from elmo_amd.xmc_classifiers import Fp8XMCBCEChunkedHeadKahanLayer, Fp8XMCBCEChunkedLayer, XMCBCECHUNKEDLayer

MODULE_LABELS = 150_000
LEARNING_RATE = 0.05
DEVICE = "cuda:0"


def _case(name, layer, call, labels, chunks, batch, features=768, rounding="", positives=5.0, zipf=1.0, k=0):
    c = dict(layer=layer, call=call, labels=labels, chunks=chunks, batch=batch, features=features, rounding=rounding,
             positives=positives, zipf=zipf, k=k)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest training call: a few thousand labels, a small batch; launches and host work count
        _case("fp8_train_4k_b16", "fp8", "train", 4_000, 1, 16, rounding="sr_fast"),
        # an ordinary small dataset through the module
        _case("fp8_train_131k_b96", "fp8", "train", 131_073, 2, 96, rounding="sr_fast"),
        # the headline benchmark: 670 K labels, batch 128
        _case("fp8_train_670k_b128", "fp8", "train", 670_091, 11, 128, rounding="sr_fast", positives=5.4),
        # the same label space with the shipped configuration's batch and chunking
        _case("fp8_train_670k_b256", "fp8", "train", 670_091, 2, 256, rounding="sr_fast", positives=5.4),
        # the largest benchmark workload
        _case("fp8_train_8m6_b256", "fp8", "train", 8_600_000, 33, 256, rounding="sr_fast", positives=8.0, zipf=1.1),
        # simulated FP8 (bf16 products), the reference's stochastic rounding
        _case("simfp8_train_500k_b128", "simfp8", "train", 500_000, 8, 128, rounding="sr_philox", positives=4.8, zipf=1.05),
        # bf16 layer: the benchmark's small batch with round to nearest ...
        _case("bf16_train_131k_b32", "bf16", "train", 131_072, 8, 32, rounding="rtn", zipf=1.1),
        # ... the shipped configurations with the reference's stochastic rounding: a large batch,
        _case("bf16_train_131k_b512", "bf16", "train", 131_073, 2, 512, rounding="sr_philox"),
        # and a large label space
        _case("bf16_train_501k_b128", "bf16", "train", 501_070, 3, 128, rounding="sr_philox", positives=4.8),
        # a fifth of the labels compensated (bf16 terms)
        _case("kahan_train_670k_b128", "kahan_bf16", "train", 670_091, 3, 128, rounding="sr_fast", positives=5.4),
        # evaluation: dense logits of a last, ragged batch
        _case("fp8_logits_131k_b40", "fp8", "logits", 131_073, 2, 40),
        # evaluation: the 100 best labels of every row
        _case("fp8_topk_670k_b128", "fp8", "topk", 670_091, 11, 128, k=100),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fp8", "fp8", "fp8_wide", "simfp8", "bf16", "bf16", "kahan", "logits", "topk"])
    rows = rng.choice([16_384, 65_536, 131_072, 262_144])           # label rows per chunk, roughly
    chunks = lambda labels: max(1, min(64, round(labels / rows)))   # noqa: E731
    pos = dict(positives=round(rng.choice([rng.uniform(2.0, 10.0), rng.uniform(2.0, 10.0), 36.0]), 1),
               zipf=round(rng.uniform(0.9, 1.1), 2))
    sixteens = lambda lo, hi: 16 * rng.randint(lo // 16, hi // 16)  # noqa: E731
    if kind == "fp8":          # batches of up to 128 rows
        labels = _log_int(rng, 2_000, 2_812_281)
        return _case("", "fp8", "train", labels, chunks(labels), sixteens(16, 128),
                     rounding=rng.choice(["sr_fast", "sr_fast", "sr_philox", "rtn"]), **pos)
    if kind == "fp8_wide":     # larger batches, and layers of 1,024 features
        labels = _log_int(rng, 8_000, 2_000_000)
        features = rng.choice([768, 768, 1024])
        return _case("", "fp8", "train", labels, chunks(labels), sixteens(144, 512) if features == 768 else sixteens(32, 512),
                     features=features, rounding=rng.choice(["sr_fast", "sr_fast", "sr_philox", "rtn"]), **pos)
    if kind == "simfp8":
        labels = _log_int(rng, 2_000, 700_000)
        return _case("", "simfp8", "train", labels, chunks(labels), rng.randint(1, 256), features=rng.choice([768, 768, 1024]),
                     rounding=rng.choice(["sr_philox", "sr_philox", "rtn"]), **pos)
    if kind == "bf16":
        labels = _log_int(rng, 2_000, 1_500_000)
        return _case("", "bf16", "train", labels, chunks(labels), _log_int(rng, 8, 512), features=rng.choice([768, 768, 1024]),
                     rounding=rng.choice(["sr_philox", "sr_philox", "rtn", "sr_fast"]), **pos)
    if kind == "kahan":
        labels = _log_int(rng, 8_000, 900_000)
        return _case("", rng.choice(["kahan_bf16", "kahan_e5m2"]), "train", labels, max(1, min(4, chunks(labels))),
                     sixteens(16, 128), rounding=rng.choice(["sr_fast", "sr_fast", "rtn"]), **pos)
    if kind == "logits":
        labels = _log_int(rng, 2_000, 1_000_000)
        return _case("", "fp8", "logits", labels, chunks(labels), rng.randint(1, 256))
    labels = _log_int(rng, 2_000, 2_812_281)
    return _case("", "fp8", "topk", labels, chunks(labels), rng.randint(1, 256), k=rng.choice([1, 5, 5, 20, 100]))


def _rows_per_chunk(case):
    """Rows of a chunk as the layers cut the label space (FP8 layers pad it, the bf16 layer does not)."""
    labels, nc = case["labels"], case["chunks"]
    if case["layer"] == "bf16":
        return -(-labels // nc)
    return (labels + 16 * nc - labels % (16 * nc)) // nc


def _num_head(case):
    rows = _rows_per_chunk(case)
    return min(int(0.2 * rows * case["chunks"]), rows) if case["layer"].startswith("kahan") else 0


def _through_module(case):
    return case["layer"] == "bf16" or case["labels"] <= MODULE_LABELS


def _config(case):
    """The attribute-style configuration the modules read."""
    ns = types.SimpleNamespace
    rows = _rows_per_chunk(case)
    xmc = ns(simulated_fp8=case["layer"] == "simfp8", momentum=0, wd=0)
    if case["rounding"]:
        xmc.rounding = case["rounding"]
    # the head is given as a share of the padded label space; half a row is added so that the product truncates to it
    head = (_num_head(case) + 0.5) / (rows * case["chunks"])
    return ns(environment=ns(device=DEVICE), data=ns(num_labels=case["labels"], batch_size=case["batch"]),
              model=ns(xmc=ns(num_chunks=case["chunks"], input_features=case["features"],
                              dtype="bfloat16" if case["layer"] == "bf16" else "float8")),
              training=ns(xmc=xmc, precision=ns(mode="custom", purelp_dtype="bfloat16"),
                          FP8=ns(using_head_kahan=case["layer"].startswith("kahan"),
                                 fp8_head_kahan=case["layer"] == "kahan_e5m2", head_ratio=head)))


def _positives(case, rng):
    """COO int32 [n, 2] positives, row by row: Poisson many per row, drawn from a bounded Zipf law over the labels by the
    inverse of its continuous distribution function, without repetition within a row."""
    L, s = float(case["labels"]), case["zipf"]
    counts = rng.poisson(case["positives"], size=case["batch"])
    u = rng.random(int(counts.sum()))
    if abs(s - 1.0) < 1e-9:
        rank = np.exp(u * math.log(L))
    else:
        rank = ((L ** (1.0 - s) - 1.0) * u + 1.0) ** (1.0 / (1.0 - s))
    pairs = np.stack([np.repeat(np.arange(case["batch"]), counts), np.clip(rank.astype(np.int64) - 1, 0, int(L) - 1)], axis=1)
    return np.unique(pairs, axis=0).astype(np.int32).reshape(-1, 2)


def prepare(case, seed):
    """Weights (or the module that holds them), one batch of embeddings and its positives, on the GPU."""
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    x = torch.randn(case["batch"], case["features"], generator=gen, device=DEVICE)
    x = (x / x.norm(dim=1, keepdim=True)).to(torch.bfloat16)
    state = dict(case=case, x=x)
    if case["call"] == "train":
        state["positives"] = torch.from_numpy(_positives(case, rng)).to(DEVICE)
    torch.manual_seed(seed)        # the modules draw their initial weights and every step's rounding seeds from here
    if _through_module(case):
        layer = {"fp8": Fp8XMCBCEChunkedLayer, "simfp8": Fp8XMCBCEChunkedLayer, "bf16": XMCBCECHUNKEDLayer}.get(
            case["layer"], Fp8XMCBCEChunkedHeadKahanLayer)
        state["module"] = layer(_config(case))
        return state
    nc, rows, feats = case["chunks"], _rows_per_chunk(case), case["features"]
    state["chunks"] = []
    for _ in range(nc):
        w = torch.randn(rows, feats, generator=gen, device=DEVICE)
        state["chunks"].append(w.mul_(0.02).to(torch.float8_e4m3fn))
        del w
    state["seeds"] = rng
    if case["call"] == "train" and (case["layer"] == "simfp8" or case["batch"] > ops.MAX_BATCH or feats != ops.FEATURES):
        state["workspace"] = ops.alloc_tiled_workspace(nc, rows, torch.device(DEVICE), case["batch"], feats)
    else:
        state["workspace"] = ops.alloc_workspace(nc, rows, torch.device(DEVICE))
    if case["layer"].startswith("kahan"):
        state["kahan"] = torch.zeros(_num_head(case), feats, device=DEVICE,
                                     dtype=torch.bfloat16 if case["layer"] == "kahan_bf16" else torch.float8_e5m2)
    return state


def run(state):
    case, x = state["case"], state["x"]
    if "module" in state:
        m = state["module"]
        if case["call"] == "logits":
            return m.xfc_forward(x)
        if case["call"] == "topk":
            return m.xfc_forward_topk(x, case["k"])
        m.xfc_forward_backward(x, state["positives"], [LEARNING_RATE])
        out = {"grad": m.grad_input, "weights": [w.detach() for w in m.xfc_weight] if case["layer"] != "bf16" else m.xfc_weight}
        if case["layer"].startswith("kahan"):
            out["compensation"] = m.head_kahan
        return out
    chunks, ws = state["chunks"], state["workspace"]
    if case["call"] == "logits":
        return ops.fp8_forward(chunks, x, case["labels"], workspace=ws)
    if case["call"] == "topk":
        return ops.fp8_forward_topk(chunks, x, case["labels"], case["k"], workspace=ws)
    seeds = state["seeds"].integers(0, 1_000_000, size=len(chunks))
    out = {"weights": chunks}
    if case["layer"].startswith("kahan"):
        out["grad"] = ops.fp8_kahan_step(chunks, state["kahan"], _num_head(case), x, state["positives"], LEARNING_RATE,
                                         seeds=seeds, round_mode=case["rounding"], workspace=ws)
        out["compensation"] = state["kahan"]
    elif case["layer"] == "fp8" and case["batch"] <= ops.MAX_BATCH and case["features"] == ops.FEATURES:
        out["grad"] = ops.fp8_step(chunks, x, state["positives"], LEARNING_RATE, seeds=seeds, round_mode=case["rounding"],
                                   workspace=ws)
    else:      # simulated FP8, more than 128 batch rows or 1,024 features: the three-kernel path
        true_fp8 = case["layer"] == "fp8"
        out["grad"] = ops.tiled_step(chunks, chunks[0].shape[0], "e4m3", x, state["positives"], LEARNING_RATE, seeds=seeds,
                                     round_mode=case["rounding"], workspace=ws, quantize_x=true_fp8, saturate=true_fp8)
    return out


def work(case):
    """A training step reads and writes every weight once and is three products of [batch x features x labels]; inference
    reads the weights once, is one product and writes the logits or the k best."""
    b, d = case["batch"], case["features"]
    if case["call"] != "train":
        labels = case["labels"]
        out = 2 * b * labels if case["call"] == "logits" else 10 * b * case["k"]
        return {"bytes": labels * d + 2 * b * d + out, "flops": 2 * b * labels * d}
    labels = case["labels"] if case["layer"] == "bf16" else _rows_per_chunk(case) * case["chunks"]
    weight = 2 if case["layer"] == "bf16" else 1
    terms = _num_head(case) * d * {"kahan_bf16": 2, "kahan_e5m2": 1}.get(case["layer"], 0)
    return {"bytes": 2 * labels * d * weight + 2 * terms + 4 * b * d + 8 * int(b * case["positives"]), "flops": 6 * b * labels * d}


def tolerance(case):
    # bf16 gradients and weights, e4m3 weights of which a few may land on the neighbouring grid point; indices may trade
    # places where two logits round to the same bf16 value.  A compensation term turns over with its weight.
    if case["call"] == "topk":
        return {"rel": 1e-2, "differ": 1e-2}
    if case["layer"].startswith("kahan"):
        return {"rel": 1e-2, "max": 0.99}
    return {"rel": 1e-2}
