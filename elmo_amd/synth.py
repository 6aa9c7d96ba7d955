"""Seeded synthetic inputs of the shapes the benchmark configurations name.

X       fp32 N(0,1) rows, L2-normalised in fp32, rounded to bf16
labels  per row n_i ~ Poisson(mean) positives drawn from a bounded Zipf over label ranks 1..L
        (p(r) ~ r^-s, inverse-CDF sampling), label id = r-1, de-duplicated within a row, emitted as the
        COO int32 [Nb, 2] (row-in-batch, label) array the reference's collate produces (src/data.py:16-33)
W       fp32 N(0, std) -- generated by the caller on the device it needs it on (see weights_*)
"""
from dataclasses import dataclass

import numpy as np


@dataclass(frozen=True)
class StepConfig:
    name: str
    num_labels: int
    batch: int
    dim: int
    chunk: int            # target rows per chunk; num_chunks = ceil(L / chunk)
    pos_mean: float
    zipf_s: float
    seed: int
    weights: str          # "e4m3" | "bf16"
    lr: float = 0.05
    init_std: float = 0.02

    @property
    def num_chunks(self):
        return -(-self.num_labels // self.chunk)


CONFIGS = {
    "cfg1_bf16_131k": StepConfig("cfg1_bf16_131k", 131072, 32, 768, 16384, 5.0, 1.1, 0, "bf16"),
    "cfg2_fp8_670k": StepConfig("cfg2_fp8_670k", 670091, 128, 768, 65536, 5.4, 1.0, 1, "e4m3"),
    "cfg3_simfp8_500k": StepConfig("cfg3_simfp8_500k", 500000, 128, 768, 65536, 4.8, 1.05, 3, "e4m3"),
    "cfg4_fp8_3m": StepConfig("cfg4_fp8_3m", 2812281, 128, 768, 131072, 36.0, 0.9, 4, "e4m3"),
    "cfg5_fp8_8m6": StepConfig("cfg5_fp8_8m6", 8600000, 256, 768, 262144, 8.0, 1.1, 5, "e4m3"),
    # the first and the third workload with an encoder of 1024 features (tiled step)
    "cfg1_bf16_131k_d1024": StepConfig("cfg1_bf16_131k_d1024", 131072, 32, 1024, 16384, 5.0, 1.1, 0, "bf16"),
    "cfg3_simfp8_500k_d1024": StepConfig("cfg3_simfp8_500k_d1024", 500000, 128, 1024, 65536, 4.8, 1.05, 3, "e4m3"),
}


def make_x(batch, dim, seed):
    """bf16-valued fp32 array [batch, dim] with unit-norm rows (before the bf16 rounding)."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((batch, dim)).astype(np.float32)
    x /= np.linalg.norm(x, axis=1, keepdims=True).astype(np.float32)
    u = x.view(np.uint32).astype(np.uint64)
    u = ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).astype(np.uint32)
    return u.view(np.float32)


def make_labels(batch, num_labels, pos_mean, zipf_s, seed):
    """COO int32 [Nb, 2] positives, row-major order."""
    rng = np.random.default_rng(seed + 7919)
    ranks = np.arange(1, num_labels + 1, dtype=np.float64)
    cdf = np.cumsum(ranks ** (-zipf_s))
    cdf /= cdf[-1]
    out = []
    counts = rng.poisson(pos_mean, size=batch)
    for b in range(batch):
        if counts[b] == 0:
            continue
        ids = np.searchsorted(cdf, rng.random(counts[b]), side="left")
        ids = np.unique(np.minimum(ids, num_labels - 1))
        out.append(np.stack([np.full(len(ids), b, dtype=np.int64), ids], axis=1))
    if not out:
        return np.zeros((0, 2), dtype=np.int32)
    return np.concatenate(out, axis=0).astype(np.int32)


def make_weights_np(rows, dim, seed, std=0.02):
    """fp32 N(0, std) [rows, dim] on the CPU (for small shapes / the oracle)."""
    rng = np.random.default_rng(seed + 104729)
    return (rng.standard_normal((rows, dim)) * std).astype(np.float32)
