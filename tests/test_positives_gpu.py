"""Tiles with many positives: the counts at which the step kernels change the way they read a tile's keys (eight, a wavefront's
worth, four of those), with repetitions and in no order, against the oracle."""
import numpy as np
import pytest

import helpers as H
import test_cluster_gpu as T
import test_three_kernel_gpu as K
from test_fp8_step_gpu import check_rtn

pytestmark = pytest.mark.gpu

ROWS = 208


def crowded(n, batch, rows):
    """n positives of 64 labels (the second tile of the second chunk), a few of them twice, and one of each neighbouring label."""
    rng = np.random.default_rng(n)
    first = rows + 64
    rows_of = rng.integers(0, batch, n)
    labels = first + rng.integers(0, 64, n)
    both = np.stack([rows_of, labels], axis=1)
    both[n - n // 3:] = both[:n // 3]
    return np.concatenate([both[rng.permutation(n)], [[0, first - 1], [batch - 1, first + 64]]]).astype(np.int32)


@pytest.mark.parametrize("n", [1, 8, 9, 64, 65, 256, 257, 5000, 32766])
@pytest.mark.parametrize("batch", [16, 128])
def test_fused_step(gpu, n, batch):
    """At 16 rows the variant of the role kernel for one block of 32, which larger label spaces take: more than 4,096 pairs keep so few labels
    off the small step's kernel, and pairs outside the batch are ignored."""
    case = H.make_case(3, ROWS, batch, 70 + n)
    case["labels"] = crowded(n, batch, ROWS)
    ignored = 4097 if batch == 16 and n < 4096 else 0
    check_rtn(case, gpu, device_labels=np.concatenate([case["labels"], np.tile([[-1, 0]], (ignored, 1))]))


@pytest.mark.parametrize("n", [1, 8, 9, 64, 65, 256, 257, 510, 511, 1000, 4094])     # (two more in all: 512 threads, 4,096 at most)
@pytest.mark.parametrize("batch", [16, 32])
def test_small_step(gpu, n, batch):
    case = H.make_case(3, ROWS, batch, 70 + n)
    case["labels"] = crowded(n, batch, ROWS)
    check_rtn(case, gpu)


@pytest.mark.parametrize("kind,batch", [("bf16", 20), ("bf16", 512), ("sim", 64), ("sim", 128), ("fp8", 64), ("fp8", 256), ("fp8", 300)])
@pytest.mark.parametrize("n", [8, 9, 257, 5000])
def test_one_pass_step(gpu, kind, batch, n, monkeypatch):
    labels = crowded(n, batch, ROWS)
    make_case, bf16_case = H.make_case, T.bf16_case
    monkeypatch.setattr(H, "make_case", lambda *a, **k: dict(make_case(*a, **k), labels=labels))
    monkeypatch.setattr(T, "bf16_case", lambda *a, **k: bf16_case(*a, **k)[:2] + (labels,))
    T.test_one_pass_step_matches_the_oracle(gpu, kind, 3, ROWS, batch, "rtn")


@pytest.mark.parametrize("kind,batch", [("bf16", 20), ("bf16", 300), ("sim", 128), ("fp8", 64), ("fp8", 300)])
@pytest.mark.parametrize("n", [8, 9, 257, 5000, 32761])     # (the most, 32,768, less two neighbours and five edges of the bf16 case)
def test_three_kernel_step(gpu, kind, batch, n, monkeypatch):
    labels = crowded(n, batch, ROWS)
    make_case, bf16_case = H.make_case, K.bf16_case
    monkeypatch.setattr(H, "make_case", lambda *a, **k: dict(make_case(*a, **k), labels=labels))
    monkeypatch.setattr(K, "bf16_case", lambda *a, **k: bf16_case(*a, **k)[:2] + (labels,))
    K.test_step_with_weight_decay_matches_the_oracle(gpu, kind, 3, ROWS, batch, "rtn")


@pytest.mark.parametrize("n", [9, 5000])
def test_loss(gpu, n, monkeypatch):
    labels, bf16_case = crowded(n, 300, ROWS), K.bf16_case
    monkeypatch.setattr(K, "bf16_case", lambda *a, **k: bf16_case(*a, **k)[:2] + (labels,))
    K.test_loss_over_four_halves(gpu)
