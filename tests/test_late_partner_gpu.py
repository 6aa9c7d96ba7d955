"""Waits that expire for a partner that is merely late (a polling limit of 1, set from the host; with 0 the partner leaves): the
workgroup that gave up and the one that goes on must both stop.  Every kernel ends; each member's share of a row either keeps its old
codes or holds the oracle's update; a step whose error word is clear is complete; and the next step is clean."""
import numpy as np
import pytest

import helpers as H
from oracle import step as O

pytestmark = pytest.mark.gpu

NC, ROWS = 2, 8192


@pytest.mark.parametrize("entry,batch,members", [("fused", 32, 4), ("fused", 64, 4), ("fused", 128, 4), ("one pass", 128, 2), ("one pass", 192, 3),
                                                 ("one pass", 256, 4), ("one pass", 384, 6), ("one pass", 512, 8)])
def test_gives_up_cleanly(gpu, entry, batch, members):
    import torch
    from elmo_amd import ops
    # the labels of a tile positive for the first batch rows, six times over: members with the first 256 batch rows go through 24 K
    # keys, those of the others (clusters of six and eight) through none, and wait some ten thousand clocks; two polls take a thousand
    dense = [[b, 1024 + l] for _ in range(6) for l in range(64) for b in range(min(batch, 64))]
    case = H.make_case(NC, ROWS, batch, 619, extra_labels=dense)
    chunks, x, labels = H.to_device_case(case, gpu)
    ref, _, _ = O.fp8_step(case["chunks"], case["x"], case["labels"], 0.05, sr_mode="rtn")
    if entry == "fused":
        ws = ops.alloc_workspace(NC, ROWS, gpu)
    else:
        ws = ops.alloc_tiled_workspace(NC, ROWS, gpu, batch)

    def step():
        """The error word of a step from the old codes on, and for every member's share of a row whether it is old, whether it is right."""
        for c, old in zip(chunks, case["chunks"]):
            c.view(torch.uint8).copy_(torch.from_numpy(old))
        if entry == "fused":
            ops.fp8_step(chunks, x, labels, 0.05, round_mode="rtn", workspace=ws)
            word = ops.step_error_word(ws, NC, ROWS)
        else:
            ops.tiled_step(chunks, ROWS, "e4m3", x, labels, 0.05, round_mode="rtn", workspace=ws, quantize_x=True, saturate=True)
            off = ops.tiled_error_offset()
            word = int(ws[off:off + 4].view(torch.int32).item())
        new = H.chunks_to_numpy(chunks)
        shape = (-1, members, 768 // members)
        same = [(n == old).reshape(shape).all(axis=2) for n, old in zip(new, case["chunks"])]
        good = [(H.e4m3_ulp_distance(n, r) <= 1).reshape(shape).all(axis=2) for n, r in zip(new, ref)]
        return word, same, good

    expired = 0
    prev = ops.debug_spin_limit(1)
    try:
        for _ in range(4):
            word, same, good = step()
            assert word in (0, 1)
            expired += word
            for s, g in zip(same, good):
                assert np.all(s | g), "weights were updated from incomplete data"
            assert word == 1 or all(g.all() for g in good)
    finally:
        assert ops.debug_spin_limit(prev) == 1
    print("%d of 4 steps gave up" % expired)     # (where all members read the same keys, who is late is a question of timing)
    assert expired == 4 or members <= 4
    word, _, good = step()
    assert word == 0 and all(g.all() for g in good)
