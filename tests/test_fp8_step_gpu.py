"""Parity of the fused HIP step (through the C ABI) against the CPU oracle on identical seeded inputs.

Tolerances (round-to-nearest mode): updated weights within 1 e4m3 grid step of the oracle, with all but a
small fraction identical; grad_X fp32 accumulator within 1e-2 relative (measured against the largest entry),
bf16 grad_input within 1 bf16 ulp wherever the accumulator is not within rounding noise of zero."""
import numpy as np
import pytest

import helpers as H
from oracle import codecs as C
from oracle import step as O

pytestmark = pytest.mark.gpu


def run_rtn(case, device, lr=0.05, scale_w=1.0, scale_x=1.0, device_labels=None, **extra):
    import torch
    from elmo_amd import ops
    chunks, x, labels = H.to_device_case(case, device)
    if device_labels is not None:      # what the device is handed, when it differs from what the oracle is handed
        labels = torch.from_numpy(np.ascontiguousarray(device_labels, dtype=np.int32)).to(device)
    ws = ops.alloc_workspace(len(chunks), chunks[0].shape[0], device)
    g, gf = ops.fp8_step(chunks, x, labels, lr, round_mode="rtn", scale_w=scale_w, scale_x=scale_x, workspace=ws,
                         want_f32=True, **extra)
    assert ops.step_error_word(ws, len(chunks), chunks[0].shape[0]) == 0
    new = H.chunks_to_numpy(chunks)
    ref_codes, ref_gx, ref_gb = O.fp8_step(case["chunks"], case["x"], case["labels"], lr, sr_mode="rtn",
                                           scale_w=scale_w, scale_x=scale_x, **extra)
    return new, gf.cpu().numpy(), H.bf16_tensor_to_f32_numpy(g), ref_codes, ref_gx, ref_gb


def check_rtn(case, device, **kw):
    new, gx, gb, ref_codes, ref_gx, ref_gb = run_rtn(case, device, **kw)
    total = mism = 0
    for a, b in zip(new, ref_codes):
        d = H.e4m3_ulp_distance(a, b)
        assert d.max() <= 1, f"weights differ by {d.max()} grid steps"
        mism += int((d != 0).sum())
        total += d.size
    assert mism / total < 2e-3, f"{mism}/{total} updated weights differ from the oracle"
    scale = np.abs(ref_gx).max()
    assert np.abs(gx - ref_gx).max() <= 1e-2 * scale
    assert np.abs(gx - ref_gx).max() <= 1e-3 * scale      # fp32 reassociation plus a few 1-ulp flips of bf16 G
    # grad_input is the round-to-nearest-even bf16 image of the fp32 accumulator ...
    assert np.array_equal(C.bf16_bits(gb), C.bf16_bits(C.bf16_round(gx)))
    # ... and within 1 bf16 ulp of the oracle's wherever the two accumulators agree to a quarter ulp
    ulp = np.abs(ref_gb) * 2.0 ** -8 + 1e-30
    close = np.abs(gx - ref_gx) < 0.25 * ulp
    assert close.mean() > 0.5
    assert H.bf16_ulp_distance(gb, ref_gb)[close].max() <= 1
    return mism / total


def off_the_small_step(labels):
    """The same positives among more than 4,096 pairs, which small layers with up to 32 batch rows take the role kernel for: the rest lie
    outside the batch and are ignored."""
    return np.concatenate([labels, np.tile([[-1, 0]], (4097, 1))])


@pytest.mark.parametrize("nc,rows,batch,seed", [
    (1, 64, 16, 11),          # a single tile
    (1, 16, 16, 12),          # a single ragged tile
    (3, 208, 32, 13),         # ragged last tile in every chunk
    (2, 4096, 128, 14),       # one tile per workgroup pair, full batch
    (5, 2000, 64, 15),        # several tiles per pair, ragged
])
def test_rtn_parity_small(gpu, nc, rows, batch, seed):
    case = H.make_case(nc, rows, batch, seed)
    check_rtn(case, gpu)
    if batch <= 32:
        check_rtn(case, gpu, device_labels=off_the_small_step(case["labels"]))


def test_quads_run_on_one_xcd_each(gpu):
    """The four workgroups of a quad exchange G through the L2 of one XCD.  After a step the XCC ids the workgroups
    recorded are read back: every quad's four are equal (the device makes the same comparison at the end of the step
    and raises bit 1 of the error word otherwise), and the error word is clear."""
    import ctypes
    import torch
    from elmo_amd import _lib, ops
    lib = _lib.load()
    case = H.make_case(2, 4096, 32, 17)
    chunks, x, labels = H.to_device_case(case, gpu)
    ws = ops.alloc_workspace(2, 4096, gpu)
    ops.fp8_step(chunks, x, labels, 0.05, round_mode="rtn", workspace=ws)
    n = lib.xmc_step_workgroups()
    assert n >= 32 and n % 32 == 0
    ids = (ctypes.c_int32 * n)()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(lib.xmc_step_xcc_ids(ws.data_ptr(), ids, n, stream), "xmc_step_xcc_ids")
    assert lib.xmc_quad_placement_check(ids, n) == 0, list(ids)
    assert len(set(ids)) == 8 and all(0 <= v < 8 for v in ids)      # eight XCDs, all in use
    assert ops.step_error_word(ws, 2, 4096) == 0
    # the asynchronous form of the error check (what the module does after every step)
    off = lib.xmc_step_error_offset()
    assert int(ws[off:off + 4].view(torch.int32).item()) == 0


def test_rtn_parity_medium_full_batch(gpu):
    case = H.make_case(2, 20000 // 16 * 16, 128, 21, pos_mean=5.4)
    frac = check_rtn(case, gpu)
    print("mismatch fraction", frac)


def test_duplicate_and_dense_positives(gpu):
    # duplicates must count once; one head label positive for every row; two labels of one row in one tile
    extra = [(0, 0), (0, 0), (3, 0), (3, 5), (3, 5), (7, 63), (7, 64), (15, 127)] + [(b, 1) for b in range(16)]
    case = H.make_case(2, 64, 16, 31, extra_labels=extra)
    check_rtn(case, gpu)
    check_rtn(case, gpu, device_labels=off_the_small_step(case["labels"]))


def test_many_positives_boundary_labels_and_ignored_entries(gpu):
    """Close to the 32,768 pairs a step accepts (the launch that groups them by tile then uses its largest LDS
    footprint), with positives on the first and last label, on both sides of the chunk boundary and in every batch
    row; pairs whose row or label lies outside the batch or the label space are ignored."""
    nc, rows, batch = 2, 4096, 128
    L = nc * rows
    rng = np.random.default_rng(77)
    flat = rng.choice(batch * L, size=32000, replace=False)
    valid = np.stack([flat // L, flat % L], axis=1).astype(np.int32)
    edge = np.array([[0, 0], [127, L - 1], [5, rows - 1], [5, rows], [64, rows - 1], [0, L - 1]], dtype=np.int32)
    valid = np.concatenate([valid, edge], axis=0)
    bogus = np.array([[-1, 3], [batch, 3], [255, 3], [1000, 3], [3, -5], [3, L], [3, (1 << 24) - 1], [3, 1 << 30]], dtype=np.int32)
    mixed = np.concatenate([valid, bogus], axis=0)
    mixed = mixed[rng.permutation(len(mixed))]
    case = H.make_case(nc, rows, batch, 78)
    case["labels"] = valid
    check_rtn(case, gpu, device_labels=mixed)


def test_no_positives(gpu):
    case = H.make_case(2, 128, 16, 32)
    case["labels"] = np.zeros((0, 2), dtype=np.int32)
    check_rtn(case, gpu)


def test_scales(gpu):
    # weights stored as w / 2^-4, so most codes sit in the normal range
    case = H.make_case(2, 512, 32, 33, w_scale=2.0 ** -4)
    check_rtn(case, gpu, scale_w=2.0 ** -4, scale_x=0.5)


@pytest.mark.parametrize("wd,p,sw", [(0.05, 0.0, 1.0), (0.0, 0.3, 1.0), (0.02, 0.1, 2.0 ** -4)])
def test_weight_decay_and_fused_dropout(gpu, wd, p, sw):
    """T = c - (lr / s)(A + wd s c) and the dropout of X inside the step, against the oracle (which is pinned by closed
    forms for both).  lr and wd are large enough that the decay term moves a good share of the weights by itself."""
    import torch
    from elmo_amd import ops
    case = H.make_case(3, 1008, 48, 35, w_scale=sw)
    check_rtn(case, gpu, lr=0.5, scale_w=sw, weight_decay=wd, dropout_p=p, dropout_seed=0xABCDEF0123)
    plain = O.fp8_step(case["chunks"], case["x"], case["labels"], 0.5, scale_w=sw)
    extra = O.fp8_step(case["chunks"], case["x"], case["labels"], 0.5, scale_w=sw, weight_decay=wd, dropout_p=p,
                       dropout_seed=0xABCDEF0123)
    assert np.mean(np.concatenate(plain[0]) != np.concatenate(extra[0])) > 0.02      # the options matter on this case
    # the stochastic modes take the same decayed T: the reference's recipe is bit-identical wherever T is
    chunks, x, labels = H.to_device_case(case, gpu)
    seeds = [5, 6, 7]
    ops.fp8_step(chunks, x, labels, 0.5, seeds=seeds, round_mode="sr_philox", scale_w=sw, weight_decay=wd, dropout_p=p,
                 dropout_seed=0xABCDEF0123)
    ref = O.fp8_step(case["chunks"], case["x"], case["labels"], 0.5, seeds=seeds, sr_mode="reference", scale_w=sw,
                     weight_decay=wd, dropout_p=p, dropout_seed=0xABCDEF0123)[0]
    got = H.chunks_to_numpy(chunks)
    d = np.concatenate([H.e4m3_ulp_distance(a, b).ravel() for a, b in zip(got, ref)])
    assert d.max() <= 1 and (d != 0).mean() < 2e-3


def test_x_not_modified_and_deterministic(gpu):
    import torch
    from elmo_amd import ops
    case = H.make_case(2, 1024, 32, 34)
    outs = []
    for _ in range(2):
        chunks, x, labels = H.to_device_case(case, gpu)
        x0 = x.clone()
        g, gf = ops.fp8_step(chunks, x, labels, 0.05, round_mode="rtn", want_f32=True)
        assert torch.equal(x.view(torch.int16), x0.view(torch.int16))
        outs.append(([c.view(torch.uint8).clone() for c in chunks], gf.clone()))
    for a, b in zip(outs[0][0], outs[1][0]):
        assert torch.equal(a, b)
    assert torch.equal(outs[0][1], outs[1][1])      # fixed-order reduction: bitwise reproducible


def test_step_replays_in_a_captured_graph(gpu):
    """The step allocates nothing, never synchronises and clears its counters in a kernel, so a caller may record it
    into a graph.  Three replays, with eager work and synchronisations between them, must give bit for bit what three
    eager steps give (round-to-nearest, fixed-order grad_X)."""
    import torch
    from elmo_amd import ops
    case = H.make_case(2, 4096, 128, 35)
    chunks, x, labels = H.to_device_case(case, gpu)
    start = [c.view(torch.uint8).clone() for c in chunks]
    ws = ops.alloc_workspace(len(chunks), chunks[0].shape[0], gpu)
    gout = torch.empty(128, 768, dtype=torch.bfloat16, device=gpu)
    eager = []
    for _ in range(3):
        ops.fp8_step(chunks, x, labels, 0.05, round_mode="rtn", workspace=ws, grad_out=gout)
        eager.append(([c.view(torch.uint8).clone() for c in chunks], gout.view(torch.int16).clone()))
    for c, s in zip(chunks, start):
        c.view(torch.uint8).copy_(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.fp8_step(chunks, x, labels, 0.05, round_mode="rtn", workspace=ws, grad_out=gout)
    for c, s in zip(chunks, start):      # the capture must not have run anything
        assert torch.equal(c.view(torch.uint8), s)
    for k in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert ops.step_error_word(ws, len(chunks), chunks[0].shape[0]) == 0
        for c, e in zip(chunks, eager[k][0]):
            assert torch.equal(c.view(torch.uint8), e), f"weights differ after replay {k}"
        assert torch.equal(gout.view(torch.int16), eager[k][1]), f"grad_input differs after replay {k}"
        scratch = torch.randn(1 << 20, device=gpu).sum().item()      # unrelated eager work between the replays
        assert scratch == scratch


@pytest.mark.parametrize("nnz", [1, 63, 64, 65, 193, 1025, 4609])
def test_sort_pads_the_positives_to_whole_blocks_only(gpu, nnz):
    """Numbers of positives around whole wavefronts of 64, from which the grouping by tile takes them, in random order and with repetitions, against the oracle."""
    case = H.make_case(2, 1040, 64, 90 + nnz)
    rng = np.random.default_rng(nnz)
    case["labels"] = np.stack([rng.integers(0, 64, nnz), rng.integers(0, 2 * 1040, nnz)], axis=1).astype(np.int32)
    check_rtn(case, gpu)
