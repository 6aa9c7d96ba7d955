"""The three-kernel form of the tiled step at 768 features.  Loss, weight decay and a compensated head take it, plain steps
do not (they run as one kernel: test_cluster_gpu.py and most of test_tiled_gpu.py); weight decay selects it here.  Cases at the
edges of its split: batch halves, tiles, chunks that share launches, the feature-split update (e4m3, two halves) and the FP8
logits (more than 128 rows).  Oracle and tolerances as in test_tiled_gpu.py."""
import numpy as np
import pytest

import helpers as H
from oracle import codecs as C
from oracle import step as O
from test_other_workloads_fullsize_gpu import check_sampled_rows, sample_rows, snapshot
from test_tiled_gpu import bf16_case, check_bf16_weights, check_gx

pytestmark = pytest.mark.gpu

DECAY = 0.02


def bf16_views(w, nc, device):
    import torch
    wt = torch.from_numpy(C.bf16_bits(w).view(np.int16)).to(device).view(torch.bfloat16)
    return wt, wt.split((w.shape[0] + nc - 1) // nc)


@pytest.mark.parametrize("kind,nc,rows,batch,mode", [
    ("bf16", 1, 1, 1, "rtn"),
    ("bf16", 3, 33, 32, "sr_philox"),        # chunks of one tile and a row, one per launch
    ("bf16", 10, 1024, 16, "sr_philox"),     # launches of eight chunks and two
    ("bf16", 4, 1024, 128, "sr_fast"),
    ("bf16", 2, 1024, 200, "sr_philox"),     # two halves, the second one short
    ("bf16", 2, 545, 256, "rtn"),
    ("bf16", 3, 700, 300, "sr_fast"),        # three halves, run as four
    ("bf16", 2, 1000, 512, "rtn"),
    ("sim", 3, 208, 32, "sr_philox"),
    ("sim", 2, 2064, 128, "rtn"),
    ("sim", 2, 1040, 250, "sr_philox"),      # feature-split update
    ("sim", 1, 16, 512, "sr_philox"),
    ("fp8", 7, 208, 96, "sr_fast"),
    ("fp8", 1, 16, 144, "rtn"),              # FP8 logits, feature-split update, a single partial tile
    ("fp8", 3, 3088, 256, "sr_philox"),
    ("fp8", 2, 1040, 272, "sr_fast"),
    ("fp8", 5, 848, 512, "rtn"),
    # batches that end in front of, at and behind a K step of 32 rows, and whose last halves have no rows
    ("bf16", 2, 300, 33, "sr_philox"),
    ("bf16", 2, 300, 65, "rtn"),
    ("bf16", 1, 300, 385, "rtn"),
    ("sim", 1, 304, 64, "sr_philox"),
    ("sim", 1, 304, 97, "rtn"),
    ("fp8", 1, 304, 257, "rtn"),
    ("fp8", 2, 304, 416, "sr_fast"),
])
def test_step_with_weight_decay_matches_the_oracle(gpu, kind, nc, rows, batch, mode):
    import torch
    from elmo_amd import ops
    seeds = None if mode == "rtn" else [77 + 31 * c for c in range(nc)]
    L = nc * rows - (nc - 1 if kind == "bf16" else 0)      # bf16: the last chunk is shorter
    edges = np.array([[batch - 1, L - 1], [0, 0], [0, 0], [batch // 2, min(rows, L - 1)], [batch // 2, rows - 1]], np.int32)
    opts = dict(seeds=seeds, round_mode=mode, want_f32=True, weight_decay=DECAY)
    if kind == "bf16":
        x, w, labels = bf16_case(L, batch, 500 + batch)
        labels = np.concatenate([edges, labels])
        wt, views = bf16_views(w, nc, gpu)
        xt = torch.from_numpy(C.bf16_bits(x).view(np.int16)).to(gpu).view(torch.bfloat16)
        g, gf = ops.tiled_step(views, views[0].shape[0], "bf16", xt, torch.from_numpy(labels).to(gpu), 0.5, **opts)
        sr = {"rtn": "rtn", "sr_philox": "reference", "sr_fast": "fast"}[mode]
        ref_w, ref_gx, _ = O.bf16_step(w, x, labels, 0.5, nc, seeds=seeds, sr_mode=sr, weight_decay=DECAY)
        check_bf16_weights(wt.float().cpu().numpy(), ref_w, w, x, lr=0.5)
        check_gx(gf.cpu().numpy(), g.float().cpu().numpy(), ref_gx, tol=4e-3)
        return
    case = H.make_case(nc, rows, batch, 500 + batch, extra_labels=edges.tolist())
    chunks, x, labels = H.to_device_case(case, gpu)
    true_fp8 = kind == "fp8"
    g, gf = ops.tiled_step(chunks, rows, "e4m3", x, labels, 0.5, quantize_x=true_fp8, saturate=true_fp8, **opts)

    def rand_fn(c, offs):
        return C.fast_sr_words(seeds[c], c * rows + offs // 768, offs % 768)

    kw = dict(sr_mode="exact", rand_fn=rand_fn) if mode == "sr_fast" else dict(sr_mode="rtn" if mode == "rtn" else "reference", seeds=seeds)
    ref_codes, ref_gx, _ = O.fp8_step(case["chunks"], case["x"], case["labels"], 0.5, simulated=not true_fp8, weight_decay=DECAY, **kw)
    dist = np.concatenate([H.e4m3_ulp_distance(a, b).ravel() for a, b in zip(H.chunks_to_numpy(chunks), ref_codes)])
    assert dist.max() <= 1 and (dist != 0).mean() < 5e-3, (dist.max(), (dist != 0).mean())
    check_gx(gf.cpu().numpy(), g.float().cpu().numpy(), ref_gx)


@pytest.mark.parametrize("kind", ["bf16", "sim", "fp8"])
@pytest.mark.parametrize("batch", [1, 32, 33, 64, 65, 129, 161, 257, 300, 385])
def test_nothing_is_read_of_rows_that_the_batch_does_not_have(gpu, kind, batch):
    """G of K steps without batch rows is not written: a workspace full of NaN gives bit for bit what one of zeros gives."""
    import torch
    from elmo_amd import ops
    rows, d = 400, 1024
    gen = torch.Generator(device=gpu).manual_seed(batch)
    w0 = torch.randn(rows, d, generator=gen, device=gpu) * 0.02
    x = torch.randn(batch, d, generator=gen, device=gpu).to(torch.bfloat16)
    labels = torch.tensor([[0, 0], [batch - 1, rows - 1]], dtype=torch.int32, device=gpu)
    out = []
    for fill in (0, 255):
        w = w0.to(torch.bfloat16 if kind == "bf16" else torch.float8_e4m3fn)
        ws = torch.full((ops.tiled_workspace_bytes(1, rows, batch, d),), fill, dtype=torch.uint8, device=gpu)
        g = ops.tiled_step([w], rows, "bf16" if kind == "bf16" else "e4m3", x, labels, 0.1, workspace=ws, quantize_x=kind == "fp8", saturate=kind == "fp8")
        out.append((w.view(torch.uint8), g))
    assert torch.isfinite(out[1][1].float()).all()
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


@pytest.mark.parametrize("kind", ["bf16", "sim"])
@pytest.mark.parametrize("batch", [16, 33, 257, 300])
def test_a_loss_writes_no_more_than_its_shares(gpu, kind, batch):
    """Rows that the batch does not have, whole halves among them, are left out with a loss as without: beyond its two shares a tile
    it touches nothing of the workspace that the step without one leaves alone."""
    import torch
    from elmo_amd import ops
    rows, d, tiles = 400, 1024, 7
    gen = torch.Generator(device=gpu).manual_seed(batch)
    w0 = (torch.randn(rows, d, generator=gen, device=gpu) * 0.02).to(torch.bfloat16 if kind == "bf16" else torch.float8_e4m3fn)
    x = torch.randn(batch, d, generator=gen, device=gpu).to(torch.bfloat16)
    labels = torch.tensor([[0, 0], [batch - 1, rows - 1], [batch // 2, 200]], dtype=torch.int32, device=gpu)
    loss, out = torch.zeros(1, device=gpu), []
    for loss_out in (None, loss):
        w = w0.clone()
        ws = torch.full((ops.tiled_workspace_bytes(1, rows, batch, d),), 255, dtype=torch.uint8, device=gpu)
        g = ops.tiled_step([w], rows, "bf16" if kind == "bf16" else "e4m3", x, labels, 0.1, workspace=ws, loss_out=loss_out)
        out.append((w.view(torch.uint8), g, ws != 255))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
    assert int((out[1][2] & ~out[0][2]).sum()) <= 2 * tiles * 4
    z = (x.float() @ w0.float().t()).to(torch.bfloat16).double()
    ref = z.clamp(min=0).sum() - z[labels[:, 0].long(), labels[:, 1].long()].sum() + torch.log1p(torch.exp(-z.abs())).sum()
    assert abs(loss.item() - ref.item()) <= 1e-4 * abs(ref.item())      # (as in test_loss_over_four_halves)


def test_loss_over_four_halves(gpu):
    """Ragged chunks and a batch that ends inside the third half: rows that pad either do not count."""
    import torch
    from elmo_amd import ops
    L, nc, batch = 1300, 3, 300
    x, w, labels = bf16_case(L, batch, 44)
    wt, views = bf16_views(w, nc, gpu)
    xt = torch.from_numpy(C.bf16_bits(x).view(np.int16)).to(gpu).view(torch.bfloat16)
    loss = torch.zeros(1, dtype=torch.float32, device=gpu)
    ops.tiled_step(views, views[0].shape[0], "bf16", xt, torch.from_numpy(labels).to(gpu), 0.05, loss_out=loss)
    ref_w, _, _, ref_loss = O.bf16_step(w, x, labels, 0.05, nc, sr_mode="rtn", return_loss=True)
    assert abs(loss.item() - ref_loss) <= 1e-4 * abs(ref_loss), (loss.item(), ref_loss)
    check_bf16_weights(wt.float().cpu().numpy(), ref_w, w, x)


def test_replays_of_a_captured_step_with_weight_decay(gpu):
    """Kernels only (no memset, no allocation, no synchronisation): three replays, with eager work between them, give bit for
    bit what three eager steps give."""
    import torch
    from elmo_amd import ops
    x, w, labels = bf16_case(3000, 200, 36)
    wt, views = bf16_views(w, 2, gpu)
    start = wt.clone()
    xt = torch.from_numpy(C.bf16_bits(x).view(np.int16)).to(gpu).view(torch.bfloat16)
    lab = torch.from_numpy(labels).to(gpu).contiguous()
    ws = ops.alloc_tiled_workspace(2, 1500, gpu, 200)
    gout = torch.empty(200, 768, dtype=torch.bfloat16, device=gpu)

    def step():
        ops.tiled_step(views, 1500, "bf16", xt, lab, 0.05, workspace=ws, grad_out=gout, weight_decay=DECAY)

    eager = []
    for _ in range(3):
        step()
        eager.append((wt.view(torch.int16).clone(), gout.view(torch.int16).clone()))
    wt.copy_(start)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for k in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(wt.view(torch.int16), eager[k][0]) and torch.equal(gout.view(torch.int16), eager[k][1]), k
        scratch = torch.randn(1 << 20, device=gpu).sum().item()      # unrelated eager work between the replays
        assert scratch == scratch


def test_label_space_above_2_24_with_weight_decay(gpu):
    """The positives are taken in two segments of the label space (63 chunks + 1): positives and sampled rows on both sides of
    the segment boundary, at label 2^24 and at the end."""
    import torch
    from elmo_amd import ops
    from elmo_amd import synth
    nc, rows, batch = 64, 262272, 32
    L = nc * rows
    gen = torch.Generator(device=gpu).manual_seed(9)
    chunks = [(torch.randn(rows, 768, generator=gen, device=gpu) * 0.02).to(torch.float8_e4m3fn) for _ in range(nc)]
    x_np = synth.make_x(batch, 768, 9)
    special = np.array([(0, 63 * rows - 1), (1, 63 * rows), (2, (1 << 24) - 1), (3, 1 << 24), (5, L - 1), (7, 62 * rows + 5)], np.int32)
    labels_np = np.concatenate([synth.make_labels(batch, L, 6.0, 1.0, 9), special]).astype(np.int32)
    sample = np.unique(np.concatenate([sample_rows(labels_np, nc, rows, 4), special[:, 1], np.arange(63 * rows - 70, 63 * rows + 70)]))
    before = snapshot(chunks, rows, sample)
    ops.tiled_step(chunks, rows, "e4m3", torch.from_numpy(x_np).to(gpu).to(torch.bfloat16), torch.from_numpy(labels_np).to(gpu), 0.5,
                   quantize_x=True, saturate=True, weight_decay=DECAY)
    check_sampled_rows(chunks, rows, sample, before, x_np, labels_np, 0.5, weight_decay=DECAY)
    del chunks
    torch.cuda.empty_cache()
