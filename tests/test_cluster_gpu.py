"""The one-pass step (bf16 weights, simulated FP8, true FP8 above 128 batch rows) at the sizes where its split changes: the
cluster sizes' batch limits, partial tiles and chunks, fewer tiles than clusters, chunk boundaries within a cluster's range.
Oracle and tolerances as in test_tiled_gpu.py."""
import numpy as np
import pytest

import helpers as H
from oracle import codecs as C
from oracle import step as O
from test_tiled_gpu import bf16_case, check_bf16_weights, check_gx, run_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,nc,rows,batch,mode", [
    ("bf16", 1, 1, 1, "rtn"),                # one label, one row: a cluster of one, 32 batch rows
    ("bf16", 3, 33, 32, "sr_philox"),        # chunks of one tile and a row
    ("bf16", 2, 31, 33, "sr_fast"),          # 64 batch rows
    ("bf16", 40, 320, 64, "rtn"),            # more tiles than clusters, several chunks to a cluster
    ("bf16", 1, 65, 65, "sr_fast"),          # clusters of two, fewer tiles than clusters
    ("bf16", 3, 4100, 128, "sr_philox"),
    ("bf16", 2, 545, 129, "rtn"),            # clusters of four
    ("bf16", 60, 96, 257, "sr_philox"),      # clusters of eight, a chunk boundary at every third tile
    ("bf16", 2, 2000, 511, "sr_fast"),
    ("sim", 2, 48, 32, "sr_philox"),
    ("sim", 3, 4112, 64, "rtn"),
    ("sim", 2, 2064, 100, "sr_philox"),
    ("sim", 2, 1040, 250, "rtn"),
    ("sim", 1, 16, 512, "sr_philox"),
    ("fp8", 7, 208, 96, "sr_fast"),          # clusters of two, tiles of 64 rows
    ("fp8", 1, 16, 144, "rtn"),              # clusters of four, a single partial tile
    ("fp8", 3, 3088, 256, "sr_philox"),
    ("fp8", 2, 1040, 272, "sr_fast"),        # clusters of eight, tiles of 32 rows
    ("fp8", 5, 848, 512, "rtn"),
])
def test_one_pass_step_matches_the_oracle(gpu, kind, nc, rows, batch, mode):
    from elmo_amd import ops
    seeds = None if mode == "rtn" else [77 + 31 * c for c in range(nc)]
    L = nc * rows - (nc - 1 if kind == "bf16" else 0)      # bf16: the last chunk is shorter
    edges = np.array([[batch - 1, L - 1], [0, 0], [0, 0], [batch // 2, min(rows, L - 1)], [batch // 2, rows - 1]], np.int32)
    if kind == "bf16":
        x, w, labels = bf16_case(L, batch, 500 + batch)
        labels = np.concatenate([edges, labels])
        new, gf, gb = run_bf16(x, w, labels, nc, gpu, mode, seeds)
        sr = {"rtn": "rtn", "sr_philox": "reference", "sr_fast": "fast"}[mode]
        ref_w, ref_gx, _ = O.bf16_step(w, x, labels, 0.05, nc, seeds=seeds, sr_mode=sr)
        check_bf16_weights(new, ref_w, w, x)
        check_gx(gf, gb, ref_gx, tol=4e-3)
        return
    case = H.make_case(nc, rows, batch, 500 + batch, extra_labels=edges.tolist())
    chunks, x, labels = H.to_device_case(case, gpu)
    true_fp8 = kind == "fp8"
    g, gf = ops.tiled_step(chunks, rows, "e4m3", x, labels, 0.05, seeds=seeds, round_mode=mode, want_f32=True,
                           quantize_x=true_fp8, saturate=true_fp8)

    def rand_fn(c, offs):
        return C.fast_sr_words(seeds[c], c * rows + offs // 768, offs % 768)

    kw = dict(sr_mode="exact", rand_fn=rand_fn) if mode == "sr_fast" else dict(sr_mode="rtn" if mode == "rtn" else "reference", seeds=seeds)
    ref_codes, ref_gx, _ = O.fp8_step(case["chunks"], case["x"], case["labels"], 0.05, simulated=not true_fp8, **kw)
    dist = np.concatenate([H.e4m3_ulp_distance(a, b).ravel() for a, b in zip(H.chunks_to_numpy(chunks), ref_codes)])
    assert dist.max() <= 1 and (dist != 0).mean() < 5e-3, (dist.max(), (dist != 0).mean())
    check_gx(gf.cpu().numpy(), g.float().cpu().numpy(), ref_gx)


@pytest.mark.parametrize("nc,rows,batch,mode", [
    (1, 16, 16, "sr_fast"),                  # one partial tile, 32-row slices
    (3, 80, 32, "sr_philox"),                # a tile and a quarter to a chunk
    (5, 4112, 33, "rtn"),                    # 64-row slices, more tiles than clusters
    (2, 9232, 64, "sr_philox"),              # one to three tiles to a cluster
    (2, 16400, 24, "sr_fast"),
])
def test_one_pass_step_with_fp8_logits_in_clusters_of_one(gpu, nc, rows, batch, mode):
    test_one_pass_step_matches_the_oracle(gpu, "fp8", nc, rows, batch, mode)


@pytest.mark.parametrize("nc,tiles,batch,mode,dropout", [
    (1, 384, 16, "sr_fast", 0.0),            # the first size that takes the one-pass form (256 compute units), 32-row slices
    (3, 128, 32, "rtn", 0.3),                # the same, a partial tile at the end of every chunk
    (2, 512, 32, "sr_philox", 0.0),
    (4, 256, 48, "sr_fast", 0.3),            # 64-row slices
    (4, 256, 64, "rtn", 0.0),
    (3, 1024, 64, "sr_philox", 0.0),
])
def test_small_batches_take_the_one_pass_form_with_the_same_results(gpu, nc, tiles, batch, mode, dropout):
    """xmc_fp8_step on both of its forms: a batch of at most 64 rows, and the same batch with rows of zeros up to 80, which
    takes the fused kernel.  The added rows contribute exact zeros, so the weights
    agree to the bit."""
    import torch
    from elmo_amd import ops
    rows = 64 * tiles - 48
    seeds = None if mode == "rtn" else [5 + 3 * c for c in range(nc)]
    g = torch.Generator(device=gpu).manual_seed(900 + batch)
    chunks = [torch.randn(rows, 768, generator=g, device=gpu).mul_(0.05).to(torch.float8_e4m3fn) for _ in range(nc)]
    padded = [c.clone() for c in chunks]
    x = torch.randn(batch, 768, generator=g, device=gpu).to(torch.bfloat16)
    x80 = torch.cat([x, torch.zeros(80 - batch, 768, dtype=torch.bfloat16, device=gpu)])
    n = 9 * batch
    labels = torch.stack([torch.arange(n, device=gpu) % batch, torch.randint(0, nc * rows, (n,), generator=g, device=gpu)], 1)
    edges = [[batch - 1, nc * rows - 1], [0, 0], [0, 0], [0, rows - 1], [-1, 3], [0, nc * rows]]        # (the last two are ignored)
    labels = torch.cat([labels, torch.tensor(edges, device=gpu)]).to(torch.int32).contiguous()
    ws = ops.alloc_workspace(nc, rows, gpu)
    off = ops.step_sticky_error_offset()
    for _ in range(2):                       # (the second step on what the first left in the workspace)
        g1, f1 = ops.fp8_step(chunks, x, labels, 0.05, seeds=seeds, round_mode=mode, workspace=ws, want_f32=True, dropout_p=dropout, dropout_seed=7)
        g2, f2 = ops.fp8_step(padded, x80, labels, 0.05, seeds=seeds, round_mode=mode, workspace=ws, want_f32=True, dropout_p=dropout, dropout_seed=7)
        for a, b in zip(chunks, padded):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
        # two groupings of one fp32 sum (of at most 256 partial sums behind one another): 2^8 roundings of 2^-24 at most
        tol = 2 ** -16 * f2[:batch].abs().max().item()
        assert (f1 - f2[:batch]).abs().max().item() <= tol and torch.allclose(g1.float(), g2[:batch].float(), rtol=2 ** -7, atol=tol)
        assert ops.step_error_word(ws, nc, rows) == 0 and int(ws[off:off + 4].view(torch.int32).item()) == 0


def test_fp8_step_in_the_one_pass_form_records_the_xcds_too(gpu):
    """xmc_step_xcc_ids reads the ids of the last step, whichever form it took: here one in clusters of one, in a workspace whose
    previous ids are no XCDs."""
    import ctypes
    import torch
    from elmo_amd import _lib, ops
    lib = _lib.load()
    nc, rows = 1, 64 * 512
    ws = ops.alloc_workspace(nc, rows, gpu)
    ws.fill_(0x55)
    off = ops.step_sticky_error_offset()
    ws[off:off + 4].zero_()
    w = torch.zeros(rows, 768, device=gpu).to(torch.float8_e4m3fn)
    ops.fp8_step([w], torch.zeros(16, 768, dtype=torch.bfloat16, device=gpu), torch.zeros(0, 2, dtype=torch.int32, device=gpu), 0.05,
                 workspace=ws)
    n = lib.xmc_step_workgroups()
    ids = (ctypes.c_int32 * n)()
    _lib.check(lib.xmc_step_xcc_ids(ws.data_ptr(), ids, n, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "xmc_step_xcc_ids")
    assert len(set(ids)) == 8 and all(0 <= v < 8 for v in ids), list(ids)


def test_one_pass_step_gives_up_cleanly(gpu):
    """A polling limit of 0, set from the host: the second member leaves after three tiles, and its partners' waits expire.  Every kernel
    ends, the error words say so, no weight is updated from missing data, the layer raises, and the next step is clean."""
    import torch
    from elmo_amd import ops
    from test_host_cpu import make_cfg
    from xmc_classifiers.chunked_fp8xmc_clf import Fp8XMCBCEChunkedLayer
    nc, rows, batch = 2, 8192, 256
    cfg = make_cfg("cuda:0", nc * rows - 16, nc, rounding="rtn")
    cfg.data.batch_size = batch
    xfc = Fp8XMCBCEChunkedLayer(cfg)
    assert xfc.xfc_weight[0].shape[0] == rows
    case = H.make_case(nc, rows, batch, 611)
    chunks, x, labels = H.to_device_case(case, gpu)
    ref_codes, _, _ = O.fp8_step(case["chunks"], case["x"], case["labels"], 0.05, sr_mode="rtn")
    prev = ops.debug_spin_limit(0)
    try:
        for wt, c in zip(xfc.xfc_weight, chunks):
            wt.data.copy_(c.view(torch.float8_e4m3fn))
        with pytest.raises(RuntimeError, match="gave up waiting"):
            xfc.xfc_forward_backward(x, labels, [0.05])
            xfc.check_steps()
        assert xfc.last_step_error() == 1
        for wt, old, ref in zip(xfc.xfc_weight, case["chunks"], ref_codes):
            new = wt.data.view(torch.uint8).cpu().numpy()
            # the unit of the update is a member's quarter of the features of a row
            same_old = (new == old).reshape(-1, 4, 192).all(axis=2)
            good = (H.e4m3_ulp_distance(new, ref) <= 1).reshape(-1, 4, 192).all(axis=2)
            assert np.all(same_old | good), "weights were updated from incomplete data"
    finally:
        ops.debug_spin_limit(prev)
    xfc.xfc_forward_backward(x, labels, [0.05])
    xfc.check_steps()
    assert xfc.last_step_error() == 0
