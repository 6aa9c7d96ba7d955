"""The update kernel of the three-kernel form walks streams of tiles.  Here a stream takes a second tile and the last tile is partial: the
loads of the next tile, the seed and chunk that change inside a stream, and the end of a compensated head in a stream's later tile.
Oracle and tolerances as in test_three_kernel_gpu.py and test_tiled_width_1024_gpu.py."""
import numpy as np
import pytest

import helpers as H
import test_three_kernel_gpu as K
from elmo_amd import _lib
from oracle import codecs as C
from oracle import step as O
from test_tiled_gpu import check_bf16_weights, check_gx
from test_tiled_width_1024_gpu import FEATS, bf16_case, code_mismatch, run_bf16

pytestmark = pytest.mark.gpu


def check_second_tile(features, batch, rows, device):
    """Some stream of a launch over `rows` label rows takes a second tile (pair of tiles), on this device."""
    import torch
    tiles = (rows + 63) // 64
    streams = _lib.load().xmc_tiled_update_streams(torch.cuda.get_device_properties(device).multi_processor_count, features, batch, tiles)
    units = tiles if batch <= 128 else (tiles + 1) // 2
    assert units > streams, (tiles, streams)


@pytest.mark.parametrize("kind,nc,rows,batch,mode", [
    ("bf16", 8, 1728, 20, "sr_philox"),      # chunks that share a launch: streams cross from one to another
    ("bf16", 1, 13100, 64, "sr_philox"),
    ("bf16", 8, 1664, 128, "sr_fast"),
    ("bf16", 8, 1152, 130, "sr_philox"),
    ("bf16", 5, 1792, 300, "sr_philox"),
    ("sim", 1, 13104, 128, "sr_philox"),
    ("sim", 1, 8976, 300, "sr_philox"),
    ("fp8", 1, 13104, 32, "sr_fast"),
    ("fp8", 1, 8976, 272, "rtn"),
    ("fp8", 1, 8976, 400, "sr_fast"),
])
def test_768_features(gpu, kind, nc, rows, batch, mode):
    check_second_tile(768, batch, nc * rows - (nc - 1), gpu)
    K.test_step_with_weight_decay_matches_the_oracle(gpu, kind, nc, rows, batch, mode)


@pytest.mark.parametrize("L,nc,batch,mode", [
    (7161, 8, 30, "sr_philox"),              # (chunks of 896 rows)
    (6500, 1, 64, "sr_fast"),
    (6500, 1, 128, "rtn"),
    (4602, 4, 200, "sr_philox"),             # (1,152)
    (2500, 1, 500, "sr_fast"),
    (2555, 5, 300, "sr_philox"),             # (512)
])
def test_bf16_weights_1024_features(gpu, L, nc, batch, mode):
    check_second_tile(FEATS, batch, L, gpu)
    x, w, labels = bf16_case(L, batch, 300 + batch)
    seeds = None if mode == "rtn" else [91 + 13 * c for c in range(nc)]
    new, gf, gb = run_bf16(x, w, labels, nc, gpu, mode, seeds)
    ref_w, ref_gx, _ = O.bf16_step(w, x, labels, 0.05, nc, seeds=seeds, sr_mode={"rtn": "rtn", "sr_philox": "reference", "sr_fast": "fast"}[mode])
    check_bf16_weights(new, ref_w, w, x)
    check_gx(gf, gb, ref_gx, tol=4e-3)


@pytest.mark.parametrize("batch,rows", [(32, 6512), (128, 6512), (256, 4560), (400, 2512)])
@pytest.mark.parametrize("true_fp8", [False, True])
def test_e4m3_weights_1024_features(gpu, batch, rows, true_fp8):
    from elmo_amd import ops
    check_second_tile(FEATS, batch, rows, gpu)
    case = H.make_case(1, rows, batch, 400 + batch, features=FEATS)
    chunks, x, labels = H.to_device_case(case, gpu)
    seeds = [515151]
    g, gf = ops.tiled_step(chunks, rows, "e4m3", x, labels, 0.05, seeds=seeds, round_mode="sr_philox", want_f32=True, quantize_x=true_fp8, saturate=true_fp8)
    ref_codes, ref_gx, _ = O.fp8_step(case["chunks"], case["x"], case["labels"], 0.05, seeds=seeds, sr_mode="reference", simulated=not true_fp8)
    assert code_mismatch(H.chunks_to_numpy(chunks), ref_codes) < 2e-3
    check_gx(gf.cpu().numpy(), g.float().cpu().numpy(), ref_gx)


@pytest.mark.parametrize("features,batch,rows,head", [(768, 24, 13104, 12500), (768, 260, 8976, 8700), (768, 200, 8976, 8700),
                                                      (1024, 128, 6512, 6300), (1024, 200, 4560, 4300), (1024, 300, 2512, 2300)])
def test_compensated_head_that_ends_in_a_later_tile(gpu, features, batch, rows, head):
    import torch
    from elmo_amd import ops
    check_second_tile(features, batch, head, gpu)
    case = H.make_case(1, rows, batch, 181 + batch, features=features)
    k0 = C.bf16_round(np.random.default_rng(2).standard_normal((head, features)).astype(np.float32) * 1e-3)
    chunks, x, labels = H.to_device_case(case, gpu)
    kt = torch.from_numpy(C.bf16_bits(k0).view(np.int16)).to(gpu).view(torch.bfloat16)
    g, gf = ops.tiled_step(chunks, rows, "e4m3", x, labels, 0.05, seeds=[77], round_mode="sr_philox", want_f32=True, quantize_x=True, saturate=True,
                           kahan=kt, num_head=head)
    ref_codes, ref_k, ref_gx, _ = O.fp8_kahan_step(case["chunks"], k0, case["x"], case["labels"], 0.05, head, kahan_type="bf16", seeds=[77], sr_mode="reference")
    new = H.chunks_to_numpy(chunks)
    assert code_mismatch(new, ref_codes) < 4e-3
    check_gx(gf.cpu().numpy(), g.float().cpu().numpy(), ref_gx)
    tot_g = C.e4m3_decode(new[0][:head]).astype(np.float64) + kt.float().cpu().numpy()
    tot_r = C.e4m3_decode(ref_codes[0][:head]).astype(np.float64) + ref_k
    assert np.abs(tot_g - tot_r).max() <= 2.0 ** -6 * np.abs(ref_k).max() + 2.0 ** -16


@pytest.mark.parametrize("features,batch", [(768, 40), (768, 300), (1024, 200)])
@pytest.mark.parametrize("last", [1, 70, 640])
def test_short_last_chunk_of_a_launch(gpu, features, batch, last):
    """Chunks that lie one behind the other share a launch and its ranges of grad_X, of which a short last chunk has fewer than the
    others: the same step with a launch for every chunk gives the same weights, and grad_X up to a chunk's bf16 rounding."""
    import torch
    from elmo_amd import ops
    rows, nc = 1024, 4
    gen = torch.Generator(device=gpu).manual_seed(last + batch)
    w0 = (torch.randn(rows * (nc - 1) + last, features, generator=gen, device=gpu) * 0.02).to(torch.bfloat16)
    x = torch.randn(batch, features, generator=gen, device=gpu).to(torch.bfloat16)
    labels = torch.tensor([[0, 0], [batch - 1, w0.shape[0] - 1], [batch // 2, rows]], dtype=torch.int32, device=gpu)
    out = []
    for together in (True, False):
        w = w0.clone()
        views = w.split(rows) if together else [v.clone() for v in reversed(w.split(rows))][::-1]
        g, gf = ops.tiled_step(views, rows, "bf16", x, labels, 0.1, weight_decay=0.02, want_f32=True)
        out.append((torch.cat([v.view(torch.int16) for v in views]), gf))
    assert torch.equal(out[0][0], out[1][0])
    # each of the four chunks' sums is rounded to bf16; another order of its fp32 sum moves a sum near a tie by one unit, 2^-8 of it
    assert (out[0][1] - out[1][1]).abs().max() <= nc * 2.0 ** -8 * out[1][1].abs().max()
    # and few are near one: the sums differ by some 2^-20 of their terms' sum, a tie comes every 2^-8 of the value
    assert (out[0][1] != out[1][1]).float().mean() < 0.05
