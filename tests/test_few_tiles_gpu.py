"""Fused steps of few tiles, which take fewer quads of workgroups than the device holds: against the oracle, in workspaces whose contents
are not read before they are written, and with no workgroup's XCD recorded wrongly."""
import numpy as np
import pytest

import helpers as H
from oracle import step as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [48, 128])
@pytest.mark.parametrize("nc,rows", [(1, 16), (1, 496), (1, 512), (1, 528), (1, 1040), (2, 1024), (1, 2064), (4, 1024), (1, 4112), (8, 1024), (3, 2736)])
def test_step(gpu, nc, rows, batch):
    """1 to 129 tiles, on either side of 8, 16, 32, 64 and 128, where the number of quads or their tiles change."""
    import ctypes
    import torch
    from elmo_amd import _lib, ops
    case = H.make_case(nc, rows, batch, 3 * nc + rows + batch)
    ref_codes, ref_gx, _ = O.fp8_step(case["chunks"], case["x"], case["labels"], 0.05, sr_mode="rtn")
    ws = ops.alloc_workspace(nc, rows, gpu)
    ws[: ops.step_sticky_error_offset()].fill_(0x7F)
    ws[ops.step_sticky_error_offset() + 4:].fill_(0x7F)      # (as fp32 sums: NaN)
    for _ in range(2):
        chunks, x, labels = H.to_device_case(case, gpu)
        _, gf = ops.fp8_step(chunks, x, labels, 0.05, round_mode="rtn", workspace=ws, want_f32=True)
        assert ops.step_error_word(ws, nc, rows) == 0
        for a, b in zip(H.chunks_to_numpy(chunks), ref_codes):
            assert H.e4m3_ulp_distance(a, b).max() <= 1 and np.mean(a == b) > 0.998
        assert np.abs(gf.cpu().numpy() - ref_gx).max() <= 1e-3 * np.abs(ref_gx).max()
    lib = _lib.load()
    n = lib.xmc_step_workgroups()
    ids = (ctypes.c_int32 * n)()
    _lib.check(lib.xmc_step_xcc_ids(ws.data_ptr(), ids, n, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "xmc_step_xcc_ids")
    assert lib.xmc_quad_placement_check(ids, n) == 0


@pytest.mark.parametrize("tiles,batch,mode,decay,quads", [
    (32, 48, "rtn", 0.0, 32), (33, 16, "rtn", 0.0, 40), (64, 16, "sr_fast", 0.0, 64), (65, 16, "rtn", 0.0, 40), (64, 32, "sr_fast", 0.0, 32), (64, 32, "sr_fast", 0.01, 64),
    (57, 48, "rtn", 0.01, 32), (57, 96, "sr_philox", 0.0, 64), (57, 112, "sr_philox", 0.01, 32), (128, 128, "rtn", 0.0, 64), (129, 16, "rtn", 0.0, 64)])
def test_quads(gpu, tiles, batch, mode, decay, quads):
    """How many quads a step of few tiles takes: one for every tile where that is faster (the figures stand beside the rule)."""
    import ctypes
    import torch
    from elmo_amd import _lib, ops
    lib = _lib.load()
    n = lib.xmc_step_workgroups()
    if n != 256:
        pytest.skip("the quads of a whole device")
    case = H.make_case(1, 64 * tiles - 16, batch, tiles + batch, extra_labels=[[-1, 0]] * 4097)     # (more pairs than the small step takes)
    chunks, x, labels = H.to_device_case(case, gpu)
    ws = ops.alloc_workspace(1, 64 * tiles - 16, gpu)
    ops.fp8_step(chunks, x, labels, 0.05, seeds=[3], round_mode=mode, workspace=ws, weight_decay=decay)
    ids = (ctypes.c_int32 * n)()
    _lib.check(lib.xmc_step_xcc_ids(ws.data_ptr(), ids, n, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "xmc_step_xcc_ids")
    assert 8 * sum(v != 0 for v in ids) == 7 * 4 * quads      # (an eighth ran on XCD 0, the others did not run)


@pytest.mark.parametrize("batch", [32, 128])
@pytest.mark.parametrize("nc,rows,head", [(1, 64, 40), (1, 640, 640), (1, 1040, 70), (1, 4160, 4160), (2, 2080, 520), (2, 4160, 4128), (1, 8256, 100), (2, 8256, 8240)])
def test_compensated_head(gpu, nc, rows, head, batch):
    """Heads of 1 to 129 tiles with fewer, as many and more tiles behind them: the second launch continues the sums of the first one's
    quads and of no others'."""
    import torch
    from elmo_amd import ops
    case = H.make_case(nc, rows, batch, 5 * nc + rows + head + batch)
    rng = np.random.default_rng(head)
    k0 = torch.from_numpy(rng.normal(size=(head, 768)).astype(np.float32) * 2.0 ** -10).to(torch.bfloat16)
    ref_codes, ref_k, ref_gx, _ = O.fp8_kahan_step(case["chunks"], k0.float().numpy(), case["x"], case["labels"], 0.05, head, kahan_type="bf16", sr_mode="rtn")
    ws = ops.alloc_workspace(nc, rows, gpu, 128)
    ws[: ops.step_sticky_error_offset()].fill_(0x7F)
    ws[ops.step_sticky_error_offset() + 4:].fill_(0x7F)
    chunks, x, labels = H.to_device_case(case, gpu)
    terms = k0.to(gpu)
    _, gf = ops.fp8_kahan_step(chunks, terms, head, x, labels, 0.05, round_mode="rtn", workspace=ws, want_f32=True)
    assert ops.step_error_word(ws, nc, rows) == 0
    for a, b in zip(H.chunks_to_numpy(chunks), ref_codes):
        assert H.e4m3_ulp_distance(a, b).max() <= 1 and np.mean(a == b) > 0.998
    assert np.mean(terms.float().cpu().numpy() == ref_k) > 0.99      # (a term turns over with its weight)
    assert np.abs(gf.cpu().numpy() - ref_gx).max() <= 1e-3 * np.abs(ref_gx).max()


@pytest.mark.parametrize("mode", ["rtn", "sr_philox"])
@pytest.mark.parametrize("weights", ["bf16", "e4m3", "fp8"])
@pytest.mark.parametrize("batch,labels", [
    (20, 4600), (20, 4630), (20, 8192), (64, 2560), (64, 2570), (64, 8192),      # clusters of one
    (100, 1504), (100, 1530), (100, 3072), (100, 4096), (100, 4128),             # of two
    (200, 990), (200, 1024), (200, 1536), (200, 2048), (200, 4096)])             # of four
@pytest.mark.parametrize("nc", [1, 3])
def test_one_pass_step_with_half_the_clusters(gpu, nc, batch, labels, weights, mode):
    """Either side of the lines from which on a cluster takes two tiles, against the same layer with chunks that go on in rows of zeros, whose
    tiles are more than the clusters there are.  A row's update depends on no other row, so the weights agree to the bit.  Rows of zeros add
    nothing to grad_X: the same fp32 sum in another grouping (2^-16 of its largest value); with bf16 weights the sum of a chunk is
    rounded to bf16 by itself, where a neighbour may come out: 2^-8 of it, and the largest of three sums that partly cancel is taken to
    be at most four times the largest of their total."""
    import torch
    from elmo_amd import ops
    rows = labels // nc // 16 * 16
    more = 9600 // nc // 16 * 16
    g = torch.Generator(device=gpu).manual_seed(batch + labels)
    dtype = torch.bfloat16 if weights == "bf16" else torch.float8_e4m3fn
    chunks = [torch.randn(rows, 768, generator=g, device=gpu).mul_(0.05).to(dtype) for _ in range(nc)]
    others = [torch.cat([c.float(), torch.zeros(more - rows, 768, device=gpu)]).to(dtype) for c in chunks]
    x = torch.randn(batch, 768, generator=g, device=gpu).to(torch.bfloat16)
    pos = torch.stack([torch.arange(5 * batch, device=gpu) % batch, torch.randint(0, nc * rows, (5 * batch,), generator=g, device=gpu)], 1).to(torch.int32)
    pos_others = torch.stack([pos[:, 0], pos[:, 1] // rows * more + pos[:, 1] % rows], 1).contiguous()
    kind, fp8 = "bf16" if weights == "bf16" else "e4m3", weights == "fp8"
    out = []
    for w, n, labs in ((chunks, rows, pos), (others, more, pos_others)):
        ws = ops.alloc_tiled_workspace(nc, n, gpu, batch)
        off = ops.tiled_error_offset()
        ws[off + 8:].fill_(0x7F)
        out.append(ops.tiled_step(w, n, kind, x, labs, 0.05, seeds=[3 + c for c in range(nc)], round_mode=mode, workspace=ws, want_f32=True,
                                  quantize_x=fp8, saturate=fp8)[1])
        assert int(ws[off:off + 4].view(torch.int32).item()) == 0
    for a, b in zip(chunks, others):
        assert torch.equal(a.view(torch.uint8), b[:rows].view(torch.uint8))
    tol = (2 ** -16 if weights != "bf16" else 4 * nc * 2 ** -8) * out[1].abs().max().item()
    assert (out[0] - out[1]).abs().max().item() <= tol
