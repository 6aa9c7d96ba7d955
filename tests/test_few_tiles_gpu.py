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
