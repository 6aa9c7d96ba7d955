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
