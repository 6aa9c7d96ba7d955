"""Rows of the two-pass top-k whose candidate list overflows are done over on the device, by workgroups that share the groups of 32
rows with such a row: one group or several, slices of the labels that are ragged, ties at the k-th value within a slice and over several,
values and ids as the general path gives them."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,rows_done_over", [(1, "all"), (40, "last"), (128, "one"), (128, "two groups"), (97, "three groups"), (128, "all"),
                                                  (129, "last"), (256, "one"), (250, "five groups"), (256, "all")])
@pytest.mark.parametrize("nc,rows,drop,k,ties", [(1, 20016, 0, 1, 3000), (2, 10000, 7, 64, 19000), (3, 20016, 21, 65, 2500), (1, 66000, 1, 128, 40000),
                                                 (7, 12816, 16, 100, 6000)])
def test_against_the_general_path(gpu, batch, rows_done_over, nc, rows, drop, k, ties):
    import torch
    from elmo_amd import ops
    g = torch.Generator(device=gpu).manual_seed(batch + k)
    labels = nc * rows - drop
    w = torch.randn(nc * rows, 768, generator=g, device=gpu).mul_(0.02)
    first = (labels - ties) * 2 // 3
    w[first:first + ties] = w[first]                                     # labels alike, the best of the rows below but for a few
    codes = w.to(torch.float8_e4m3fn)
    x = torch.randn(batch, 768, generator=g, device=gpu)
    which = {"all": range(batch), "last": [batch - 1], "one": [77], "two groups": [3, 31, 96], "three groups": [0, 33, 96],
             "five groups": [1, 60, 100, 161, 249]}[rows_done_over]
    for i, r in enumerate(which):
        best = codes[(first + 97 * i) % labels].float() if i % 2 else codes[first].float()     # the label alike, or another one above them
        x[r] = 27 * (best / best.norm() + (codes[first].float() / codes[first].float().norm() if i % 2 else 0))
    x = x.to(torch.bfloat16)
    chunks = [codes[c * rows:(c + 1) * rows].contiguous() for c in range(nc)]
    want_v, want_i = ops.fp8_forward_topk(chunks, x, labels, k, fused=False)
    for lo in range(0, batch, 128):
        status = ops.fp8_forward_topk(chunks, x[lo:lo + 128].contiguous(), labels, k, defer_check=True)[2]
        assert int(status[0]) & 1 or not any(lo <= r < lo + 128 for r in which)
    ws = ops.alloc_workspace(nc, rows, gpu)
    ws.view(torch.uint8)[: ops.step_sticky_error_offset()].fill_(0xFF)      # nothing of it is read before it is written
    for _ in range(2):
        got_v, got_i = ops.fp8_forward_topk(chunks, x, labels, k, workspace=ws)
        assert torch.equal(got_i, want_i) and torch.equal(got_v.view(torch.int16), want_v.view(torch.int16))
