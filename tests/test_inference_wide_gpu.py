"""Inference of 129 to 256 batch rows in one pass over the weights: the same results, to the bit, as slices of 128 rows."""
import pytest

pytestmark = pytest.mark.gpu


def layer(gpu, nc, rows, batch, seed):
    import torch
    g = torch.Generator(device=gpu).manual_seed(seed)
    chunks = [torch.randn(rows, 768, generator=g, device=gpu).mul_(0.05).to(torch.float8_e4m3fn) for _ in range(nc)]
    return chunks, torch.randn(batch, 768, generator=g, device=gpu).to(torch.bfloat16)


@pytest.mark.parametrize("batch", [129, 144, 161, 200, 255, 256, 257, 400])
@pytest.mark.parametrize("nc,rows,labels", [(1, 16, 1), (1, 48, 47), (3, 80, 233), (2, 16400, 32799), (5, 2064, 10307)])
def test_logits(gpu, nc, rows, labels, batch):
    import torch
    from elmo_amd import ops
    chunks, x = layer(gpu, nc, rows, batch, 31 + batch)
    ws = ops.alloc_workspace(nc, rows, gpu)
    ws.view(torch.uint8)[: ops.step_sticky_error_offset()].fill_(0xFF)      # nothing of it is read before it is written
    got = ops.fp8_forward(chunks, x, labels, 0.5, 2.0, workspace=ws)
    assert got.shape == (batch, labels) and got.dtype == torch.bfloat16
    for lo in range(0, batch, 128):
        want = ops.fp8_forward(chunks, x[lo:lo + 128].contiguous(), labels, 0.5, 2.0, workspace=ws)
        assert torch.equal(got[lo:lo + 128].contiguous().view(torch.int16), want.contiguous().view(torch.int16))


@pytest.mark.parametrize("batch,k", [(129, 1), (129, 100), (160, 5), (200, 20), (255, 128), (256, 100), (300, 5), (500, 100)])
@pytest.mark.parametrize("nc,rows,labels", [(1, 640, 639), (3, 4112, 12300), (2, 16400, 32799), (5, 20496, 102480)])
@pytest.mark.parametrize("alike", [False, True])
def test_topk(gpu, nc, rows, labels, batch, k, alike):
    """alike: rows with all logits the same, whose candidates overflow every list and are done over."""
    import torch
    from elmo_amd import ops
    chunks, x = layer(gpu, nc, rows, batch, 71 + batch + k)
    if alike:
        x[3] = 0
        x[batch - 1] = 0
        x[140 % batch] = 0
    ws = ops.alloc_workspace(nc, rows, gpu)
    ws.view(torch.uint8)[: ops.step_sticky_error_offset()].fill_(0xFF)
    for _ in range(2):
        vals, idx = ops.fp8_forward_topk(chunks, x, labels, k, workspace=ws)
        for lo in range(0, batch, 128):
            want_v, want_i = ops.fp8_forward_topk(chunks, x[lo:lo + 128].contiguous(), labels, k, workspace=ws)
            assert torch.equal(idx[lo:lo + 128], want_i) and torch.equal(vals[lo:lo + 128].view(torch.int16), want_v.view(torch.int16))


@pytest.mark.parametrize("nc,rows,labels", [(1, 262144, 262144), (1, 262160, 262113), (2, 131104, 262199), (3, 87376, 262121)])
def test_logits_of_many_labels(gpu, nc, rows, labels):
    """The sizes from which up to 128 rows are written in runs of four tiles, against more rows, which are not."""
    import torch
    from elmo_amd import ops
    chunks, x = layer(gpu, nc, rows, 144, labels % 97)
    want = ops.fp8_forward(chunks, x, labels)
    for batch in (17, 40, 128):
        got = ops.fp8_forward(chunks, x[:batch].contiguous(), labels)
        assert torch.equal(got.contiguous().view(torch.int16), want[:batch].contiguous().view(torch.int16))


@pytest.mark.parametrize("defer,entry", [(False, "xmc_fp8_forward_topk_wide"), (True, "xmc_fp8_forward_topk_fused_rows")])
def test_a_refused_call_names_its_function(gpu, defer, entry):
    from elmo_amd import _lib, ops
    chunks, x = layer(gpu, 2, 16400, 20, 5)
    workspace = ops.alloc_workspace(2, 16400, gpu)[:1024]        # too small: refused before anything is launched
    with pytest.raises(_lib.XmcError, match="^%s failed: workspace too small" % entry):
        ops.fp8_forward_topk(chunks, x, 32800, 5, workspace=workspace, defer_check=defer)
