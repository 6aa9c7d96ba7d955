"""Inference logits of up to 64 batch rows, whose X the workgroups convert themselves: the same results, to the bit, as rows of a larger
batch, which take the operand image of X (the conversion is the same arithmetic, the products the same instructions)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 15, 16, 17, 32, 33, 47, 48, 49, 63, 64])
@pytest.mark.parametrize("nc,rows,labels", [(1, 16, 1), (1, 8208, 8200), (3, 8208, 24600), (1, 32784, 32768), (1, 32784, 32769), (2, 32784, 65540)])
def test_logits(gpu, nc, rows, labels, batch):
    """1 label, less than a tile, to several tiles for every workgroup, with and without some for all of the buffers that are loaded
    beside X; either side of the line up to which 49 to 64 rows are converted."""
    import torch
    from elmo_amd import ops
    g = torch.Generator(device=gpu).manual_seed(batch + labels)
    chunks = [torch.randn(rows, 768, generator=g, device=gpu).mul_(0.05).to(torch.float8_e4m3fn) for _ in range(nc)]
    x = torch.randn(80, 768, generator=g, device=gpu)
    x[0, :8] = torch.tensor([1e30, -1e30, float("inf"), -float("inf"), 1e-30, -0.0, 2 ** -9, 500.0], device=gpu)   # saturate, vanish
    x[batch // 2, 760:] *= 1e-3
    x = x.to(torch.bfloat16)
    ws = ops.alloc_workspace(nc, rows, gpu)
    for sw, sx in ((1.0, 1.0), (0.5, 0.37)):
        want = ops.fp8_forward(chunks, x, labels, sw, sx, workspace=ws)[:batch]
        got = ops.fp8_forward(chunks, x[:batch].contiguous(), labels, sw, sx, workspace=ws)
        assert torch.equal(got.contiguous().view(torch.int16), want.contiguous().view(torch.int16))
    nan = x[:batch].clone()
    nan[batch - 1, 5] = float("nan")          # (e4m3's smallest value, as in the image)
    want = ops.fp8_forward(chunks, torch.cat([nan, x[batch:]]), labels, workspace=ws)[:batch]
    got = ops.fp8_forward(chunks, nan, labels, workspace=ws)
    assert torch.equal(got.contiguous().view(torch.int16), want.contiguous().view(torch.int16))


@pytest.mark.parametrize("batch", [1, 16, 17, 32, 33, 48])
def test_logits_in_runs_of_tiles(gpu, batch):
    """From 32 tiles of 32 labels a compute unit on, up to 48 rows: runs of four tiles, with one to three of a workgroup's first tiles loaded beside
    X; a ragged end, the last round's tiles taken singly.  Rows of a larger batch read the image."""
    import torch
    from elmo_amd import _lib, ops
    nc, rows, labels = 2, 133136, 266263
    assert nc * rows // 32 > 32 * _lib.load().xmc_step_workgroups()
    g = torch.Generator(device=gpu).manual_seed(batch)
    chunks = [torch.randn(rows, 768, generator=g, device=gpu).mul_(0.05).to(torch.float8_e4m3fn) for _ in range(nc)]
    x = torch.randn(80, 768, generator=g, device=gpu).to(torch.bfloat16)
    ws = ops.alloc_workspace(nc, rows, gpu)
    want = ops.fp8_forward(chunks, x, labels, 0.5, 0.37, workspace=ws)[:batch]
    got = ops.fp8_forward(chunks, x[:batch].contiguous(), labels, 0.5, 0.37, workspace=ws)
    assert torch.equal(got.contiguous().view(torch.int16), want.contiguous().view(torch.int16))
