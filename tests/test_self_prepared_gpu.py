"""One-pass steps in clusters of one whose workgroups take X and up to 1,024 positives as they come, against the same steps behind the launch
that prepares both: more pairs take that one, and pairs outside the batch or the label space are ignored.  Everything else is the same, so
weights and gradients agree to the bit."""
import pytest

pytestmark = pytest.mark.gpu

WEIGHTS = [("bf16", "rtn"), ("bf16", "sr_philox"), ("e4m3", "rtn"), ("e4m3", "sr_fast")]


def compare(gpu, nc, rows, last, batch, weights, mode, seed, positives):
    """The step with the pairs as they are, with ignored ones among them up to 1,024 in any order (every thread holds two, 512 apart), and
    with 1,025.  positives(generator, labels): int64 [n, 2]."""
    import torch
    from elmo_amd import ops
    if weights == "e4m3":
        last = rows               # (chunks of e4m3 weights are equally long)
    g = torch.Generator(device=gpu).manual_seed(seed)
    total = rows * (nc - 1) + last
    w0 = torch.randn(total, 768, generator=g, device=gpu).mul_(0.05).to(torch.bfloat16 if weights == "bf16" else torch.float8_e4m3fn)
    x = torch.randn(batch, 768, generator=g, device=gpu).to(torch.bfloat16)
    pos = positives(g, total).to(torch.int32)
    assert pos.shape[0] <= 1024
    ignored = torch.tensor([[-1, 0]], dtype=torch.int32, device=gpu)
    mixed = torch.cat([pos, ignored.expand(1024 - pos.shape[0], 2)])[torch.randperm(1024, generator=g, device=gpu)]
    real = mixed[:, 0] != -1
    assert bool(real[:512].any()) and bool(real[512:].any())        # first and second pairs of threads
    ws = ops.alloc_tiled_workspace(nc, rows, gpu, batch)
    off = ops.tiled_error_offset()
    out = []
    for labels in (pos.contiguous(), mixed.contiguous(), torch.cat([mixed, ignored]).contiguous()):
        w = w0.clone()
        ws[off + 8:].fill_(0x7F)                        # nothing of it is read before it is written
        ws[off:off + 4].fill_(0x7F)                     # the error word: cleared by the step
        gb, gf = ops.tiled_step([w[c * rows:(c + 1) * rows] for c in range(nc)], rows, weights, x, labels, 0.05, seeds=[9 + c for c in range(nc)],
                                round_mode=mode, workspace=ws, want_f32=True)
        assert int(ws[off:off + 4].view(torch.int32).item()) == 0
        out.append((w.view(torch.uint8), gf, gb))
    for got in out[:2]:
        assert torch.equal(got[0], out[2][0]) and torch.equal(got[1], out[2][1]) and torch.equal(got[2].view(torch.int16), out[2][2].view(torch.int16))
    assert not torch.equal(out[0][0], w0.view(torch.uint8))
    return pos, total


@pytest.mark.parametrize("weights,mode", WEIGHTS)
@pytest.mark.parametrize("batch", [1, 16, 20, 32, 33, 49, 64])
@pytest.mark.parametrize("nc,rows,last", [(1, 16, 16), (1, 48, 48), (1, 2000, 2000), (3, 2720, 2720), (3, 2720, 17), (64, 64, 64), (1, 20000, 20000), (3, 30016, 29000)])
def test_the_same_as_behind_the_launch(gpu, nc, rows, last, batch, weights, mode):
    import torch

    def positives(g, total):
        n = 5 * batch
        rnd = torch.rand(n, generator=g, device=gpu)
        zipf = (rnd.mul(torch.log(torch.tensor(float(total), device=gpu))).exp() - 1).long().clamp(0, total - 1)       # a third in the first tiles
        pos = torch.stack([torch.arange(n, device=gpu) % batch, zipf], 1)
        edges = [[batch - 1, total - 1], [0, 0], [0, 0], [0, min(rows, total) - 1], [0, min(rows, total - 1)], [-1, 3], [batch, 3], [0, total], [0, -1], [0, 2 ** 31 - 1]]
        return torch.cat([pos, torch.tensor(edges, device=gpu)])

    compare(gpu, nc, rows, last, batch, weights, mode, rows + batch, positives)


@pytest.mark.parametrize("weights,mode", WEIGHTS)
@pytest.mark.parametrize("batch,a_row", [(16, 36), (28, 36), (64, 16)])
@pytest.mark.parametrize("nc,rows", [(1, 2000), (3, 2720), (3, 30016)])
def test_two_pairs_a_thread(gpu, nc, rows, batch, a_row, weights, mode):
    """576, 1,008 and 1,024 positives, spread over all labels."""
    import torch

    def positives(g, total):
        n = batch * a_row
        return torch.stack([torch.arange(n, device=gpu) // a_row, torch.randint(0, total, (n,), generator=g, device=gpu)], 1)

    compare(gpu, nc, rows, rows, batch, weights, mode, nc + rows + batch, positives)


@pytest.mark.parametrize("weights,mode", WEIGHTS)
@pytest.mark.parametrize("nc,rows,last", [(1, 600016, 600016), (3, 200016, 190000)])
def test_more_than_64_tiles_a_workgroup(gpu, nc, rows, last, weights, mode):
    """Positives in the tiles at either side of position 64 of every workgroup's sequence, where the sum over the tiles' counts goes on."""
    import torch
    from elmo_amd import _lib
    workgroups = _lib.load().xmc_step_workgroups()

    def positives(g, total):
        n = 1000
        return torch.stack([torch.arange(n, device=gpu) % 16, torch.randint(0, total, (n,), generator=g, device=gpu)], 1)

    pos, total = compare(gpu, nc, rows, last, 16, weights, mode, rows, positives)
    assert total // 32 > 70 * workgroups     # (so that a tenth of the positives lie behind position 64)
