"""bf16 weights in clusters of six (257 to 384 batch rows), whose loads move within a tile's work where the weights pass 256 MB: a
layer just below the line, which the oracle pins at smaller sizes, and the same layer with rows of zeros up to and past it."""
import pytest

pytestmark = pytest.mark.gpu

LINE = (256 << 20) // 1536 // 32 * 32      # label rows; the tiles are 32 rows


@pytest.mark.parametrize("batch,mode", [(257, "rtn"), (384, "sr_fast"), (300, "sr_philox")])
def test_both_sides_of_the_line(gpu, batch, mode):
    import torch
    from elmo_amd import ops
    g = torch.Generator(device=gpu).manual_seed(batch)
    below = LINE - 32 * 7 - 5
    weights = torch.randn(below, 768, generator=g, device=gpu).mul_(0.05).to(torch.bfloat16)
    x = torch.randn(batch, 768, generator=g, device=gpu).to(torch.bfloat16)
    n = 9 * batch
    labels = torch.stack([torch.arange(n, device=gpu) % batch, torch.randint(0, below, (n,), generator=g, device=gpu)], 1).to(torch.int32).contiguous()
    off, results = ops.tiled_error_offset(), []
    for rows in (below, LINE, LINE + 1, LINE + 32 * 9 + 17):
        chunk = torch.zeros(rows, 768, dtype=torch.bfloat16, device=gpu)
        chunk[:below] = weights
        ws = ops.alloc_tiled_workspace(1, rows, gpu, batch)
        grads = []
        for seed in (5, 6):
            grads.append(ops.tiled_step([chunk], rows, "bf16", x, labels, 0.05, seeds=[seed], round_mode=mode, workspace=ws, want_f32=True)[1])
            assert int(ws[off:off + 4].view(torch.int32).item()) == 0
        results.append((chunk[:below].view(torch.int16), grads[0]))
    for chunk, grad in results[1:]:
        assert torch.equal(chunk, results[0][0])            # a row's update is a matter of its tile alone
        # rows of zeros add nothing to the first step's grad_X: two groupings of one fp32 sum (at most 2^8 roundings of 2^-24), each
        # rounded to bf16
        tol = 2 ** -16 * results[0][1].abs().max().item()
        assert torch.allclose(grad, results[0][1], rtol=2 ** -7, atol=tol)
