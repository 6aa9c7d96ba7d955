"""One-pass steps of batches around the blocks of 16 rows and the clusters' halves: sums of blocks that the batch does not have are neither
written nor read.  A workspace full of huge numbers, and one that a full batch has used, give what a fresh one does, and the batch extended by
zero rows to all that its cluster holds gives the same weights and the same rows of grad_X, to the bit."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weights,mode", [("bf16", "rtn"), ("bf16", "sr_fast"), ("bf16", "sr_philox"), ("e4m3", "rtn"), ("e4m3", "sr_fast"), ("e4m3", "sr_philox"),
                                          ("fp8", "rtn"), ("fp8", "sr_fast"), ("fp8", "sr_philox")])
@pytest.mark.parametrize("batch,rows", [(b, 6016) for b in (1, 16, 17, 33, 48, 65, 80, 81, 129, 144, 177, 193, 241, 257, 273, 385, 497)] +
                         [(b, 10256) for b in (129, 144, 145, 161, 177)])
def test_neither_written_nor_read(gpu, batch, rows, weights, mode):
    """Clusters of all sizes: of three, for 129 to 192 rows, from 7,680 labels on with FP8 logits and 10,240 otherwise."""
    import torch
    from elmo_amd import ops
    members = next(c for c, most in ((1, 64), (2, 128), (3 if rows >= (7680 if weights == "fp8" else 10240) else 4, 192), (4, 256), (6, 384), (8, 512))
                   if batch <= most)
    cap = 32 if batch <= 32 else 64 * members       # rows that the cluster of this batch holds
    g = torch.Generator(device=gpu).manual_seed(batch)
    w0 = torch.randn(rows, 768, generator=g, device=gpu).mul_(0.05).to(torch.bfloat16 if weights == "bf16" else torch.float8_e4m3fn)
    x = torch.randn(512, 768, generator=g, device=gpu).to(torch.bfloat16)
    pos = torch.randint(0, rows, (4 * batch, 2), generator=g, device=gpu, dtype=torch.int32)
    pos[:, 0] = torch.arange(4 * batch, device=gpu, dtype=torch.int32) % batch
    off = ops.tiled_error_offset()

    def step(b, fill, xb, ws=None):
        ws = ops.alloc_tiled_workspace(1, rows, gpu, b) if ws is None else ws
        if fill is not None:
            ws[off + 8:].fill_(fill)
        w = w0.clone()
        _, gf = ops.tiled_step([w], rows, "bf16" if weights == "bf16" else "e4m3", xb, pos, 0.05, seeds=[7], round_mode=mode, workspace=ws, want_f32=True,
                               quantize_x=weights == "fp8", saturate=weights == "fp8")
        return w.view(torch.uint8), gf, ws

    fresh = step(batch, 0, x[:batch])
    assert torch.isfinite(fresh[1]).all() and not torch.equal(fresh[0], w0.view(torch.uint8))
    poisoned = step(batch, 0x7F, x[:batch])                                 # (3.4e38 in every word)
    full = (batch + 15) // 16 * 16
    ws = step(full, 0, x[:full])[2]
    used = step(batch, None, x[:batch], ws)
    for got in (poisoned, used):
        assert torch.equal(got[0], fresh[0]) and torch.equal(got[1], fresh[1])
    padded = torch.zeros(cap, 768, device=gpu, dtype=torch.bfloat16)
    padded[:batch] = x[:batch]
    whole = step(cap, 0, padded)
    assert torch.equal(whole[0], fresh[0]) and torch.equal(whole[1][:batch], fresh[1])
