"""Small true-FP8 steps, which take a workgroup for every 32 labels (xmc_fp8_small.hip), against the same steps on the fused kernel: more
than 4,096 (row, label) pairs take that one, and pairs outside the batch or the label space are ignored.  The weights are the same to the
bit; grad_X's fp32 sums are grouped by other labels, at most 255 additions of 256 partial sums whose rounding is 2^-24 of a sum that stays
below the sum of the magnitudes: 2^-16 of the largest value, as between the other forms."""
import numpy as np
import pytest

import helpers as H
from oracle import step as O
from test_fp8_step_gpu import check_rtn

pytestmark = pytest.mark.gpu


def both(gpu, nc, rows, batch, mode, extra=None, scale_w=1.0, scale_x=1.0):
    """Weights, fp32 and bf16 gradients of the step on either path, from the same inputs."""
    import torch
    from elmo_amd import ops
    case = H.make_case(nc, rows, batch, 17 * nc + rows + batch, extra_labels=extra, w_scale=scale_w)
    ws = ops.alloc_workspace(nc, rows, gpu)
    ws[: ops.step_sticky_error_offset()].fill_(0x7F)      # nothing of it is read before it is written
    out = []
    for ignored in (0, 4097):
        chunks, x, labels = H.to_device_case(case, gpu)
        labels = torch.cat([labels, torch.tensor([[-1, 0]], dtype=torch.int32, device=gpu).expand(ignored, 2)]).contiguous()
        g, gf = ops.fp8_step(chunks, x, labels, 0.05, seeds=[7 + 5 * c for c in range(nc)], round_mode=mode, scale_w=scale_w, scale_x=scale_x,
                             workspace=ws, want_f32=True)
        assert ops.step_error_word(ws, nc, rows) == 0
        out.append((H.chunks_to_numpy(chunks), gf, g))
    return case, out


@pytest.mark.parametrize("mode", ["rtn", "sr_fast", "sr_philox"])
@pytest.mark.parametrize("batch", [16, 32])
@pytest.mark.parametrize("nc,rows", [(1, 16), (1, 32), (1, 48), (3, 208), (2, 1040), (33, 32), (64, 16), (1, 2048), (1, 2064), (5, 1024), (2, 2576), (2, 4096), (1, 8208)])
def test_the_same_as_the_fused_kernel(gpu, nc, rows, batch, mode):
    _, ((w1, f1, g1), (w2, f2, g2)) = both(gpu, nc, rows, batch, mode)
    for a, b in zip(w1, w2):
        assert np.array_equal(a, b)
    tol = 2 ** -16 * f2.abs().max().item()
    assert (f1 - f2).abs().max().item() <= tol
    assert (g1.float() - f1).abs().max().item() <= 2 ** -8 * f1.abs().max().item()


@pytest.mark.parametrize("batch", [16, 32])
def test_positives(gpu, batch):
    """Repeated pairs, pairs outside the batch and the label space, a label of every row, the last labels of chunks; against the oracle."""
    nc, rows = 3, 208
    L = nc * rows
    extra = [(0, 0)] * 700 + [(b, 31) for b in range(batch)] + [(3, 32), (4, rows - 1), (5, rows), (6, L - 1)]
    ignored = [(batch, 2), (-1, 2), (1000, 2), (2, -1), (2, L), (2, 2 ** 31 - 1), (2, -2 ** 31)]
    case, ((w1, f1, _), (w2, _, _)) = both(gpu, nc, rows, batch, "rtn", extra=extra + ignored, scale_w=0.5, scale_x=2.0)
    for a, b in zip(w1, w2):
        assert np.array_equal(a, b)
    labels = np.array([p for p in case["labels"].tolist() if 0 <= p[0] < batch and 0 <= p[1] < L], dtype=np.int32)
    codes, gx, _ = O.fp8_step(case["chunks"], case["x"], labels, 0.05, sr_mode="rtn", scale_w=0.5, scale_x=2.0)
    for a, b in zip(w1, codes):
        assert H.e4m3_ulp_distance(a, b).max() <= 1 and np.mean(a == b) > 0.998
    assert np.abs(f1.cpu().numpy() - gx).max() <= 1e-3 * np.abs(gx).max()


@pytest.mark.parametrize("nc,rows,batch", [(1, 16, 16), (1, 48, 32), (33, 32, 16), (64, 16, 32), (2, 2576, 16), (5, 1024, 32), (1, 8192, 16)])
def test_against_the_oracle(gpu, nc, rows, batch):
    """One tile, partial tiles, many chunks, the most tiles of either batch."""
    check_rtn(H.make_case(nc, rows, batch, 23 * nc + rows + batch), gpu)


@pytest.mark.parametrize("mode", ["rtn", "sr_fast", "sr_philox"])
@pytest.mark.parametrize("batch", [16, 32])
def test_infinities_nan_and_the_largest_weights(gpu, batch, mode):
    """Weights at e4m3's largest values and NaN, embeddings that saturate, vanish or are no numbers: the same bits as the fused kernel's, and
    what is not finite in grad_X in the same places."""
    import torch
    from elmo_amd import ops
    nc, rows = 2, 80                                     # (chunks end in the middle of a tile)
    g = torch.Generator(device=gpu).manual_seed(batch)
    w0 = [torch.randn(rows, 768, generator=g, device=gpu).mul_(0.05).to(torch.float8_e4m3fn) for _ in range(nc)]
    w0[0].view(torch.uint8)[3, ::2] = 0x7E              # 448
    w0[0].view(torch.uint8)[4, ::3] = 0xFE              # -448
    x0 = torch.randn(batch, 768, generator=g, device=gpu)
    x0[0, :6] = torch.tensor([1e30, -1e30, 500.0, 2 ** -9, 1e-30, -0.0], device=gpu)
    special = x0.clone()
    special[1, 7], special[2, 8], special[batch - 1, 9] = float("inf"), -float("inf"), float("nan")
    pos = torch.stack([torch.arange(5 * batch, device=gpu) % batch, torch.randint(0, nc * rows, (5 * batch,), generator=g, device=gpu)], 1).to(torch.int32)
    ignored = torch.tensor([[-1, 0]], dtype=torch.int32, device=gpu)
    ws = ops.alloc_workspace(nc, rows, gpu)
    for x in (x0, special):
        for code in (0x30, 0x7F):                        # 0.5, NaN: in the last row of a chunk
            out = []
            for extra in (0, 4097):
                w = [c.clone() for c in w0]
                w[1].view(torch.uint8)[rows - 1, 5] = code
                labels = torch.cat([pos, ignored.expand(extra, 2)]).contiguous()
                _, gf = ops.fp8_step(w, x.to(torch.bfloat16), labels, 40.0, seeds=[7, 12], round_mode=mode, workspace=ws, want_f32=True)
                assert ops.step_error_word(ws, nc, rows) == 0
                out.append((torch.cat([c.view(torch.uint8) for c in w]), gf))
            (w1, f1), (w2, f2) = out
            assert torch.equal(w1, w2)
            assert bool(((w1 & 0x7F) == 0x7E).any())     # some updates saturate
            assert torch.equal(torch.isfinite(f1), torch.isfinite(f2))
            fin = torch.isfinite(f2)
            assert (f1 - f2)[fin].abs().max().item() <= 2 ** -16 * f2[fin].abs().max().item()
