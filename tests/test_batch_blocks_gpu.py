"""The fused FP8 step in its variants for 32, 64, 96 and 128 batch rows, and the sizes from which batches of up to 64 rows take the
one-pass form: a batch and the same batch with rows of zeros up to 128 have the same weights, to the bit."""
import pytest

pytestmark = pytest.mark.gpu


def compare(gpu, nc, rows, batch, mode, dropout=0.0):
    import torch
    from elmo_amd import ops
    seeds = None if mode == "rtn" else [5 + 3 * c for c in range(nc)]
    g = torch.Generator(device=gpu).manual_seed(900 + batch)
    chunks = [torch.randn(rows, 768, generator=g, device=gpu).mul_(0.05).to(torch.float8_e4m3fn) for _ in range(nc)]
    padded = [c.clone() for c in chunks]
    x = torch.randn(batch, 768, generator=g, device=gpu).to(torch.bfloat16)
    x128 = torch.cat([x, torch.zeros(128 - batch, 768, dtype=torch.bfloat16, device=gpu)])
    n = 9 * batch
    labels = torch.stack([torch.arange(n, device=gpu) % batch, torch.randint(0, nc * rows, (n,), generator=g, device=gpu)], 1)
    edges = [[batch - 1, nc * rows - 1], [0, 0], [0, 0], [0, rows - 1], [-1, 3], [0, nc * rows]]        # (the last two are ignored)
    if nc * rows <= 8192 and batch <= 32:
        edges += [[-1, 3]] * 4097        # (more pairs than the small step's kernel takes)
    labels = torch.cat([labels, torch.tensor(edges, device=gpu)]).to(torch.int32).contiguous()
    ws = ops.alloc_workspace(nc, rows, gpu)
    ws.view(torch.uint8)[: ops.step_sticky_error_offset()].fill_(0xFF)      # nothing of it is read before it is written
    for _ in range(2):
        g1, f1 = ops.fp8_step(chunks, x, labels, 0.05, seeds=seeds, round_mode=mode, workspace=ws, want_f32=True, dropout_p=dropout, dropout_seed=7)
        g2, f2 = ops.fp8_step(padded, x128, labels, 0.05, seeds=seeds, round_mode=mode, workspace=ws, want_f32=True, dropout_p=dropout, dropout_seed=7)
        for a, b in zip(chunks, padded):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
        # at most two groupings of one fp32 sum (of at most 256 partial sums behind one another): 2^8 roundings of 2^-24
        tol = 2 ** -16 * f2[:batch].abs().max().item()
        assert (f1 - f2[:batch]).abs().max().item() <= tol and torch.allclose(g1.float(), g2[:batch].float(), rtol=2 ** -7, atol=tol)
        assert ops.step_error_word(ws, nc, rows) == 0


@pytest.mark.parametrize("nc,rows", [(1, 16), (3, 4112), (2, 9232), (2, 12816), (5, 5136), (3, 16400)])    # 1 to 13 tiles of a quad
@pytest.mark.parametrize("batch,mode", [(16, "sr_fast"), (32, "rtn"), (48, "sr_philox"), (64, "sr_fast"), (80, "rtn"), (96, "sr_fast"),
                                        (96, "sr_philox"), (112, "sr_fast")])
def test_fewer_batch_rows(gpu, nc, rows, batch, mode):
    compare(gpu, nc, rows, batch, mode, dropout=0.3 if batch == 80 else 0.0)


@pytest.mark.parametrize("tiles,batch,mode", [(6 * 256, 32, "rtn"), (20 * 256, 64, "rtn"), (32 * 256, 16, "sr_fast"), (64 * 256, 48, "sr_fast")])
def test_first_sizes_of_the_one_pass_form(gpu, tiles, batch, mode):
    compare(gpu, 8, tiles * 8 - 48, batch, mode)


@pytest.mark.parametrize("rows,num_head", [(4112, 1), (4112, 17), (4112, 4112), (9232, 6000), (20496, 20480)])   # partial tiles, 1 to 5 of a quad
@pytest.mark.parametrize("batch,mode,kind", [(16, "sr_fast", "bfloat16"), (64, "rtn", "float8_e5m2"), (48, "sr_philox", "bfloat16"), (96, "sr_fast", "float8_e5m2")])
def test_compensated_head(gpu, rows, num_head, batch, mode, kind):
    """The head's launch at two and at four blocks: weights, compensation terms (all of a row of NaN terms behind the head's end
    unread, untouched) and sums."""
    import torch
    from elmo_amd import ops
    nc = 2
    seeds = None if mode == "rtn" else [5, 8]
    g = torch.Generator(device=gpu).manual_seed(num_head + batch)
    chunks = [torch.randn(rows, 768, generator=g, device=gpu).mul_(0.05).to(torch.float8_e4m3fn) for _ in range(nc)]
    terms = torch.randn(num_head + 1, 768, generator=g, device=gpu).mul_(1e-3).to(getattr(torch, kind))
    terms.view(torch.uint8)[-1] = 0xFF
    padded, padded_terms = [c.clone() for c in chunks], terms.clone()
    x = torch.randn(batch, 768, generator=g, device=gpu).to(torch.bfloat16)
    x128 = torch.cat([x, torch.zeros(128 - batch, 768, dtype=torch.bfloat16, device=gpu)])
    n = 9 * batch
    labels = torch.stack([torch.arange(n, device=gpu) % batch, torch.randint(0, nc * rows, (n,), generator=g, device=gpu)], 1).to(torch.int32).contiguous()
    ws = ops.alloc_workspace(nc, rows, gpu)
    for _ in range(2):
        g1, f1 = ops.fp8_kahan_step(chunks, terms[:-1], num_head, x, labels, 0.05, seeds=seeds, round_mode=mode, workspace=ws, want_f32=True)
        g2, f2 = ops.fp8_kahan_step(padded, padded_terms[:-1], num_head, x128, labels, 0.05, seeds=seeds, round_mode=mode, workspace=ws, want_f32=True)
        for a, b in zip(chunks + [terms], padded + [padded_terms]):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
        tol = 2 ** -16 * f2[:batch].abs().max().item()        # as above
        assert (f1 - f2[:batch]).abs().max().item() <= tol
        assert ops.step_error_word(ws, nc, rows) == 0
    assert bool((terms.view(torch.uint8)[-1] == 0xFF).all())
