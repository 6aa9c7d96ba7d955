"""Calls of the layers that have no gradient of their own, with an embedding and weights that require one, in grad mode: no result carries
a graph, none differs from the call under torch.no_grad(), and the embedding's graph is left as it was."""
import pytest

from test_host_cpu import make_cfg

pytestmark = pytest.mark.gpu


def embedding(device, features, dtype):
    import torch
    gen = torch.Generator(device=device).manual_seed(3)
    leaf = torch.randn(32, features, generator=gen, device=device).to(dtype).requires_grad_(True)
    return leaf, leaf * 0.05


def check(results, under_no_grad):
    import torch
    for r, n in zip(results, under_no_grad):
        assert not r.requires_grad and r.grad_fn is None
        assert torch.equal(r, n)


@pytest.mark.parametrize("simulated,features", [(False, 768), (False, 1024), (True, 768)])
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_inference_of_the_fp8_layer(gpu, simulated, features, dtype):
    import torch
    from xmc_classifiers.chunked_fp8xmc_clf import Fp8XMCBCEChunkedLayer
    cfg = make_cfg("cuda:0", 5000, 2, simulated=simulated)
    cfg.model.xmc.input_features = features
    torch.manual_seed(0)
    xfc = Fp8XMCBCEChunkedLayer(cfg).requires_grad_(True)
    assert all(w.requires_grad for w in xfc.xfc_weight)
    leaf, emb = embedding(gpu, features, getattr(torch, dtype))
    results = (xfc.xfc_forward(emb), *xfc.xfc_forward_topk(emb, 5))
    with torch.no_grad():
        check(results, (xfc.xfc_forward(emb), *xfc.xfc_forward_topk(emb, 5)))
    emb.sum().backward()
    assert torch.equal(leaf.grad, torch.full_like(leaf, 0.05))
    assert all(w.grad is None for w in xfc.xfc_weight)


@pytest.mark.parametrize("weights", ["bfloat16", "float32"])
@pytest.mark.parametrize("skip_loss", [True, False])
def test_step_of_the_bf16_layer(gpu, weights, skip_loss):
    import torch
    from xmc_classifiers.chunked import XMCBCECHUNKEDLayer
    labels = torch.tensor([[0, 3], [0, 999], [5, 17], [31, 500]], dtype=torch.int32, device=gpu)
    out = []
    for grad_mode in (True, False):
        cfg = make_cfg("cuda:0", 1000, 2, rounding="rtn")
        cfg.model.xmc.dtype = weights
        torch.manual_seed(0)
        xfc = XMCBCECHUNKEDLayer(cfg)
        xfc.xfc_weight.requires_grad_(grad_mode)
        leaf, emb = embedding(gpu, 768, torch.bfloat16)
        with torch.set_grad_enabled(grad_mode):
            loss = xfc.xfc_forward_backward(emb, labels, [0.05], skip_loss=skip_loss)
            logits = xfc.xfc_forward(emb.to(xfc._dtype))
        assert isinstance(loss, (int, float)) and xfc.iteration == 1 and "grad_input" not in dict(xfc.named_buffers())
        out.append((xfc.grad_input, logits, xfc.xfc_weight))
        if grad_mode:
            emb.backward(xfc.grad_input.to(emb.dtype))
            assert leaf.grad is not None and xfc.xfc_weight.grad is None and xfc.xfc_weight.grad_fn is None
    check(out[0][:2], out[1][:2])
    assert torch.equal(out[0][2], out[1][2])
