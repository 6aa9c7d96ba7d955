"""Failed steps that ran in a workspace of their own (a batch larger than the layer's workspace, a call without one) are
reported like every other.  The failure is forced from the host: with a polling limit of 0 the second member of every
group that exchanges G leaves after three tiles, its partners' waits expire, every kernel ends normally and the step's
error word says so.  A call without a workspace reports the failure of the one before it."""
import pytest

import helpers as H
from test_host_cpu import make_cfg

pytestmark = pytest.mark.gpu

NC, ROWS = 2, 8192


def inputs(batch, gpu):
    # (every label of six tiles is positive for the rows of a cluster's first member)
    dense = [[b, 1024 * t + l] for t in range(6) for l in range(64) for b in range(64)]
    return H.to_device_case(H.make_case(NC, ROWS, batch, 611, extra_labels=dense), gpu)


def failing(step):
    """Runs `step` with a polling limit of 0, twice if need be, until it raises the report of a failed step; returns whether it did."""
    from elmo_amd import ops
    prev = ops.debug_spin_limit(0)
    try:
        for _ in range(2):
            try:
                step()
            except RuntimeError as e:
                assert "gave up waiting" in str(e)
                return True
        return False
    finally:
        ops.debug_spin_limit(prev)


def layer(kind, configured):
    from xmc_classifiers.chunked import XMCBCECHUNKEDLayer
    from xmc_classifiers.chunked_fp8xmc_clf import Fp8XMCBCEChunkedLayer
    cfg = make_cfg("cuda:0", NC * ROWS - 16, NC, rounding="rtn")
    cfg.data.batch_size = configured
    if kind == "bf16":
        cfg.model.xmc.dtype = "bfloat16"
        return XMCBCECHUNKEDLayer(cfg)
    return Fp8XMCBCEChunkedLayer(cfg)


@pytest.mark.parametrize("kind,configured,batch", [
    ("bf16", 32, 256),       # the layer's workspace is for 128 rows
    ("fp8", 144, 512),       # ... for 144
    ("fp8", 32, 256),        # the layer has no workspace for batches of this size
])
def test_layer_reports_a_failed_step_of_a_larger_batch(gpu, kind, configured, batch):
    xfc = layer(kind, configured)
    _, x, labels = inputs(batch, gpu)
    words = []

    def step():
        xfc.xfc_forward_backward(x, labels, [0.05])
        if kind == "fp8":
            words.append(xfc.last_step_error())
        xfc.check_steps()

    assert failing(step)
    assert words[-1:] == ([1] if kind == "fp8" else [])
    xfc.xfc_forward_backward(x, labels, [0.05])      # reported once; the next step is clean
    xfc.check_steps()
    if kind == "fp8":
        assert xfc.last_step_error() == 0


def test_larger_batch_does_not_hide_an_earlier_failure(gpu):
    xfc = layer("fp8", 32)
    _, x, labels = inputs(256, gpu)
    xfc.xfc_forward_backward(x[:32].contiguous(), labels, [0.05])
    xfc._errors.words[0].fill_(1)                    # as the last kernel of a failed step of 32 rows would have left it
    xfc.xfc_forward_backward(x, labels, [0.05])
    with pytest.raises(RuntimeError, match="gave up waiting"):
        xfc.check_steps()
    xfc.check_steps()


def test_step_in_a_workspace_that_is_too_small_leaves_its_error_word_in_it(gpu):
    import torch
    from elmo_amd import ops
    chunks, x, labels = inputs(256, gpu)
    ws = ops.alloc_tiled_workspace(NC, ROWS, gpu, 128)
    (sticky,) = ops.sticky_error_words(tiled_workspace=ws)

    def step():
        ops.tiled_step(chunks, ROWS, "e4m3", x, labels, 0.05, workspace=ws, quantize_x=True, saturate=True)
        if int(sticky.item()):
            raise RuntimeError("gave up waiting")

    assert failing(step)
    off = ops.tiled_error_offset()
    assert int(ws[off:off + 4].view(torch.int32).item()) == 1
    ops.tiled_step(chunks, ROWS, "e4m3", x, labels, 0.05, workspace=ws, quantize_x=True, saturate=True)
    assert int(ws[off:off + 4].view(torch.int32).item()) == 0 and int(sticky.item()) == 1


@pytest.mark.parametrize("entry", ["tiled", "fused"])
def test_step_without_a_workspace_is_reported(gpu, entry):
    """By ops.check_steps, or by the next call without a workspace, whichever comes first."""
    import torch
    from elmo_amd import ops
    chunks, x, labels = inputs(256 if entry == "tiled" else 64, gpu)

    def call():
        if entry == "tiled":
            ops.tiled_step(chunks, ROWS, "e4m3", x, labels, 0.05, quantize_x=True, saturate=True)
        else:
            ops.fp8_step(chunks, x, labels, 0.05)
        torch.cuda.synchronize()

    def step():
        call()
        ops.check_steps(gpu)

    ops.check_steps(gpu)
    assert failing(step)
    assert failing(call)
    ops.check_steps(gpu)       # reported once, and the call that raised has run no step
    call()
    ops.check_steps(gpu)


def test_replays_of_a_captured_step_without_a_workspace_are_reported(gpu):
    """The passing on of the error word is part of the graph: every replay that fails is reported."""
    import torch
    from elmo_amd import ops
    chunks, x, labels = inputs(256, gpu)
    gout = torch.empty(256, 768, dtype=torch.bfloat16, device=gpu)

    def call():
        ops.tiled_step(chunks, ROWS, "e4m3", x, labels, 0.05, quantize_x=True, saturate=True, grad_out=gout)

    call()
    ops.check_steps(gpu)
    prev = ops.debug_spin_limit(0)       # (a kernel parameter: the captured step keeps it)
    try:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            call()
    finally:
        ops.debug_spin_limit(prev)

    def step():
        graph.replay()
        ops.check_steps(gpu)

    assert failing(step) and failing(step)
    call()
    ops.check_steps(gpu)
