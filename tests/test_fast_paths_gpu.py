"""GPU tests of dispatch branches that a size, a value range or the calling mode selects, at the sizes where they can go wrong."""
import pytest
import torch

from helpers import make_inputs, rel_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mode", ["no_grad", "inference", "detached"])
def test_loss_without_gradients_allocates_no_gradients(mode, dtype):
    """A parameter under no_grad needs no gradient: the call computes the loss alone (the same bits) and takes less
    memory than a weight gradient would."""
    from linear_cross_entropy_loss_amd import LinearCrossEntropyLoss

    N, H, V = 300, 256, 8192
    x, y, w = make_inputs(N, H, V, dtype, 3, ignore_frac=0.1, device="cuda")
    mod = LinearCrossEntropyLoss(H, V, device="cuda", dtype=dtype, ignore_index=-1, init_method=lambda t: t.data.copy_(w))
    mod.monitoring = True
    want = mod(x.clone().requires_grad_(), y).detach()
    want_max = mod.latest_metrics["logit_max"]
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    if mode == "detached":
        mod.weight.requires_grad_(False)
        loss = mod(x, y)
    else:
        with torch.no_grad() if mode == "no_grad" else torch.inference_mode():
            loss = mod(x, y)
    torch.cuda.synchronize()
    assert not loss.requires_grad
    # (fp32 takes one product of bf16 pairs at a time either way; bf16 sums of the loss may be cut at other places)
    assert torch.allclose(loss, want, rtol=1e-6, atol=0)
    assert torch.allclose(mod.latest_metrics["logit_max"], want_max, rtol=1e-6, atol=0)
    if dtype == torch.bfloat16:
        assert torch.cuda.max_memory_allocated() - before < H * V * 2
