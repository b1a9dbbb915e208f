"""Vocabularies so large that the rows of a full-width 16-bit copy of an fp32 weight stored (H, V) would lie further apart than 32-bit
offsets reach over a tile: loss and gradients against 64 bits, the last hidden columns (the rows that lie furthest) by themselves.

x and the weight are rounded to the compute type in the oracle too, so what differs is dz and the results, each rounded once: half a
unit of 8 bits (bf16) for either, 2^-9 * 2^0.5 at most in the 2-norm; fp32 tensors go through products of bf16 pairs, 16 bits of
mantissa, 2^-17 a factor and three factors."""
import pytest
import torch

pytestmark = pytest.mark.gpu

BOUND = {torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -15}


def _exact(x, y, w, dtype, step=1 << 18):
    """Loss, dx and dW (in rows of the last 8 hidden columns) in 64 bits, the vocabulary in pieces."""
    N, V = x.shape[0], w.shape[1]
    xd, rows = x.detach().double(), torch.arange(N, device=x.device)
    lse = torch.full((N,), -torch.inf, dtype=torch.float64, device=x.device)
    target = torch.zeros_like(lse)
    for v in range(0, V, step):
        z = xd @ w[:, v:v + step].detach().to(dtype).double()
        lse = torch.logaddexp(lse, torch.logsumexp(z, 1))
        here = (y >= v) & (y < v + step)
        target[here] = z[rows[here], y[here] - v]
    dx, dw = torch.zeros_like(xd), torch.empty((8, V), dtype=torch.float64, device=x.device)
    for v in range(0, V, step):
        wv = w[:, v:v + step].detach().to(dtype).double()
        p = torch.exp(xd @ wv - lse[:, None])
        here = (y >= v) & (y < v + step)
        p[rows[here], y[here] - v] -= 1
        p /= N
        dx += p @ wv.t()
        dw[:, v:v + step] = xd[:, -8:].t() @ p
    return (lse - target).mean(), dx, dw


@pytest.mark.parametrize("N,H,V,dtype,route", [
    (100, 128, 8388608 + 1000, torch.bfloat16, True),  # a hidden size of the kernels without a stage
    (60, 256, 4194304 + 1000, torch.float32, True),  # fp32 tensors, whose logits are kept below that
    (60, 256, 4194304 + 1000, torch.bfloat16, "always"),  # an fp32 weight under 16-bit activations, one pass below that
])
def test_gradients_at_vocabularies_beyond_32_bit_offsets(N, H, V, dtype, route):
    from linear_cross_entropy_loss_amd import linear_cross_entropy, ops

    print(f"wide vocabulary N={N} H={H} V={V} {dtype} route={route}", flush=True)
    ops.one_pass.set(route)
    g = torch.Generator(device="cuda").manual_seed(H + N)
    x = torch.randn((N, H), generator=g, device="cuda").to(dtype).requires_grad_(True)
    w = torch.randn((H, V), generator=g, device="cuda").mul_(H ** -0.5).requires_grad_(True)
    y = torch.randint(0, V, (N,), generator=g, device="cuda")
    loss = linear_cross_entropy(x, y, w)[0]
    dx, dw = torch.autograd.grad(loss, (x, w))
    loss64, dx64, dw64 = _exact(x, y, w, dtype)
    assert abs(loss.item() / loss64.item() - 1) < 1e-5
    for got, ref in ((dx, dx64), (dx[:, -8:], dx64[:, -8:]), (dw[-8:], dw64)):
        assert ((got.double() - ref).norm() / ref.norm()).item() < BOUND[dtype]
