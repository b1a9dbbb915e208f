"""lce_forward_backward with LCE_ROUTE_KEEP_LOGITS (fp32 tensors): the logits computed once, kept in fp32 and turned into dz in place,
against lce_forward + lce_backward, which compute them twice.

dz has the same bits on both ways if lse has; lse is summed in another order (fp32 rounding, 2^-22 of a logit of order 10), and dx and
dW add the same products in another order: sums of up to 20000 fp32 products, 20000^0.5 * 2^-24 * 2 = 1.7e-5 at most, 1e-5 in the
2-norm at these sizes."""
import ctypes

import pytest
import torch

from helpers import make_inputs, rel_errors
from linear_cross_entropy_loss_amd._lib import GRADS_LARGE, GRADS_SMALL

pytestmark = pytest.mark.gpu


def P(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else ctypes.c_void_p(0)


def _rows(t):
    pad = torch.zeros(t.shape[0], t.shape[1] + (-t.shape[1]) % 4, dtype=t.dtype, device="cuda")
    pad[:, :t.shape[1]] = t.cuda()
    return pad[:, :t.shape[1]]


def _check(N, H, V, n_chunk, chunks, mon, plan=None):
    """`plan`: the kernels of the gradients, whether they cut dx along K, whether dx has fewer workgroups than compute units."""
    from linear_cross_entropy_loss_amd import _lib, ops

    print(f"kept logits N={N} H={H} V={V} n_chunk={n_chunk} mon={mon} pack={ops.pack_rows.get()}", flush=True)
    lib = _lib.load()
    x, y, w = make_inputs(N, H, V, torch.float32, seed=N + V, ignore_frac=0.3 if N > 1 else 0.0)
    x, w, y = _rows(x), _rows(w), y.cuda()
    f32, hp, vp = torch.float32, H + (-H) % 4, V + (-V) % 4
    g = torch.full((1,), 1.5, device="cuda")
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def run(route):
        prob = _lib.make_problem(N, H, V, x.stride(0), w.stride(0), hp, vp, f32, f32, f32, f32, -1, 0.7, 1e-3, n_chunk, mon, 0,
                                 ops.pack_rows.get(), 0, 0, route)
        got = _lib.forward_backward_plan(prob)[0]
        if plan is not None and route != _lib.ROUTE_TWO_PASS:
            kernels, dx_cuts, _, limit = _lib.gradient_kernels(prob, one_pass=True)
            assert (kernels, dx_cuts > 1, limit > 0) == plan, (kernels, dx_cuts, limit)
        nbytes = _lib.forward_backward_workspace_bytes(prob)
        assert got == 0 or nbytes <= n_chunk * V * 4
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        lse, out5, n = torch.empty(N, device="cuda"), torch.empty(5, device="cuda"), torch.empty(1, dtype=torch.int64, device="cuda")
        dx, dw = torch.full((N, hp), float("nan"), device="cuda"), torch.full((H, vp), float("nan"), device="cuda")
        _lib.raise_for_status(lib.lce_forward_backward(ctypes.byref(prob), P(x), P(w), P(y), P(g), P(lse), P(out5), P(n), P(dx), P(dw),
                                                       P(ws), nbytes, st), "lce_forward_backward")
        torch.cuda.synchronize()
        return got, out5, n, dx[:, :H], dw[:, :V]

    got, out5, n, dx, dw = run(_lib.ROUTE_ONE_PASS | _lib.ROUTE_KEEP_LOGITS)
    _, out_t, n_t, dx_t, dw_t = run(_lib.ROUTE_TWO_PASS)
    assert got >= chunks, got
    assert n.item() == n_t.item() and (dx[y == -1] == 0).all()
    k = 5 if mon else 2
    assert torch.allclose(out5[:k], out_t[:k], rtol=2e-6, atol=2e-6)
    for a, b in ((dx, dx_t), (dw, dw_t)):
        assert torch.isfinite(a).all()
        assert rel_errors(a, b)[1] <= 1e-5


@pytest.mark.parametrize("N,H,V,n_chunk,chunks,mon", [
    (1, 8, 200, 4096, 1, False),        # one tile, nearly all of it outside
    (130, 72, 1001, 4096, 1, True),     # the vocabulary's end inside a run of eight columns, small tiles, monitoring values
    (700, 300, 5000, 2048, 1, False),
    (2500, 136, 3003, 1024, 3, False),  # several chunks on small tiles, the last one short
    (2048, 1024, 12000, 2304, 2, False),  # several chunks; packed rows on large tiles
    (900, 264, 20000, 2048, 1, True)])
def test_kept_logits_give_the_gradients_of_the_two_calls(N, H, V, n_chunk, chunks, mon, pack_mode):
    _check(N, H, V, n_chunk, chunks, mon)


@pytest.mark.parametrize("N,H,V,n_chunk,chunks,plan", [
    (2500, 136, 3003, 1024, 3, (GRADS_SMALL, True, False)),     # small tiles, dx cut in every chunk
    (2048, 2048, 16384, 4096, 2, (GRADS_LARGE, False, True)),   # large tiles, dx on as many workgroups as the bound has room for
    (3000, 2048, 20001, 6144, 2, (GRADS_LARGE, False, False))])  # large tiles, the last chunk short
def test_chunks_on_either_tiles(N, H, V, n_chunk, chunks, plan):
    from linear_cross_entropy_loss_amd import _lib, ops

    ops.pack_rows.set(_lib.PACK_NEVER)  # (packed rows are for the large tiles alone)
    _check(N, H, V, n_chunk, chunks, False, plan)
