"""dx and dW on 128 x 128 tiles (lce_bwd_small.hip) against the persistent kernels on 256 x 256 tiles, which run where a call
limits its workgroups, on the same staged dz.

The two add the same products in another order: fp32 sums that differ by rounding, which moves a 16-bit result by at most one
unit in the last place (2^-7 of a bf16 number, 2^-10 of an fp16 one) and only where a sum lies next to a boundary.  In the 2-norm
that stays below a quarter of such a unit; fp32 results (sums of up to n products) stay within n^0.5 * 2^-24 * 2, 1e-5 up to 7000.

(Hidden sizes up to 128 in 16 bits have kernels of their own, lce_narrow.hip: test_gradients_on_small_tiles holds those to the same.)"""
import ctypes

import pytest
import torch

from helpers import make_inputs, rel_errors

pytestmark = pytest.mark.gpu

BOUND = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12, torch.float32: 1e-5}


def P(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else ctypes.c_void_p(0)


def _rows(t):
    m = 4 if t.dtype == torch.float32 else 8
    pad = torch.zeros(t.shape[0], t.shape[1] + (-t.shape[1]) % m, dtype=t.dtype, device="cuda")
    pad[:, :t.shape[1]] = t.cuda()
    return pad[:, :t.shape[1]]


def _check(N, H, V, n_chunk, dtype, w_dtype, layout, plan=None):
    """Both gradients against the persistent kernels, one alone against both.  `plan`: whether there are several slabs, dx is cut along
    K, dW is."""
    from linear_cross_entropy_loss_amd import _lib

    print(f"small tiles N={N} H={H} V={V} n_chunk={n_chunk} {dtype} {w_dtype} layout={layout}", flush=True)
    lib = _lib.load()
    x, y, w = make_inputs(N, H, V, dtype, seed=N + V, ignore_frac=0.2 if N > 1 else 0.0, w_dtype=w_dtype)
    x, w, y = _rows(x), _rows(w.t() if layout else w), y.cuda()
    g = torch.full((1,), 1024.0 if dtype == torch.float16 else 1.5, device="cuda")
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    m = 4 if dtype == torch.float32 else 8

    def run(workgroups, want_dx=True, want_dw=True):
        lddx, cols = H + (-H) % m, H if layout else V
        lddw = cols + (-cols) % 8
        prob = _lib.make_problem(N, H, V, x.stride(0), w.stride(0), lddx, lddw, dtype, w.dtype, dtype, w.dtype, -1, 0.7, 1e-3,
                                 n_chunk, False, 0, _lib.PACK_NEVER, workgroups, layout)
        if workgroups == 0 and plan is not None:
            slabs, (kernels, dx_cuts, dw_cuts, _) = _lib.backward_plan(prob)[0], _lib.gradient_kernels(prob)
            assert kernels == _lib.GRADS_SMALL and (slabs > 1, dx_cuts > 1, dw_cuts > 1) == plan, (slabs, kernels, dx_cuts, dw_cuts)
        fb, bb = _lib.workspace_bytes(prob)
        ws = torch.empty(max(fb, bb), dtype=torch.uint8, device="cuda")
        lse, out5 = torch.empty(N, device="cuda"), torch.empty(5, device="cuda")
        n = torch.empty(1, dtype=torch.int64, device="cuda")
        dx = torch.full((N, lddx), float("nan"), dtype=dtype, device="cuda") if want_dx else None
        dw = torch.full((V if layout else H, lddw), float("nan"), dtype=w.dtype, device="cuda") if want_dw else None
        a = (ctypes.byref(prob), P(x), P(w), P(y), P(lse))
        _lib.raise_for_status(lib.lce_forward(*a, P(out5), P(n), P(ws), fb, st), "lce_forward")
        _lib.raise_for_status(lib.lce_backward(*a, P(n), P(g), P(dx), P(dw), P(ws), bb, st), "lce_backward")
        torch.cuda.synchronize()
        return dx[:, :H] if want_dx else None, dw[:, :cols] if want_dw else None

    dx, dw = run(0)
    dx_p, dw_p = run(1 << 20)
    for got, ref in ((dx, dx_p), (dw, dw_p)):
        assert torch.isfinite(got).all()
        if ref.double().norm() > 0:
            longest = max(N, V) ** 0.5 * 2.0 ** -23
            assert rel_errors(got, ref)[1] <= max(BOUND[got.dtype], longest if got.dtype == torch.float32 else 0)
    assert (dx[y == -1] == 0).all()
    # one gradient alone: the same bits
    assert torch.equal(run(0, want_dw=False)[0], dx) and torch.equal(run(0, want_dx=False)[1], dw)


@pytest.mark.parametrize("dtype,w_dtype,layout", [(torch.bfloat16, None, 0), (torch.bfloat16, None, 1), (torch.float16, None, 0),
                                                  (torch.float16, torch.float32, 0), (torch.bfloat16, torch.float32, 1),
                                                  (torch.float32, None, 0)])
@pytest.mark.parametrize("N,H,V,n_chunk", [(1, 8, 8, 4096), (127, 128, 128, 4096), (129, 136, 1003, 4096), (300, 1000, 260, 4096),
                                           (700, 72, 4999, 4096), (2000, 264, 1501, 600), (5000, 64, 640, 2048)])
def test_gradients_on_small_tiles(N, H, V, n_chunk, dtype, w_dtype, layout):
    _check(N, H, V, n_chunk, dtype, w_dtype, layout)


@pytest.mark.parametrize("dtype,w_dtype,layout", [(torch.bfloat16, None, 0), (torch.bfloat16, None, 1), (torch.float16, None, 0),
                                                  (torch.float16, torch.float32, 0), (torch.bfloat16, torch.float32, 1),
                                                  (torch.float32, None, 0)])
@pytest.mark.parametrize("N,H,V,n_chunk,plan", [
    (129, 136, 499, 4096, (False, False, False)),    # nothing cut, the vocabulary's end inside a run of eight columns
    (700, 136, 4999, 4096, (False, True, False)),    # dx cut, one slab
    (300, 520, 9001, 4096, (False, True, False)),
    (5000, 136, 640, 16384, (False, False, True)),    # dW cut
    (200, 520, 9001, 240, (True, True, False)),      # dx cut, and summed over slabs
    (587, 296, 10053, 600, (True, True, False)),
    (6000, 136, 1300, 1024, (True, False, True))])   # dW cut in every slab
def test_cuts_and_slabs(N, H, V, n_chunk, plan, dtype, w_dtype, layout):
    _check(N, H, V, n_chunk, dtype, w_dtype, layout, plan)
