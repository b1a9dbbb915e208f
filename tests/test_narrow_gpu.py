"""Hidden sizes up to lce_internal.h's kNarrowHidden: forward and gradients without a stage (lce_narrow.hip) against the staged
kernels, which run where a call limits its workgroups.

The logits have the same bits (the same products along the same K order), and with them lse and dz; dx and dW add the same products in
another order: fp32 rounding, which moves a 16-bit result by at most one unit in the last place and only next to a boundary -- below a
quarter of such a unit in the 2-norm --, an fp32 one of n products by n^0.5 * 2^-24 * 2 at most (1e-5 up to 7000 of them)."""
import ctypes

import pytest
import torch

from helpers import make_inputs, rel_errors

pytestmark = pytest.mark.gpu

BOUND = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12, torch.float32: 1e-5}


def P(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else ctypes.c_void_p(0)


def _rows(t, extra=0):
    """Rows on 16-byte boundaries, with the largest finite numbers of the type behind them."""
    m = 4 if t.dtype == torch.float32 else 8
    pad = torch.full((t.shape[0], t.shape[1] + (-t.shape[1]) % m + extra), torch.finfo(t.dtype).max if extra else 0, dtype=t.dtype, device="cuda")
    pad[:, :t.shape[1] + (-t.shape[1]) % m] = 0
    pad[:, :t.shape[1]] = t.cuda()
    return pad[:, :t.shape[1]]


def _check(N, H, V, extra, mon, z_reg, dtype, w_dtype, layout, n_chunk=4096, pack=2, inputs=None):
    """Both directions against the persistent kernels, one gradient alone against both.  Returns what was compared and how to run it
    again.  `pack`: LCE_PACK_NEVER, or how the call says it (LCE_PACK_ALWAYS: the backward is staged); `inputs`: instead of
    make_inputs'."""
    from linear_cross_entropy_loss_amd import _lib

    print(f"narrow N={N} H={H} V={V} {dtype} {w_dtype} layout={layout}", flush=True)
    lib = _lib.load()
    x, y, w = inputs or make_inputs(N, H, V, dtype, seed=N + V, ignore_frac=0.2 if N > 1 else 0.0, w_dtype=w_dtype)
    x, w, y = _rows(x, extra), _rows(w.t() if layout else w, extra), y.cuda()
    g = torch.full((1,), 1024.0 if dtype == torch.float16 else 1.5, device="cuda")
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def run(workgroups, want_dx=True, want_dw=True):
        lddx, cols = H + (-H) % 8, H if layout else V
        lddw = cols + (-cols) % 8
        prob = _lib.make_problem(N, H, V, x.stride(0), w.stride(0), lddx, lddw, dtype, w.dtype, dtype, w.dtype, -1, 0.7, z_reg, n_chunk,
                                 mon, 0, pack, workgroups, layout)
        if workgroups == 0 and pack != _lib.PACK_ALWAYS:
            assert _lib.gradient_kernels(prob)[0] == _lib.GRADS_NARROW
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
        return out5, lse, dx[:, :H] if want_dx else None, dw[:, :cols] if want_dw else None

    out, lse, dx, dw = run(0)
    # (64 workgroups: the persistent kernels, forward and backward)
    out_p, lse_p, dx_p, dw_p = run(64)
    k = 5 if mon else 2
    assert torch.equal(lse[y != -1], lse_p[y != -1]) and (torch.equal(out[:k], out_p[:k]) or bool((y == -1).all()))
    for got, ref in ((dx, dx_p), (dw, dw_p)):
        assert torch.isfinite(got).all()
        if ref.double().norm() > 0:
            longest = max(N, V) ** 0.5 * 2.0 ** -23
            assert rel_errors(got, ref)[1] <= max(BOUND[got.dtype], longest if got.dtype == torch.float32 else 0)
    assert (dx[y == -1] == 0).all()
    # one gradient alone: the same bits
    assert torch.equal(run(0, want_dw=False)[2], dx) and torch.equal(run(0, want_dx=False)[3], dw)
    return run, x, y, out, lse, dx, dw


@pytest.mark.parametrize("dtype,w_dtype,layout", [(torch.bfloat16, None, 0), (torch.bfloat16, None, 1), (torch.float16, None, 0),
                                                  (torch.float16, torch.float32, 1), (torch.bfloat16, torch.float32, 0)])
@pytest.mark.parametrize("N,H,V,extra,mon,z_reg", [
    (1, 8, 8, 0, False, 0.0), (127, 64, 129, 0, True, 1e-3), (128, 72, 128, 16, False, 1e-3), (129, 128, 1003, 0, True, 0.0),
    (700, 40, 5001, 8, False, 0.0), (3000, 104, 300, 0, False, 1e-3), (260, 120, 777, 8, True, 1e-3), (515, 56, 2050, 0, False, 0.0)])
def test_narrow_hidden_sizes(N, H, V, extra, mon, z_reg, dtype, w_dtype, layout):
    _check(N, H, V, extra, mon, z_reg, dtype, w_dtype, layout)


@pytest.mark.parametrize("dtype,w_dtype,layout", [(torch.bfloat16, None, 0), (torch.float16, None, 1), (torch.bfloat16, torch.float32, 0)])
@pytest.mark.parametrize("N,H,V,n_chunk", [(9000, 40, 24, 512), (17000, 16, 300, 32), (262144, 64, 32, 4096)])
def test_many_tokens_and_few_classes(N, H, V, n_chunk, dtype, w_dtype, layout):
    """The bound leaves the sums over the tokens no room; they are cut all the same."""
    from linear_cross_entropy_loss_amd import _lib

    wd, ld = w_dtype or dtype, H if layout else V + (-V) % 8
    prob = _lib.make_problem(N, H, V, H, ld, H, ld, dtype, wd, dtype, wd, -1, 0.7, 0.0, n_chunk, False, 0, _lib.PACK_NEVER, 0, layout)
    assert _lib.gradient_kernels(prob)[2] > 1 and _lib.backward_workspace_bytes(prob) > n_chunk * V * 4
    _check(N, H, V, 0, False, 1e-3, dtype, w_dtype, layout, n_chunk)


def _on_device(N, H, V, dtype, w_dtype, ignored):
    g = torch.Generator(device="cuda").manual_seed(N)
    x = torch.randn((N, H), generator=g, device="cuda").to(dtype)
    w = torch.randn((H, V), generator=g, device="cuda").mul_(H ** -0.5).to(w_dtype or dtype)
    y = torch.randint(0, V, (N,), generator=g, device="cuda")
    y[torch.rand(N, generator=g, device="cuda") < ignored] = -1
    return x, y, w


@pytest.mark.parametrize("dtype,w_dtype,layout", [(torch.bfloat16, None, 0), (torch.float16, None, 1), (torch.float16, torch.float32, 0)])
@pytest.mark.parametrize("N,H,V,ignored", [(20000, 128, 107400, 0.85), (22000, 120, 104200, 0.05), (40000, 64, 107400, 0.3),
                                           (20000, 128, 107400, 0.0), (20000, 128, 107400, 1.0)])
def test_ignored_tokens_of_a_large_problem_are_packed_away(N, H, V, ignored, dtype, w_dtype, layout):
    """From 8 * N * H * V = 2^41 on the tokens with an ignored label are not worked on, and what stands in their rows of x does not
    reach a result."""
    from linear_cross_entropy_loss_amd import _lib

    assert 8 * N * H * V >= 1 << 41
    run, xr, y, out, lse, dx, dw = _check(N, H, V, 0, False, 1e-3, dtype, w_dtype, layout, 4096, _lib.PACK_AUTO,
                                          _on_device(N, H, V, dtype, w_dtype, ignored))
    if 0 < ignored < 1:
        xr[y == -1] = float("inf")
        again = run(0)
        for a, b in zip((out[:2], lse, dx, dw), (again[0][:2],) + again[1:]):
            assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,w_dtype,layout", [(torch.bfloat16, None, 0), (torch.float16, torch.float32, 1)])
@pytest.mark.parametrize("N,H,V", [(1000, 72, 1300), (129, 24, 5001), (20000, 64, 300)])
def test_forward_of_packed_rows(N, H, V, dtype, w_dtype, layout):
    """The forward on the rows that are left; the last case in two chunks of tokens."""
    from linear_cross_entropy_loss_amd import _lib

    _check(N, H, V, 0, False, 1e-3, dtype, w_dtype, layout, 4096, _lib.PACK_ALWAYS)


@pytest.mark.parametrize("mon", [False, True])
@pytest.mark.parametrize("N", [16385, 40000])
def test_several_chunks_of_tokens(N, mon):
    """The forward goes through 16384 tokens at a time."""
    _check(N, 40, 260, 0, mon, 0.0, torch.bfloat16, None, 0, 65536 // 8)


@pytest.mark.parametrize("layout", [0, 1])
def test_forward_on_slabs_of_an_fp32_weight(layout):
    """Its copies of an fp32 weight are 256 MiB at most: here two, the second one 300 columns wide."""
    _check(300, 128, (1 << 20) + 300, 0, False, 1e-3, torch.bfloat16, torch.float32, layout,
           inputs=_on_device(300, 128, (1 << 20) + 300, torch.bfloat16, torch.float32, 0.1))
