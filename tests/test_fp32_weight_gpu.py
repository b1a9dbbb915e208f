"""The loss of few tokens under an fp32 weight, which the 128 x 128 kernel reads as it is and rounds on its way to LDS, against the
16-bit copies of the weight that a call with limited workgroups makes: the same rounding, the same products in the same order, so
the same bits.  The padding of the weight's rows holds NaN, which must not come through.  N = 257 and pairs with 12287 columns or
monitoring lie beyond the rule's lines, where both calls make the copy."""
import ctypes

import pytest
import torch

from helpers import make_inputs

pytestmark = pytest.mark.gpu


def P(t):
    return ctypes.c_void_p(t.data_ptr())


def _rows(t, fill):
    m = 4 if t.dtype == torch.float32 else 8
    pad = torch.full((t.shape[0], t.shape[1] + (-t.shape[1]) % m + m), fill, dtype=t.dtype, device="cuda")
    pad[:, :t.shape[1]] = t.cuda()
    return pad[:, :t.shape[1]]


@pytest.mark.parametrize("dtype,layout", [(torch.bfloat16, 0), (torch.bfloat16, 1), (torch.float16, 0), (torch.float16, 1), (torch.float32, 0)])
@pytest.mark.parametrize("N,H,V", [(1, 8, 13000), (33, 72, 260), (33, 63, 12288), (127, 129, 12287), (128, 136, 1003), (129, 250, 13003),
                                   (256, 1000, 12801), (257, 320, 12545)])
@pytest.mark.parametrize("monitoring", [False, True])
def test_loss_of_few_tokens(N, H, V, dtype, layout, monitoring):
    from linear_cross_entropy_loss_amd import _lib

    if layout and H % 8:
        H += 8 - H % 8
    print(f"fp32 weight as it is N={N} H={H} V={V} {dtype} layout={layout} monitoring={monitoring}", flush=True)
    lib = _lib.load()
    x, y, w = make_inputs(N, H, V, dtype, seed=N + V, ignore_frac=0.2 if N > 1 else 0.0, w_dtype=torch.float32)
    x, w, y = _rows(x, 0.0), _rows(w.t() if layout else w, float("nan")), y.cuda()
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def run(workgroups):
        prob = _lib.make_problem(N, H, V, x.stride(0), w.stride(0), x.stride(0), w.stride(0), dtype, torch.float32, dtype, torch.float32, -1,
                                 0.7, 1e-3, 4096, monitoring, 0, _lib.PACK_NEVER, workgroups, layout)
        size = _lib.forward_workspace_bytes(prob)
        ws = torch.empty(size, dtype=torch.uint8, device="cuda")
        lse, out5 = torch.empty(N, device="cuda"), torch.empty(5, device="cuda")
        n = torch.empty(1, dtype=torch.int64, device="cuda")
        _lib.raise_for_status(lib.lce_forward(ctypes.byref(prob), P(x), P(w), P(y), P(lse), P(out5), P(n), P(ws), size, st), "lce_forward")
        torch.cuda.synchronize()
        return size, lse, out5, n

    size, lse, out5, n = run(0)
    size_c, lse_c, out5_c, n_c = run(100)
    assert torch.isfinite(lse).all() and torch.isfinite(out5).all()
    assert torch.equal(lse, lse_c) and torch.equal(out5, out5_c) and torch.equal(n, n_c)
    direct = N <= 256 and (dtype != torch.float32 or (V >= 12288 and not monitoring))
    assert (size < size_c) == direct  # (no room for the copy where none is made)
