"""The host extension (csrc/lce_host.cpp) against the same calls through ops.py's own host code: the same device calls, so the same
bits, over every form of input that either takes, and the same errors."""
import pytest
import torch

pytestmark = pytest.mark.gpu

N, H, V = 300, 104, 1000


def _mat(rows, cols, dtype, seed, pad=0, offset=0, transposed=False, apart=False):
    """A (rows, cols) matrix: row-major with `pad` more elements in a row, `offset` elements into its storage; `transposed`: stored
    the other way round; `apart`: elements two apart in both directions."""
    g = torch.Generator().manual_seed(seed)
    r, c = (cols, rows) if transposed else (rows, cols)
    flat = (torch.randn(offset + r * (c + pad) * (4 if apart else 1), generator=g) / 8).to(dtype).cuda()[offset:]
    t = flat.view(2 * r, 2 * (c + pad))[::2, ::2][:, :c] if apart else flat.view(r, c + pad)[:, :c]
    return t.t() if transposed else t


FORMS = {
    "plain": {},
    "3d": dict(x3=True),
    "odd hidden": dict(H=101),
    "odd vocabulary": dict(V=1003),
    "both odd, multiples of four": dict(H=100, V=996),
    "x off its boundary": dict(x=dict(offset=1)),
    "x rows apart": dict(x=dict(pad=8)),
    "x elements apart": dict(x=dict(apart=True)),
    "labels apart": dict(y2=True),
    "weight rows longer": dict(w=dict(pad=8)),
    "weight rows longer, odd": dict(w=dict(pad=3)),
    "weight off its boundary": dict(w=dict(offset=4)),
    "tied": dict(w=dict(transposed=True)),
    "tied, rows longer": dict(w=dict(transposed=True, pad=8)),
    "tied, odd hidden": dict(H=101, w=dict(transposed=True)),
    "tied, odd vocabulary": dict(V=1003, w=dict(transposed=True)),
    "weight elements apart": dict(w=dict(apart=True)),
    "one token": dict(N=1),
    "one pass": dict(N=1024, H=520, V=4096, always=True),
    "one pass, odd": dict(N=1024, H=515, V=4099, always=True),
}


@pytest.mark.parametrize("dtype,w_dtype", [(torch.bfloat16, None), (torch.float16, None), (torch.float16, torch.float32), (torch.float32, None)])
@pytest.mark.parametrize("form", FORMS)
def test_the_extension_gives_what_the_operators_own_host_code_gives(form, dtype, w_dtype, monkeypatch):
    from linear_cross_entropy_loss_amd import _lib, linear_cross_entropy, ops

    f = FORMS[form]
    n, h, v = f.get("N", N), f.get("H", H), f.get("V", V)
    print(f"host path: {form} {dtype} {w_dtype}", flush=True)
    if f.get("always"):
        ops.one_pass.set("always")
    ops._copy_warned.add("weight")
    handled = []

    def run(native):
        x = _mat(n, h, dtype, 1, **f.get("x", {}))
        if f.get("x3"):
            x = x.view(3, n // 3, h)
        x.requires_grad_(True)
        w = _mat(h, v, w_dtype or dtype, 2, **f.get("w", {})).requires_grad_(True)
        y = torch.randint(0, v, (n, 2 if f.get("y2") else 1), generator=torch.Generator().manual_seed(3)).cuda()[:, 0]
        y = y.view(3, n // 3) if f.get("x3") else y
        if n > 1:
            y.view(-1)[::7] = -100 if not f.get("y2") else y[0]
        with monkeypatch.context() as m:
            real = _lib.host()

            class Host:
                @staticmethod
                def forward(*a):
                    out = real.forward(*a) if native else None
                    handled.append(out is not None)
                    return out

                @staticmethod
                def backward(*a):
                    return real.backward(*a) if native else None

            m.setattr(_lib, "host", lambda: Host)
            out = linear_cross_entropy(x, y, w, -100, 1e-4, 0.5, 4096, True)
            first = torch.autograd.grad(out[0] * 3, (x, w), retain_graph=True)
            again = torch.autograd.grad(out[0] * 3, (x, w))
            with torch.no_grad():
                alone = linear_cross_entropy(x, y, w, -100, 1e-4, 0.5, 4096, False)
            only = torch.autograd.grad(linear_cross_entropy(x, y, w.detach(), -100, 1e-4, 0.5, 4096)[0], x)
        return [o.detach() for o in out] + [alone[0]] + list(first) + list(again) + list(only)

    got, ref = run(True), run(False)
    assert form in ("x rows apart", "x elements apart", "labels apart", "weight off its boundary", "weight elements apart") or handled[0]
    for a, b in zip(got, ref):
        assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride()
        assert torch.equal(a, b)


@pytest.mark.parametrize("what", ["label dtype", "label count", "dtypes", "hidden size", "cpu labels", "scale"])
def test_errors_are_those_of_the_operators_own_host_code(what, monkeypatch):
    from linear_cross_entropy_loss_amd import linear_cross_entropy, ops

    x = _mat(N, H, torch.bfloat16, 1)
    w = _mat(H + (8 if what == "hidden size" else 0), V, torch.float16 if what == "dtypes" else torch.bfloat16, 2)
    y = torch.zeros(N + (what == "label count"), dtype=torch.int32 if what == "label dtype" else torch.int64,
                    device="cpu" if what == "cpu labels" else "cuda")
    said = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(ops, "_native_forward", lambda *a: None)
        with pytest.raises((RuntimeError, ValueError)) as e:
            linear_cross_entropy(x, y, w, -100, 0.0, -1.0 if what == "scale" else 1.0, 4096)
        said.append((type(e.value), str(e.value)))
    assert said[0] == said[1]


@pytest.mark.parametrize("always", [False, True])
def test_numbers_of_any_kind_for_the_function_itself(always):
    """linear_cross_entropy converts its numbers; the autograd Function takes them as they come."""
    import numpy as np

    from linear_cross_entropy_loss_amd import ops

    x = _mat(N, H, torch.bfloat16, 1).requires_grad_(True)
    w = _mat(H, V, torch.bfloat16, 2).requires_grad_(True)
    y = torch.randint(0, V, (N,), generator=torch.Generator().manual_seed(3)).cuda()
    ops.one_pass.set("always" if always else False)

    def run(*numbers):
        out = ops.LinearXentImplementation.apply(x, y, w, *numbers)
        return [o.detach() for o in out] + list(torch.autograd.grad(out[0], (x, w)))

    plain = run(-100, 1e-4, 0.5, 4096, True)
    for numbers in ((-100.0, np.float64(1e-4), np.float32(0.5), 4096.0, 1),
                    (torch.tensor(-100), torch.tensor(1e-4), torch.tensor(0.5), np.int64(4096), np.bool_(True))):
        for a, b in zip(plain, run(*numbers)):
            assert torch.allclose(a, b, rtol=1e-6)
