"""GPU tests of dispatch branches that a size, a value range or the calling mode selects, at the sizes where they can go wrong."""
import pytest
import torch

from helpers import make_inputs, rel_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mode", ["no_grad", "inference", "detached"])
def test_loss_without_gradients_allocates_no_gradients(mode, dtype):
    """A parameter under no_grad needs no gradient: the call computes the loss alone and takes less memory than a weight
    gradient would, also where a call that needs gradients computes them along with the loss."""
    from linear_cross_entropy_loss_amd import LinearCrossEntropyLoss, _lib, ops

    N, H, V = 300, 256, 8192
    x, y, w = make_inputs(N, H, V, dtype, 3, ignore_frac=0.1, device="cuda")
    mod = LinearCrossEntropyLoss(H, V, device="cuda", dtype=dtype, ignore_index=-1, init_method=lambda t: t.data.copy_(w))
    mod.monitoring = True
    if dtype == torch.bfloat16:  # (fp32 activations have no such route)
        prob = _lib.make_problem(N, H, V, H, V, H, V, dtype, dtype, dtype, dtype, -1, 1.0, 0.0, mod.N_chunk_size, True, 0,
                                 _lib.PACK_AUTO, 0, _lib.W_HV, _lib.ROUTE_ONE_PASS)
        assert _lib.forward_backward_plan(prob)[0] > 0
    token = ops.one_pass.set("always")
    try:
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
    finally:
        ops.one_pass.reset(token)
    assert not loss.requires_grad
    # (the same fp32 logits; sums over columns cut at other places)
    assert torch.allclose(loss, want, rtol=1e-6, atol=0)
    assert torch.allclose(mod.latest_metrics["logit_max"], want_max, rtol=1e-6, atol=0)
    if dtype == torch.bfloat16:
        assert torch.cuda.max_memory_allocated() - before < H * V * 2


@pytest.mark.parametrize("transform, error, message", [("forward_ad", NotImplementedError, "jvp"),
                                                       ("vmap", RuntimeError, "setup_context staticmethod")])
def test_loss_without_gradients_refuses_transforms(transform, error, message):
    """Also where no input needs a gradient: a tangent is not dropped and a batch dimension not misread, the call is refused as
    the autograd Function refuses it."""
    from linear_cross_entropy_loss_amd import linear_cross_entropy

    x, y, w = make_inputs(64, 64, 256, torch.bfloat16, 3, device="cuda")
    with torch.no_grad(), pytest.raises(error, match=message):
        if transform == "vmap":
            torch.func.vmap(lambda xx: linear_cross_entropy(xx, y, w)[0])(x[None])
        else:
            with torch.autograd.forward_ad.dual_level():
                linear_cross_entropy(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)), y, w)


# full tile columns and the one that straddles the vocabulary's end in one launch: tile counts around multiples of the 256
# compute units (a last round of full tiles that is empty, full but one, all but empty; more tail tiles than workgroups)
@pytest.mark.parametrize("route", [False, "always"])
@pytest.mark.parametrize("N,V", [(100, 256 * 256 + 8), (100, 255 * 256 + 1), (300, 128 * 256 + 255), (300, 129 * 256 + 8), (66000, 264)])
def test_tail_column_in_the_launch_of_the_full_ones(N, V, route):
    from linear_cross_entropy_loss_amd import linear_cross_entropy, ops
    from oracle import lce_forward_backward_fp64

    H = 72
    x, y, w = make_inputs(N, H, V, torch.bfloat16, 5, ignore_frac=0.05, device="cuda")
    x.requires_grad_()
    w.requires_grad_()
    token = ops.one_pass.set(route)
    try:
        loss = linear_cross_entropy(x, y, w, -1, 1e-3, 1.0, 4096)[0]
        gx, gw = torch.autograd.grad(loss, (x, w))
    finally:
        ops.one_pass.reset(token)
    ref = lce_forward_backward_fp64(x.detach(), y, w.detach(), -1, 1e-3, 1.0, chunk=4096)
    assert abs(loss.item() - ref.loss.item()) <= 1e-5 * ref.loss.item()
    # (bf16: dz, dx and dW are rounded to 8 bits of mantissa, at most 2^-8 relative to the largest entry each)
    for got, want in ((gx, ref.dx), (gw, ref.dw)):
        emax, el2 = rel_errors(got, want)
        assert emax < 2e-2 and el2 < 5e-3


# packing in one launch: token counts around a wave, the sizes its three variants end at, and the first one that takes four launches
@pytest.mark.parametrize("N", [1, 63, 64, 65, 255, 4096, 4097, 16384, 16385, 32768, 32769])
@pytest.mark.parametrize("ignored", [0.0, 0.3, 1.0])
def test_packing_counts_and_order(N, ignored):
    """Rows packed or not: the same loss, lse order and dx; dropped tokens get zeros."""
    from linear_cross_entropy_loss_amd import _lib, linear_cross_entropy, ops

    H, V = 64, 512
    x, y, w = make_inputs(N, H, V, torch.bfloat16, 7, ignore_frac=ignored, device="cuda")
    if ignored == 1.0:
        y = torch.full_like(y, -1)
    got = {}
    for mode in (_lib.PACK_ALWAYS, _lib.PACK_NEVER):
        token, route = ops.pack_rows.set(mode), ops.one_pass.set("always")
        try:
            x.grad = None
            xx = x.detach().requires_grad_()
            loss = linear_cross_entropy(xx, y, w, -1, 0.0, 1.0, 65536)[0]
            lse = torch.ops.lce_amd.forward(x, y, w, -1, 0.0, 1.0, 65536, False, mode)[1]
            got[mode] = (loss.detach(), torch.autograd.grad(loss, xx)[0], lse)
        finally:
            ops.pack_rows.reset(token)
            ops.one_pass.reset(route)
    (la, da, lse_a), (lb, db, lse_b) = got[_lib.PACK_ALWAYS], got[_lib.PACK_NEVER]
    assert not lse_a[y == -1].any() and not lse_b[y == -1].any()
    # (the same logits and the same slices of columns, in tiles at other places: the last bit of an exponential's argument)
    assert torch.allclose(lse_a, lse_b, rtol=1e-6, atol=0)
    if ignored == 1.0:
        assert torch.isnan(la) and torch.isnan(lb) and not da.any() and not db.any()
        return
    # (the same logits; sums of N terms in fp64, rounded once to fp32)
    assert abs(la.item() - lb.item()) <= 1e-6 * abs(lb.item())
    assert torch.equal(da[y == -1], torch.zeros_like(da[y == -1]))
    # (each row's K sums are the same, cut into segments at other places: one bf16 rounding apart)
    assert torch.allclose(da.float(), db.float(), rtol=2.0 ** -7, atol=1e-7)


# around a wave, a workgroup and the 8192 labels of one trip; powers of two and their neighbours; the last size of one workgroup
# and the first of several, and of more than one trip of theirs
@pytest.mark.parametrize("N", [1, 64, 1023, 1024, 1025, 8191, 8192, 8193, 65536, 100003, 131072, 131073, 2097153])
def test_stand_in_gradient_is_the_power_of_two_below_the_count(N):
    from linear_cross_entropy_loss_amd import ops

    x = torch.empty((1, 8), dtype=torch.float16, device="cuda")
    for kept in sorted({0, 1, N // 3, N - 1, N}):
        y = torch.arange(N, device="cuda")
        y[kept:] = -1
        y = y.flip(0).contiguous()
        want = 2.0 ** (max(kept, 1).bit_length() - 1)
        assert ops._stand_in_gradient(x, y, -1).tolist() == [want]


def test_stand_in_gradient_of_many_labels_takes_the_whole_chip():
    """2^24 labels are 128 MiB: 4.6 ms through one compute unit, 0.1 ms through all of them and their launches."""
    from linear_cross_entropy_loss_amd import ops

    x = torch.empty((1, 8), dtype=torch.float16, device="cuda")
    y = torch.zeros(1 << 24, dtype=torch.int64, device="cuda")
    times = []
    for _ in range(5):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        pre = ops._stand_in_gradient(x, y, -1)
        end.record()
        end.synchronize()
        times.append(start.elapsed_time(end))
    assert pre.item() == 2.0 ** 24
    assert min(times) < 1.0  # ms: ten times the one, a quarter of the other


# row lengths around a 16-byte piece, the threads of a row and their four pieces each; sources at odd addresses
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows, cols", [(1, 1), (3, 7), (5, 257), (33, 511), (257, 1021), (2, 8191), (9, 50257)])
@pytest.mark.parametrize("offset, extra", [(0, 0), (1, 0), (3, 2)])
def test_padded_copy_of_rows(dtype, rows, cols, offset, extra):
    from linear_cross_entropy_loss_amd import ops

    flat = torch.randn(offset + rows * (cols + extra), device="cuda").to(dtype)
    t = flat[offset:].view(rows, cols + extra)[:, :cols]
    out = ops._aligned_rows(t)
    assert out.data_ptr() % 16 == 0 and out.stride(0) * out.element_size() % 16 == 0 and torch.equal(out, t)
    if out.data_ptr() != t.data_ptr():
        whole = torch.as_strided(out, (rows, out.stride(0)), (out.stride(0), 1))
        assert not whole[:, cols:].any()


# matrices that lie transposed: one element, edges of the 64 x 64 tiles and of 16-byte pieces, more tiles than workgroups; rows that
# start anywhere, padded rows, and a stride between them that no kernel takes
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,cols,ld", [(1, 1, 1), (1, 65, 1), (63, 64, 63), (64, 63, 64), (65, 129, 65), (481, 1003, 481),
                                          (100, 72, 104), (7, 33, 9), (3, 70000 * 64, 3), (200, 100, 199)])
def test_copies_of_transposed_matrices(rows, cols, ld, dtype):
    from linear_cross_entropy_loss_amd import ops

    g = torch.Generator(device="cuda").manual_seed(rows + cols)
    store = torch.randn(cols * ld + rows + 1, generator=g, device="cuda").to(dtype)
    t = torch.as_strided(store, (rows, cols), (1, ld), 1)  # (ld < rows: rows that overlap, copied element by element)
    out = ops._aligned_rows(t)
    assert out.data_ptr() % 16 == 0 and out.stride(0) * out.element_size() % 16 == 0 and torch.equal(out, t)
    assert not torch.as_strided(out, (rows, out.stride(0)), (out.stride(0), 1))[:, cols:].any()


# row merge and final sums: one token, a workgroup's 64 and their neighbours, more blocks than one trip of the final sums takes;
# one slice of 128 columns, less and more than the 16 groups, and than the 128 slices of one trip; the last token counts that one
# workgroup merges by itself, the slices up to which it does, and the first beyond
@pytest.mark.parametrize("N,V", [(1, 1), (63, 129), (64, 2048), (64, 40000), (65, 2049), (256, 16384), (256, 16385), (257, 16384),
                                 (300, 16385), (130, 40000), (9000, 1000), (70000, 300)])
@pytest.mark.parametrize("route", [False, "always"])
def test_row_merge_and_final_sums(N, V, route):
    from linear_cross_entropy_loss_amd import linear_cross_entropy, ops

    H = 64
    x, y, w = make_inputs(N, H, V, torch.bfloat16, 11, ignore_frac=0.1 if N > 1 else 0.0, device="cuda")
    token = ops.one_pass.set(route)
    try:
        got = linear_cross_entropy(x.clone().requires_grad_(), y, w, -1, 1e-3, 1.0, 65536, True)
    finally:
        ops.one_pass.reset(token)
    z = x.double() @ w.double()
    lse = torch.logsumexp(z, 1)
    kept = y != -1
    zr = (lse[kept] ** 2).mean()
    loss = (lse[kept] - z[kept].gather(1, y[kept, None])[:, 0]).mean() + 1e-3 * zr
    ent = lse - (torch.exp(z - lse[:, None]) * z).sum(1)
    want = (loss, zr, z.max(), ent[kept].mean(), z.norm(dim=1).mean())
    # (logits are fp32 sums of 64 exact products, each sum over columns one of fp32 terms: 2^-24 times the number of additions
    # in a chain, some tens, of the size of lse; the totals over tokens are formed in fp64)
    scale = max(1.0, lse.abs().max().item())
    for a, b in zip(got, want):
        assert abs(a.item() - b.item()) <= 1e-5 * max(scale, abs(b.item()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("route", [False, "always"])
def test_consumer_that_passes_no_gradient_gives_zeros(route, dtype):
    """A loss whose consumer returns None for its gradient has gradients of zero, not none."""
    from linear_cross_entropy_loss_amd import linear_cross_entropy, ops

    class Drop(torch.autograd.Function):
        @staticmethod
        def forward(ctx, t):
            return t.clone()

        @staticmethod
        def backward(ctx, grad):
            return None

    x, y, w = make_inputs(70, 72, 300, dtype, 3, device="cuda")
    x.requires_grad_()
    w.requires_grad_()
    token = ops.one_pass.set(route)
    try:
        loss = linear_cross_entropy(x, y, w)[0]
        gx, gw = torch.autograd.grad(Drop.apply(loss), (x, w))
    finally:
        ops.one_pass.reset(token)
    assert gx.shape == x.shape and gw.shape == w.shape and not gx.any() and not gw.any()


# fp32 rows of an odd number of 16-byte pieces, whose gradients are dense: one column piece, the edge of a tile and beyond, with
# chunks whose sums are added in the gradient itself (master weight) and without
@pytest.mark.parametrize("N,H,V,n_chunk", [(70, 4, 12, 4096), (300, 260, 1004, 4096), (1500, 252, 2052, 512), (600, 516, 508, 256)])
@pytest.mark.parametrize("x_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("route", [False, "always"])
def test_dense_fp32_gradients(N, H, V, n_chunk, x_dtype, route):
    from linear_cross_entropy_loss_amd import linear_cross_entropy, ops
    from oracle import lce_forward_backward_fp64

    x, y, w = make_inputs(N, H, V, x_dtype, 5, ignore_frac=0.05, w_dtype=torch.float32, device="cuda")
    x.requires_grad_()
    w.requires_grad_()
    token = ops.one_pass.set(route)
    try:
        loss = linear_cross_entropy(x, y, w, -1, 0.0, 1.0, n_chunk)[0]
        gx, gw = torch.autograd.grad(loss, (x, w))
    finally:
        ops.one_pass.reset(token)
    assert gw.stride() == (V, 1) and (x_dtype != torch.float32 or gx.stride() == (H, 1))
    w_used = w.detach() if x_dtype == torch.float32 else w.detach().to(x_dtype)  # (rounded once under 16-bit activations)
    ref = lce_forward_backward_fp64(x.detach(), y, w_used, -1, 0.0, 1.0, chunk=n_chunk)
    # (fp32: products of bf16 pairs, 2^-16 relative to each operand, so some 2^-15 of the 2-norm; bf16: as above)
    for got, want in ((gx, ref.dx), (gw, ref.dw)):
        assert rel_errors(got, want)[1] < (3e-5 if x_dtype == torch.float32 else 5e-3)


# Logit kernels on 128 x 128 tiles against the persistent ones, which a limit on the workgroups of a launch asks for: halves and
# quarters of a tile that do not exist, vocabularies that end in any slice, hidden sizes that end in any K tile, one workgroup and
# as many as the rule allows, both layouts, monitoring, pairs.
SMALL_TILE_CASES = [
    # N, H, V, dtype, monitoring, (V, H), ignored
    (1, 8, 1, torch.bfloat16, False, 0, 0.0), (127, 72, 127, torch.float16, True, 0, 0.1), (128, 64, 128, torch.bfloat16, False, 1, 0.0),
    (129, 200, 129, torch.bfloat16, True, 1, 0.2), (255, 130, 257, torch.float32, True, 0, 0.1), (257, 128, 255, torch.float16, False, 0, 0.0),
    (300, 1000, 1001, torch.bfloat16, False, 0, 0.3), (300, 104, 4000, torch.float32, False, 0, 0.0), (1, 4, 300, torch.float32, False, 0, 0.0),
    (2048, 256, 4096, torch.bfloat16, False, 0, 0.1), (4096, 2048, 2048, torch.float16, False, 1, 0.0), (100, 320, 70000, torch.bfloat16, True, 0, 0.1),
]


@pytest.mark.parametrize("route", ["two_pass", "one_pass"])
@pytest.mark.parametrize("N,H,V,dtype,mon,layout,ignored", SMALL_TILE_CASES)
def test_small_logit_tiles_match_the_persistent_kernels(N, H, V, dtype, mon, layout, ignored, route):
    import ctypes

    from linear_cross_entropy_loss_amd import _lib, ops

    lib = _lib.load()
    x, y, w = make_inputs(N, H, V, dtype, 17, ignore_frac=ignored, device="cuda")
    y[0] = V - 1
    x, w = ops._aligned_rows(x), ops._aligned_rows(w.t().contiguous() if layout else w)
    outs = []
    for limit in (0, torch.cuda.get_device_properties(0).multi_processor_count - 1):
        dx, dw = ops._empty_rows(N, H, dtype, "cuda"), ops._empty_rows(*w.shape, dtype, "cuda")
        prob = _lib.make_problem(N, H, V, x.stride(0), w.stride(0), dx.stride(0), dw.stride(0), dtype, dtype, dtype, dtype, -1, 1.5, 1e-3,
                                 65536, mon, 0, _lib.PACK_NEVER, limit, layout,
                                 _lib.ROUTE_ONE_PASS if route == "one_pass" else _lib.ROUTE_TWO_PASS)
        if route == "one_pass" and _lib.forward_backward_plan(prob)[0] == 0:
            pytest.skip("no such route for this problem")
        nbytes = _lib.forward_backward_workspace_bytes(prob)
        ws = torch.full((nbytes,), 0xff, dtype=torch.uint8, device="cuda")  # (NaN wherever it is read unwritten)
        lse, out5 = torch.full((N,), 7.0, device="cuda"), torch.zeros(5, device="cuda")
        nv, g = torch.zeros(1, dtype=torch.int64, device="cuda"), torch.ones(1, device="cuda")
        rc = lib.lce_forward_backward(ctypes.byref(prob), x.data_ptr(), w.data_ptr(), y.data_ptr(), g.data_ptr(), lse.data_ptr(),
                                      out5.data_ptr(), nv.data_ptr(), dx.data_ptr(), dw.data_ptr(), ws.data_ptr(), nbytes,
                                      torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        torch.cuda.synchronize()
        outs.append((lse, out5, nv, dx, dw))
    (lse, out5, nv, dx, dw), (lse_p, out5_p, nv_p, dx_p, dw_p) = outs
    # each logit is one accumulator's sum in the order of K, and a slice's sums are formed alike: the same bit for bit.  (dx and dW
    # have the workgroups that the limit leaves, and cut along K accordingly: fp32 sums of terms of one rounding, in another order,
    # and an fp32 sum next to the boundary of a 16-bit rounding may fall to either side, 2^-8 of it in bf16.)
    assert nv.item() == nv_p.item() == int((y != -1).sum())
    assert torch.equal(lse, lse_p) and torch.equal(out5, out5_p)
    for got, want in ((dx, dx_p), (dw, dw_p)):
        assert not torch.isnan(got).any()
        if want.double().norm() > 0:
            assert rel_errors(got, want)[1] <= (1e-6 if dtype == torch.float32 else 1e-3)
        else:
            assert not got.any()


# both gradients times one factor in one launch: either absent, types apart, rows that end inside a 16-byte piece, one element, a
# factor and a quotient of 1 (nothing touched), fp32 products rounded once more to the type
@pytest.mark.parametrize("shapes,dtypes", [(((1, 1), None), (torch.bfloat16, None)), (((37, 101), (5, 260)), (torch.bfloat16, torch.float32)),
                                           ((None, (300, 7)), (None, torch.float16)), (((70, 1003), (1003, 70)), (torch.float16, torch.float16))])
@pytest.mark.parametrize("factor,divisor", [(1.0, None), (0.37, None), (4096.0, 4096.0), (3.0, 7.0)])
def test_both_gradients_scaled_in_one_launch(shapes, dtypes, factor, divisor):
    from linear_cross_entropy_loss_amd import ops

    gen = torch.Generator(device="cuda").manual_seed(5)
    ts = []
    for shape, dtype in zip(shapes, dtypes):
        if shape is None:
            ts.append(None)
            continue
        t = ops._empty_rows(*shape, dtype, "cuda")
        torch.as_strided(t, (shape[0], t.stride(0)), (t.stride(0), 1)).fill_(7.0)
        t.copy_(torch.randn(shape, generator=gen, device="cuda"))
        ts.append(t)
    g = torch.full((), factor, device="cuda")
    d = None if divisor is None else torch.full((1,), divisor, device="cuda")
    f = g if d is None else g / d[0]
    want = [None if t is None else (t.float() * f).to(t.dtype) for t in ts]
    ops._scale_grads(*ts, g, d)
    for t, w in zip(ts, want):
        if t is not None:
            assert torch.equal(t, w)
            assert (torch.as_strided(t, (t.shape[0], t.stride(0)), (t.stride(0), 1))[:, t.shape[1]:] == 7.0).all()


# dx and dW launches whose plan has nothing to cut along K (as many tiles as workgroups, K too short), more workgroups than items, and no
# item at all (every label ignored): the fetch stream of every workgroup ends past the last item of its launch
@pytest.mark.parametrize("route", ["always", False])
@pytest.mark.parametrize("N,H,V,dtype,ignored", [
    (4096, 4096, 2304, torch.bfloat16, 0.0), (300, 512, 1024, torch.bfloat16, 0.0), (300, 512, 1024, torch.float32, 0.0),
    (2100, 300, 2100, torch.float16, 0.2), (600, 1100, 4096, torch.bfloat16, 1.0), (600, 72, 4096, torch.float32, 1.0),
])
def test_launches_without_work_cut_along_k(N, H, V, dtype, ignored, route):
    from linear_cross_entropy_loss_amd import linear_cross_entropy, ops

    x, y, w = make_inputs(N, H, V, dtype, 23, ignore_frac=ignored, device="cuda")
    x, w = x.requires_grad_(), w.requires_grad_()
    token = ops.one_pass.set(route)
    try:
        loss = linear_cross_entropy(x, y, w, -1)[0]
        dx, dw = torch.autograd.grad(loss, (x, w))
    finally:
        ops.one_pass.reset(token)
    keep = y != -1
    if not keep.any():
        assert torch.isnan(loss) and not dx.any() and not dw.any()
        return
    xd, wd = x.detach().double(), w.detach().double()
    p = torch.softmax(xd @ wd, 1)
    p[torch.arange(N, device="cuda"), y.clamp(min=0)] -= 1
    p *= keep[:, None] / keep.sum()
    # (the operator's tolerance of gradients in 16 bits; pairs: 2^-16 relative to each operand, some 2^-15 of the 2-norm)
    for got, want in ((dx, p @ wd.t()), (dw, xd.t() @ p)):
        assert rel_errors(got, want)[1] < (3e-5 if dtype == torch.float32 else 5e-3)
