"""The module's native path (csrc/penc_torch.cpp) against the autograd functions of funcs.py, which the rest of
the suite holds to the oracle: same kernels, so the same bits wherever no atomics are involved."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def modules(d=3, cap=1 << 12, levels=5, feat=2, **kw):
    """Two modules with the same parameters: the native path, and one whose wrapper is a subclass (the functions of funcs.py)."""
    import permutohedral_encoding_amd as pe
    from permutohedral_encoding_amd import _native

    class Instrumented(_native.EncodingWrapper):
        pass

    torch.manual_seed(d + cap)
    sig = np.geomspace(1.0, 1e-2, levels)
    native, python = (pe.PermutoEncoding(d, cap, levels, feat, sig, **kw) for _ in range(2))
    with torch.no_grad():
        native.lattice_values.uniform_(-1, 1)
    python.load_state_dict(native.state_dict())
    python.lattice.__class__ = Instrumented
    assert python.lattice.calls_replaced() and not native.lattice.calls_replaced()
    return native, python


def close_sums(a, b):
    # the same fp32 terms, accumulated in another order: 2^-24 relative per term of sums of at most a few thousand
    assert torch.allclose(a, b, rtol=1e-4, atol=1e-6 * b.abs().max().item())


def upstreams(n, cols):
    """The layouts an upstream gradient arrives in: dense rows, padded rows, level-major, broadcast, every other row, odd stride."""
    g = torch.randn(n, cols, device="cuda")
    yield g
    yield torch.nn.functional.pad(g, (0, 4))[:, :cols]
    yield g.t().contiguous().t()
    yield torch.randn(1, 1, device="cuda").expand(n, cols)
    yield torch.randn(2 * n, cols, device="cuda")[::2]
    yield torch.nn.functional.pad(g, (0, 1))[:, :cols]


@pytest.mark.parametrize("d,n,feat,kw", [(3, 1, 2, {}), (3, 5001, 2, {}), (2, 700, 4, dict(concat_points=True)), (4, 513, 8, dict(contiguous_output=True)),
                                         (3, 2049, 2, dict(lattice_half_precision=True)), (8, 300, 2, dict(concat_points=True, contiguous_output=True))])
def test_native_path_equals_the_autograd_functions(d, n, feat, kw):
    native, python = modules(d, feat=feat, **kw)
    window = torch.tensor([1, 0.5, 1, 0, 1], dtype=torch.float64)  # on the host, in another type
    pts = torch.rand(n, d, device="cuda")
    with torch.no_grad():
        a, b = native(pts, window), python(pts, window)
    assert torch.equal(a, b) and a.shape == (n, native.output_dims()) and (n == 1 or a.stride() == b.stride()) and not a.requires_grad
    for up in upstreams(n, native.output_dims()):
        results = []
        for m in (native, python):
            m.lattice_values.grad = None
            p = pts.clone().requires_grad_(True)
            u = up.clone(memory_format=torch.preserve_format).requires_grad_(True) if up.stride(0) else up
            out = m(p, window)
            normal, = torch.autograd.grad(out, p, u, create_graph=True)
            assert m.lattice_values.grad is None
            (normal * normal).sum().backward()
            second = m.lattice_values.grad.clone()
            m.lattice_values.grad = None
            m(p, window).backward(up)
            results.append((normal.detach(), u.grad, p.grad, second, m.lattice_values.grad))
        (na, ua, pa, sa, fa), (nb, ub, pb, sb, fb) = results
        assert torch.equal(na, nb) and torch.equal(pa, pb)
        assert (ua is None and ub is None) or torch.equal(ua, ub)
        close_sums(sa, sb)
        close_sums(fa, fb)


def test_native_path_graph_rules():
    native, _ = modules()
    pts = torch.rand(300, 3, device="cuda", requires_grad=True)
    # a frozen table, positions that need no gradient, neither
    native.lattice_values.requires_grad_(False)
    assert not native(pts.detach()).requires_grad
    native(pts).sum().backward()
    assert native.lattice_values.grad is None and pts.grad is not None
    native.lattice_values.requires_grad_(True)
    out = native(pts.detach())
    out.sum().backward(retain_graph=True)
    once = native.lattice_values.grad.clone()
    out.sum().backward()
    close_sums(native.lattice_values.grad, 2 * once)
    # a graph that was freed says so
    out = native(pts)
    g, = torch.autograd.grad(out.sum(), pts, create_graph=True)
    g.sum().backward()
    with pytest.raises(RuntimeError, match="second time"):
        g.sum().backward()
    # errors arrive as the Python path raises them
    with pytest.raises(ValueError, match="0 points"):
        native(pts[:0])
    with pytest.raises(ValueError, match="pos dim"):
        native(pts[:, :2])
    with pytest.raises(ValueError, match="type float"):
        native(pts.double())
    with pytest.raises(ValueError, match="anneal_window"):
        native(pts, torch.ones(3))


@pytest.mark.parametrize("kw,normals", [({}, 1), (dict(sparse_table_grad=True), 1), (dict(lattice_half_precision=torch.bfloat16), 1),
                                        (dict(contiguous_output=True, concat_points=True), 1), ({}, 2), (dict(sparse_table_grad=True), 2)])
def test_losses_on_values_and_on_position_gradients_in_one_pass(kw, normals):
    """loss(values) + loss(normals) in one backward pass, which computes both table gradients in one scatter (one more for
    every further set of normals), against the autograd functions, which compute one after the other."""
    native, python = modules(levels=6, **kw)
    n = 3001
    pts = torch.rand(n, 3, device="cuda")
    ups = [torch.randn(n, native.output_dims(), device="cuda") for _ in range(normals)]
    qs = [torch.randn(n, 3, device="cuda") for _ in range(normals)]
    g = torch.randn(n, native.output_dims(), device="cuda")
    results = []
    for m in (native, python):
        p = pts.clone().requires_grad_(True)
        us = [u.clone().requires_grad_(True) for u in ups]
        out = m(p)
        grads = [torch.autograd.grad(out, p, u, create_graph=True)[0] for u in us]
        torch.autograd.backward([out] + grads, [g] + qs)
        table = m.table_grad.grad if m.sparse_table_grad else m.lattice_values.grad
        assert m.sparse_table_grad == (m.lattice_values.grad is None)
        results.append((table.clone(), p.grad, [u.grad for u in us]))
    (ta, pa, ua), (tb, pb, ub) = results
    close_sums(ta, tb)
    assert torch.equal(pa, pb) and all(torch.equal(x, y) for x, y in zip(ua, ub))


def test_native_path_refuses_what_the_autograd_functions_refuse():
    pts = torch.rand(300, 3, device="cuda")
    for m in modules():
        out = m(pts)
        out.sum().backward()
        with pytest.raises(RuntimeError, match="second time"):
            out.sum().backward()
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            m(pts).mul_(2.0).sum().backward()
        with torch.autograd.forward_ad.dual_level(), pytest.raises(RuntimeError, match="jvp|forward"):
            m(torch.autograd.forward_ad.make_dual(pts, torch.ones_like(pts)))
        with pytest.raises(RuntimeError):
            torch.func.grad(lambda x: m(x).sum())(pts)
        with pytest.raises(RuntimeError):
            torch.vmap(m)(pts[None])


def test_forward_mode_tangents_are_refused_and_not_dropped():
    """On an upstream gradient (dual weights of the layers after the encoding), on what comes back through a position gradient
    (with and without create_graph) and on the window."""
    fa = torch.autograd.forward_ad
    dual = lambda t: fa.make_dual(t, torch.ones_like(t))
    refused = lambda: pytest.raises(NotImplementedError, match="jvp|forward-mode")
    pts = torch.rand(300, 3, device="cuda")
    for m in modules():
        p, weights = pts.clone().requires_grad_(True), torch.randn(m.output_dims(), 1, device="cuda")
        for graph in (False, True):
            out = m(p)
            with fa.dual_level(), refused():
                torch.autograd.grad((out @ dual(weights)).sum(), p, create_graph=graph)
            with fa.dual_level(), refused():
                torch.autograd.grad(m(pts), m.lattice_values, dual(torch.ones_like(out)), create_graph=graph)
        for window in (torch.ones(5, device="cuda"), torch.ones(5), torch.ones(5, dtype=torch.float64)):
            with fa.dual_level(), refused():
                m(pts, dual(window))
            with fa.dual_level(), torch.no_grad(), refused():
                m(pts, dual(window))
    native, _ = modules()
    for graph in (False, True):
        for inputs in ([weights.requires_grad_(True)], [native.lattice_values], [native.lattice_values, weights]):
            normal, = torch.autograd.grad((native(p) @ weights).sum(), p, create_graph=True)
            with fa.dual_level(), refused():
                torch.autograd.grad(normal, inputs, dual(torch.ones_like(normal)), create_graph=graph)


def test_a_window_that_requires_a_gradient_gets_none_and_is_not_ignored():
    """Its result requires a gradient too, and a backward that nothing but the window asks for is refused."""
    pts = torch.rand(300, 3, device="cuda")
    for m in modules():
        window = torch.ones(5, device="cuda", requires_grad=True)
        m(pts, window).sum().backward()
        assert window.grad is None and m.lattice_values.grad is not None
        m.lattice_values.requires_grad_(False)
        out = m(pts, window)
        assert out.requires_grad
        with pytest.raises(AssertionError, match="neither lattice_values nor positions"):
            out.sum().backward()
        with torch.no_grad():
            assert not m(pts, window).requires_grad


def test_hooks_on_the_encoding_do_not_run_in_a_pass_through_its_position_gradient_alone():
    results = []
    for m in modules():
        p = torch.full((40, 3), 0.3, device="cuda", requires_grad=True)
        u = torch.ones(40, m.output_dims(), device="cuda", requires_grad=True)
        seen = []
        out = m(p)
        out.register_hook(lambda g: seen.append(1) or 2 * g)
        normal, = torch.autograd.grad(out, p, u, create_graph=True)
        assert seen == [1]
        normal.square().sum().backward()
        assert seen == [1]
        results.append((normal.detach(), u.grad))
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("rows", [True, False])
def test_saved_tensor_hooks_see_the_upstream_gradient(rows):
    native, _ = modules()
    p = torch.rand(500, 3, device="cuda", requires_grad=True)
    u = torch.randn(500, native.output_dims(), device="cuda")
    u = u if rows else u.t().contiguous().t()
    results, packed = [], []
    for hooks in (False, True):
        native.lattice_values.grad = None
        out = native(p)
        if hooks:
            with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(1) or t.cpu().contiguous(), lambda t: t.cuda()):
                normal, = torch.autograd.grad(out, p, u, create_graph=True)
        else:
            normal, = torch.autograd.grad(out, p, u, create_graph=True)
        normal.square().sum().backward()
        results.append(native.lattice_values.grad)
    assert packed
    close_sums(*results)


def test_a_window_in_host_memory_is_not_captured():
    native, _ = modules()
    pts, stream = torch.rand(300, 3, device="cuda"), torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.no_grad(), torch.cuda.stream(stream):
        native(pts, torch.ones(5))
        graph = torch.cuda.CUDAGraph()
        graph.capture_begin()
        with pytest.raises(RuntimeError, match="host memory"):
            native(pts, torch.ones(5))
        native(pts)
        graph.capture_end()
    torch.cuda.synchronize()


def test_a_module_moved_to_the_gpu_copies_its_scale_factors_once():
    native, _ = modules(device="cpu")
    assert native.fixed_params.m_scale_factor.device.type == "cpu"
    native.cuda()
    pts, stream = torch.rand(300, 3, device="cuda"), torch.cuda.Stream()
    want = native(pts)
    moved = native.fixed_params.m_scale_factor
    assert moved.is_cuda
    with torch.no_grad():
        native(pts)
    assert native.fixed_params.m_scale_factor is moved
    # a call that copied could not be captured
    stream.wait_stream(torch.cuda.current_stream())
    with torch.no_grad(), torch.cuda.stream(stream):
        native(pts)
        graph = torch.cuda.CUDAGraph()
        graph.capture_begin()
        out = native(pts)
        graph.capture_end()
        graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, want)


def test_upstream_gradient_modified_before_the_double_backward_is_refused():
    native, _ = modules()
    p = torch.rand(100, 3, device="cuda", requires_grad=True)
    up = torch.randn(native.output_dims(), 100, device="cuda").t()  # level-major: kept as it is
    normal, = torch.autograd.grad(native(p), p, up, create_graph=True)
    up.mul_(2.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        normal.sum().backward()


@pytest.mark.parametrize("concat", [False, True])
def test_rows_kept_as_a_copy_are_the_upstream_gradient(concat):
    """The level-major copy that is kept of rows, as a saved-tensor hook sees it: whole, the columns of concatenated points too; and
    changing the rows, or handing over ones that cannot be tracked, before the double backward is refused as if they had been kept."""
    for m in modules(concat_points=concat):
        p = torch.rand(4001, 3, device="cuda", requires_grad=True)
        up, seen = torch.randn(4001, m.output_dims(), device="cuda"), []
        fill = torch.full((4001, m.output_dims()), float("nan"), device="cuda")  # (what the copy's memory holds before)
        del fill
        with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t) or t, lambda t: t):
            out = m(p)
            seen.clear()
            normal, = torch.autograd.grad(out, p, up, create_graph=True)
        kept, = seen
        assert torch.equal(kept.permute(2, 0, 1).reshape(up.shape) if kept.dim() == 3 else kept, up)
        normal.sum().backward()
        normal, = torch.autograd.grad(m(p), p, up, create_graph=True)
        up.mul_(2.0)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            normal.sum().backward()
        with torch.inference_mode():
            untracked = up.clone()
        with pytest.raises(RuntimeError, match="Inference tensors cannot be saved for backward"):
            torch.autograd.grad(m(p), p, untracked, create_graph=True)


@pytest.mark.parametrize("d,n,levels,cap,rows,feat", [(2, 1, 3, 64, False, 2), (3, 511, 4, 1 << 12, True, 2), (3, 4097, 3, 1 << 20, False, 4), (4, 9000, 5, 50000, True, 2),
                                                      (5, 1025, 2, 1 << 14, False, 2), (6, 700, 2, 1 << 12, True, 2), (8, 5000, 3, 1 << 13, False, 2),
                                                      (3, 600000, 1, (1 << 22) + 5, True, 2)])
def test_both_orders_in_one_scatter_match_the_oracle(d, n, levels, cap, rows, feat):
    """penc_backward_both_orders at edges of tiles, groups and bin widths (more than 2^22 slots: wide bins) against the sum of the
    oracle's two table gradients, within the bound of any sum in another order: 1e-4 of the sum of magnitudes."""
    from helpers import assert_sum_close, make_encoding, random_problem, to_gpu
    from oracle import api as orc
    from permutohedral_encoding_amd import _native
    p = random_problem(d, n, levels, cap, seed=60 + d, sigma_range=(1.0, 1e-3), nr_feat=feat)
    first = np.random.default_rng(3).standard_normal((levels, feat, n)).astype(np.float32)
    enc, fp = make_encoding(d, p["sigmas"], p["shift"], nr_feat=feat)
    table, pos, win, dpos, first_t = (to_gpu(x) for x in (p["table"], p["pos"], p["window"], p["dpos"], first))
    grad = to_gpu(p["grad"].transpose(2, 0, 1).reshape(n, -1) if rows else p["grad"])
    lib = _native.lib()
    ws = torch.empty(lib.penc_scatter_workspace_bytes(d, n, levels * feat // 2, cap, 0) + 4 * feat * levels * n + 1024, dtype=torch.uint8, device="cuda")
    tg, pg = torch.full_like(table, float("nan")), torch.empty_like(pos)
    rc = lib.penc_backward_both_orders(d, feat, n, levels, cap, pos.data_ptr(), table.data_ptr(), 0, fp.m_scale_factor.data_ptr(),
                                       fp.m_random_shift_per_level.data_ptr(), win.data_ptr(), grad.data_ptr(), feat * levels if rows else 0,
                                       dpos.data_ptr(), first_t.data_ptr(), tg.data_ptr(), None, pg.data_ptr(), ws.data_ptr(), ws.numel(),
                                       torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    sf = orc.scale_factors(d, p["sigmas"])
    a = orc.backward_table(p["pos"], sf, p["shift"], p["window"], p["grad"], cap, want_abs=True)
    b = orc.double_backward(p["pos"], p["table"], sf, p["shift"], p["window"], p["dpos"], first, want_abs=True)
    assert_sum_close(tg.cpu().numpy(), a["grad64"] + b["grad64"], a["abs64"] + b["abs64"], 1e-4, "both table gradients")
    wp = orc.backward_pos(p["pos"], p["table"], sf, p["shift"], p["window"], p["grad"])
    assert np.all(np.abs(pg.cpu().numpy() - wp["grad64"]) <= 1e-6 * wp["abs64"] + 1e-30)


@pytest.mark.parametrize("n", [1, 24, 128, 129, 300])
def test_upload_carries_host_values_in_the_launch(n):
    from permutohedral_encoding_amd import _native
    host = torch.randn(n)
    want, dst = host.clone(), torch.full((n + 1,), 7.0, device="cuda")
    rc = _native.lib().penc_upload(host.data_ptr(), dst.data_ptr(), n, torch.cuda.current_stream().cuda_stream)
    host.zero_()  # the caller's array is its own again
    assert rc == 0 and torch.equal(dst[:n].cpu(), want) and dst[n].item() == 7.0


@pytest.mark.parametrize("d,n,levels,cap,feat,concat", [(3, 1, 5, 64, 2, True), (2, 63, 9, 1 << 10, 4, True), (3, 64, 24, 1 << 18, 2, False), (4, 65, 8, 1000, 8, False),
                                                        (8, 1003, 31, 1 << 10, 8, False), (5, 20001, 7, 1 << 12, 2, True), (6, 9001, 8, 1 << 18, 2, True)])
def test_all_levels_of_a_block_of_points(d, n, levels, cap, feat, concat):
    """Dense rows from the forward and from the grad-grad bit for bit, the position gradient of rows within its bound and its level-major
    copy bit for bit: one point, remainders of a block, fewer and more levels than waves, 248 columns, tables inside and beyond an L2."""
    from helpers import make_encoding, random_problem, to_gpu
    from oracle import api as orc
    from permutohedral_encoding_amd import _native
    p = random_problem(d, n, levels, cap, seed=80 + d, sigma_range=(1.0, 1e-3), nr_feat=feat)
    p["window"][levels // 2] = 0.0
    _, fp = make_encoding(d, p["sigmas"], p["shift"], concat_points=concat, nr_feat=feat)
    table, pos, win, dpos = (to_gpu(p[k]) for k in ("table", "pos", "window", "dpos"))
    extra = _native.extra_levels(d, feat, concat)
    cols, stride = feat * (levels + extra), feat * (levels + extra) + 2
    grad_rows = torch.zeros(n, stride, device="cuda")
    grad_rows[:, :feat * levels] = to_gpu(p["grad"].transpose(2, 0, 1).reshape(n, -1))
    lib, st = _native.lib(), torch.cuda.current_stream().cuda_stream
    head = (d, feat, n, levels, cap, pos.data_ptr(), table.data_ptr())
    params = (fp.m_scale_factor.data_ptr(), fp.m_random_shift_per_level.data_ptr(), win.data_ptr())
    ws = torch.empty(4 * cols * n + lib.penc_positions_workspace_bytes(d, n, levels) + 512, dtype=torch.uint8, device="cuda")
    sf = orc.scale_factors(d, p["sigmas"])
    rows = torch.full((n, stride), 7.0, device="cuda")
    assert lib.penc_forward_rowmajor(*head, *params, rows.data_ptr(), stride, int(concat), 0.5, ws.data_ptr(), ws.numel(), st) == 0
    want = orc.forward(p["pos"], p["table"], sf, p["shift"], p["window"], concat_points=concat, points_scaling=0.5)
    assert np.array_equal(rows[:, :cols].cpu().numpy(), want.transpose(2, 0, 1).reshape(n, cols)) and torch.all(rows[:, cols:] == 7.0)
    assert lib.penc_grad_grad_rowmajor(*head, 0, *params, dpos.data_ptr(), rows.data_ptr(), stride, int(concat), ws.data_ptr(), ws.numel(), st) == 0
    wd = orc.double_backward(p["pos"], p["table"], sf, p["shift"], p["window"], p["dpos"], p["grad"], concat_points=concat, want32=False, want64=False)
    assert np.array_equal(rows[:, :cols].cpu().numpy(), wd["ggs"].transpose(2, 0, 1).reshape(n, cols)) and torch.all(rows[:, cols:] == 7.0)
    copy, pg = torch.empty(feat * levels, n, device="cuda"), torch.empty_like(pos)
    assert lib.penc_backward_positions_rowmajor(*head, 0, *params, grad_rows.data_ptr(), stride, copy.data_ptr(), pg.data_ptr(),
                                                ws.data_ptr(), ws.numel(), st) == 0
    assert torch.equal(copy, grad_rows[:, :feat * levels].t())
    wp = orc.backward_pos(p["pos"], p["table"], sf, p["shift"], p["window"], p["grad"])
    assert np.all(np.abs(pg.cpu().numpy() - wp["grad64"]) <= 1e-6 * wp["abs64"] + 1e-30)


@pytest.mark.parametrize("d,n,levels,cap,feat,finest", [(3, 1, 24, 64, 2, 1e-3), (2, 511, 3, (1 << 12) + 1, 8, 1e-3), (3, 512, 9, 1 << 18, 2, 1e-3), (4, 513, 5, 50001, 4, 1e-3),
                                                        (8, 1025, 4, 1 << 20, 2, 1e-3), (3, 9001, 24, 1 << 16, 2, 0.5), (2, 20001, 4, 1000, 4, 0.3), (3, 65536, 16, 1 << 12, 2, 1e-2),
                                                        (5, 17000, 3, (1 << 22) - 3, 2, 1e-3), (5, 12000, 3, (1 << 22) - 3, 2, 1e-3), (4, 12289, 4, 1 << 14, 2, 0.2),
                                                        (3, 65537, 17, 1 << 14, 2, 1e-2), (8, 4101, 2, 1 << 12, 4, 0.4)])
def test_sorted_groups_give_the_table_gradient(d, n, levels, cap, feat, finest):
    """Table gradients of small batches, dense (over what the memory held) and added twice into a sparse one: edges of groups and of slot
    ranges, one range and 512, ranges narrower than a range of the touched map, levels of a few slots, a masked level; within the bound
    of any sum in another order, 1e-4 of the sum of magnitudes.  The position gradient goes through the level-major copy."""
    from helpers import assert_sum_close, make_encoding, random_problem, to_gpu
    from oracle import api as orc
    from permutohedral_encoding_amd import _native
    p = random_problem(d, n, levels, cap, seed=90 + d, sigma_range=(1.0, finest), nr_feat=feat)
    p["window"][levels // 2] = 0.0
    _, fp = make_encoding(d, p["sigmas"], p["shift"], nr_feat=feat)
    table, pos, win = (to_gpu(p[k]) for k in ("table", "pos", "window"))
    rows = to_gpu(p["grad"].transpose(2, 0, 1).reshape(n, -1))
    lib, st = _native.lib(), torch.cuda.current_stream().cuda_stream
    args = (d, feat, n, levels, cap, pos.data_ptr(), table.data_ptr(), fp.m_scale_factor.data_ptr(), fp.m_random_shift_per_level.data_ptr(),
            win.data_ptr(), rows.data_ptr(), feat * levels)
    ws = torch.empty(lib.penc_backward_rowmajor_workspace_bytes(d, feat, n, levels, cap, 1, 1), dtype=torch.uint8, device="cuda")
    tg, pg = torch.full_like(table, float("nan")), torch.empty_like(pos)
    assert lib.penc_backward_rowmajor(*args, tg.data_ptr(), pg.data_ptr(), ws.data_ptr(), ws.numel(), st) == 0
    sf = orc.scale_factors(d, p["sigmas"])
    want = orc.backward_table(p["pos"], sf, p["shift"], p["window"], p["grad"], cap, want_abs=True)
    assert_sum_close(tg.cpu().numpy(), want["grad64"], want["abs64"], 1e-4, "dense")
    wp = orc.backward_pos(p["pos"], p["table"], sf, p["shift"], p["window"], p["grad"])
    assert np.all(np.abs(pg.cpu().numpy() - wp["grad64"]) <= 1e-6 * wp["abs64"] + 1e-30)
    sums = torch.zeros_like(table)
    touched = torch.zeros(lib.penc_touched_map_entries(feat, levels, cap), dtype=torch.int32, device="cuda")
    for _ in range(2):
        assert lib.penc_backward_sparse(*args, sums.data_ptr(), touched.data_ptr(), None, ws.data_ptr(), ws.numel(), st) == 0
    assert_sum_close(sums.cpu().numpy(), 2 * want["grad64"], 2 * want["abs64"], 1e-4, "sparse")
    assert lib.penc_clear_touched(sums.data_ptr(), feat, levels, cap, touched.data_ptr(), st) == 0
    assert not sums.any() and not touched.any()


@pytest.mark.parametrize("d,n,levels,cap,feat", [(3, 16001, 24, 1 << 17, 2), (2, 40009, 13, 1 << 18, 4), (8, 10501, 16, 1 << 17, 2), (6, 6007, 65, 1 << 15, 2),
                                                 (3, 301, 130, 64, 2), (4, 255, 64, 128, 4)])
def test_position_gradient_groups_the_levels_a_window_leaves(d, n, levels, cap, feat):
    """Groups of the levels that are left: all, none, the last alone, every third, the coarse half; at 64 levels, beyond them, and as
    one group without a workspace; against the oracle within the bound of its 32-bit sums, 1e-6 of the sum of magnitudes."""
    from helpers import make_encoding, random_problem, to_gpu
    from oracle import api as orc
    from permutohedral_encoding_amd import _native
    p = random_problem(d, n, levels, cap, seed=110 + d, sigma_range=(1.0, 1e-2), nr_feat=feat)
    _, fp = make_encoding(d, p["sigmas"], p["shift"], nr_feat=feat)
    table, pos, grad = (to_gpu(p[k]) for k in ("table", "pos", "grad"))
    lib, st = _native.lib(), torch.cuda.current_stream().cuda_stream
    ws = torch.full((lib.penc_positions_workspace_bytes(d, n, levels),), 0xFF, dtype=torch.uint8, device="cuda")
    sf, k = orc.scale_factors(d, p["sigmas"]), np.arange(levels)
    for keep in (k >= 0, k < 0, k == levels - 1, k % 3 == 1, k < levels // 2):
        window = np.where(keep, p["window"], 0).astype(np.float32)
        win = to_gpu(window)
        want = orc.backward_pos(p["pos"], p["table"], sf, p["shift"], window, p["grad"])
        for memory in (ws, None):
            pg = torch.full_like(pos, float("nan"))
            assert lib.penc_backward(d, feat, n, levels, cap, pos.data_ptr(), table.data_ptr(), fp.m_scale_factor.data_ptr(),
                                     fp.m_random_shift_per_level.data_ptr(), win.data_ptr(), grad.data_ptr(), None, pg.data_ptr(),
                                     memory.data_ptr() if memory is not None else None, memory.numel() if memory is not None else 0, st) == 0
            assert np.all(np.abs(pg.cpu().numpy() - want["grad64"]) <= 1e-6 * want["abs64"] + 1e-30)


@pytest.mark.parametrize("levels,n", [(4, 95001), (5, 78063), (6, 65537), (15, 26240), (16, 25001), (33, 12353)])
def test_rows_and_levels_change_places(levels, n):
    """8 to 66 columns (two, four and eight loads of a thread together, with and without remainders), odd row counts: the level-major
    copy of rows and back, and rows of a forward whose table is too large for the kernels that need no transpose, bit for bit."""
    from permutohedral_encoding_amd import _native
    lib, st = _native.lib(), torch.cuda.current_stream().cuda_stream
    cols, cap = 2 * levels, 1 << 19
    rows, back = torch.randn(n, cols, device="cuda"), torch.empty(cols, n, device="cuda")
    assert lib.penc_transpose(rows.data_ptr(), back.data_ptr(), n, cols, st) == 0 and torch.equal(back, rows.t())
    fp = _native.EncodingFixedParams(3, cap, levels, 2, np.geomspace(1.0, 1e-3, levels).astype(np.float32), torch.randn(levels, 3, device="cuda"), False, 1.0)
    pos, table, win = torch.rand(n, 3, device="cuda"), torch.randn(levels, cap, 2, device="cuda"), torch.ones(levels, device="cuda")
    args = (3, 2, n, levels, cap, pos.data_ptr(), table.data_ptr(), fp.m_scale_factor.data_ptr(), fp.m_random_shift_per_level.data_ptr(), win.data_ptr())
    ws = torch.empty(lib.penc_forward_rowmajor_workspace_bytes(3, 2, n, levels, 0), dtype=torch.uint8, device="cuda")
    out, dense = torch.empty(cols, n, device="cuda"), torch.full((n, cols + 2), 7.0, device="cuda")
    assert lib.penc_forward(*args, out.data_ptr(), 0, 1.0, st) == 0
    assert lib.penc_forward_rowmajor(*args, dense.data_ptr(), cols + 2, 0, 1.0, ws.data_ptr(), ws.numel(), st) == 0
    assert torch.equal(dense[:, :cols], out.t()) and torch.all(dense[:, cols:] == 7.0)
