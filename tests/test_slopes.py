"""Position derivatives from the slopes a forward keeps (penc_forward_slopes and what reads them), against fp64 sums over the
oracle's simplices, and the module's rules for keeping them."""
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def exact_slopes(p, sf, capacity):
    """-> (slope, magnitude) [levels][feat][d][n] in fp64: slope[k] = sf[k]/(d+1) * (sum_{i<=k} e[i] - (k+1) e[k+1]) with e[i] the difference of
    the two vertices whose weights the coordinate of rank m raises and lowers; `magnitude` is the same sum of absolute values."""
    from oracle import api as orc
    s = orc.simplex(p["pos"], sf, p["shift"], capacity)
    rank, slot = s["rank"].astype(np.int64), s["slot"].astype(np.int64)
    levels, n, d1 = rank.shape
    d, feat = d1 - 1, p["table"].shape[2]
    slope, mag = np.zeros((levels, feat, d, n)), np.zeros((levels, feat, d, n))
    for l in range(levels):
        v = p["table"][l].astype(np.float64)[slot[l]]  # (n, d+1, feat)
        by_rank = np.stack([v[:, d - m] - v[:, (d1 - m) % d1] for m in range(d1)], 1)
        e = np.take_along_axis(by_rank, rank[l][:, :, None], 1)
        for k in range(d):
            scale = float(sf[l, k]) / d1
            slope[l, :, k] = scale * (e[:, :k + 1].sum(1) - (k + 1) * e[:, k + 1]).T
            mag[l, :, k] = scale * (np.abs(e[:, :k + 1]).sum(1) + (k + 1) * np.abs(e[:, k + 1])).T
    return slope, mag


@pytest.mark.parametrize("d,n,levels,cap,feat,concat,fmt", [(3, 1, 5, 64, 2, True, 0), (2, 63, 9, 1 << 10, 4, True, 0), (3, 64, 24, 1 << 18, 2, False, 0),
                                                            (4, 65, 8, 1000, 8, False, 0), (8, 1003, 31, 1 << 10, 8, False, 0), (5, 20001, 7, 1 << 12, 2, True, 0),
                                                            (6, 4097, 3, 1 << 12, 4, True, 0), (7, 777, 8, 1 << 14, 2, False, 1), (3, 5000, 17, 1 << 14, 2, True, 2),
                                                            (8, 56001, 24, 1 << 10, 2, False, 0), (3, 30001, 24, 1 << 16, 2, True, 0)])
def test_derivatives_from_slopes(d, n, levels, cap, feat, concat, fmt):
    """One point, remainders of a tile, fewer and more levels than waves, 248 columns (80 and 102 KB of LDS), a masked level, padded rows, 16-bit
    tables; the result level by level and in rows, which a forward of these sizes brings out of workgroups of 64 points, or by a transpose."""
    from helpers import make_encoding, random_problem, to_gpu
    from oracle import api as orc
    from permutohedral_encoding_amd import _native
    p = random_problem(d, n, levels, cap, seed=40 + d, sigma_range=(1.0, 1e-3), nr_feat=feat)
    p["window"][levels // 2] = 0.0
    half = {0: None, 1: torch.float16, 2: torch.bfloat16}[fmt]
    table = to_gpu(p["table"]) if half is None else to_gpu(p["table"]).to(half)
    p["table"] = table.float().cpu().numpy()
    _, fp = make_encoding(d, p["sigmas"], p["shift"], concat_points=concat, nr_feat=feat)
    pos, win, dpos, grad = (to_gpu(p[k]) for k in ("pos", "window", "dpos", "grad"))
    sf = orc.scale_factors(d, p["sigmas"])
    extra = _native.extra_levels(d, feat, concat)
    encoded, cols = feat * levels, feat * (levels + extra)
    stride = cols + 2
    lib, st = _native.lib(), torch.cuda.current_stream().cuda_stream
    slopes = torch.full((levels * -(-n // 64) * 64 * d * feat,), float("nan"), device="cuda")  # what is not written must not be read
    out, rows = torch.empty(cols, n, device="cuda"), torch.full((n, stride), 7.0, device="cuda")
    kept = []
    for to_rows in (None, rows.data_ptr()):
        slopes.fill_(float("nan"))
        assert lib.penc_forward_slopes(d, feat, n, levels, cap, pos.data_ptr(), table.data_ptr(), fmt, fp.m_scale_factor.data_ptr(),
                                       fp.m_random_shift_per_level.data_ptr(), win.data_ptr(), out.data_ptr(), to_rows, stride,
                                       slopes.data_ptr(), int(concat), 0.5, st) == 0
        want = orc.forward(p["pos"], p["table"], sf, p["shift"], p["window"], concat_points=concat, points_scaling=0.5).reshape(cols, n)
        assert np.array_equal(out.cpu().numpy(), want)
        kept.append(slopes.clone())
    assert torch.allclose(*kept, rtol=0, atol=0, equal_nan=True)
    assert np.array_equal(rows[:, :cols].cpu().numpy(), want.T) and torch.all(rows[:, cols:] == 7.0)

    slope, mag = exact_slopes(p, sf, cap)
    w = p["window"].astype(np.float64)[:, None, None, None]
    u = 2.0 ** -24
    # a slope: one rounding per difference, up to d per sum, one of the product (its factor is exact to 2^-46): d + 2; then one per product
    # and sum.  Terms of a position gradient: levels x feat, added one by one at worst.
    g = p["grad"].astype(np.float64)[:, :, None, :]
    want_pos, bound_pos = (g * w * slope).sum((0, 1)).T, ((d + 4 + levels * feat) * u * np.abs(g * w) * mag).sum((0, 1)).T
    q = p["dpos"].astype(np.float64).T[None, None]
    want_gg, bound_gg = (q * w * slope).sum(2).reshape(encoded, n), ((2 * d + 4) * u * np.abs(q * w) * mag).sum(2).reshape(encoded, n)

    grad_rows = torch.full((n, stride), float("nan"), device="cuda")
    grad_rows[:, :encoded] = grad.reshape(encoded, n).t()
    for given, grad_stride, copy in ((grad, 0, None), (grad_rows, stride, None), (grad_rows, stride, torch.empty(encoded, n, device="cuda"))):
        pg = torch.full((n, d), float("nan"), device="cuda")
        assert lib.penc_backward_positions_slopes(d, feat, n, levels, slopes.data_ptr(), win.data_ptr(), given.data_ptr(), grad_stride,
                                                  None if copy is None else copy.data_ptr(), pg.data_ptr(), st) == 0
        assert np.all(np.abs(pg.cpu().numpy() - want_pos) <= bound_pos + 1e-30)
        assert copy is None or torch.equal(copy, grad.reshape(encoded, n))
    level_major = torch.full((cols, n), float("nan"), device="cuda")
    rows.fill_(7.0)
    for to, row_stride in ((level_major, 0), (rows, stride)):
        assert lib.penc_grad_grad_slopes(d, feat, n, levels, slopes.data_ptr(), win.data_ptr(), dpos.data_ptr(), to.data_ptr(), row_stride,
                                         int(concat), st) == 0
    assert torch.equal(level_major, rows[:, :cols].t()) and torch.all(rows[:, cols:] == 7.0) and torch.all(level_major[encoded:] == 0.0)
    assert np.all(np.abs(level_major[:encoded].cpu().numpy() - want_gg) <= bound_gg + 1e-30)
    # refused: odd row strides (pairs of columns are read together), rows of more than 255 columns
    assert lib.penc_backward_positions_slopes(d, feat, n, levels, slopes.data_ptr(), win.data_ptr(), grad_rows.data_ptr(), encoded + 1, None,
                                              pg.data_ptr(), st) != 0
    assert lib.penc_grad_grad_slopes(d, feat, n, 256 // feat, slopes.data_ptr(), win.data_ptr(), dpos.data_ptr(), rows.data_ptr(), 300, 0, st) != 0


N, CAP, LEVELS = 60001, 1 << 19, 8  # gathered level by level, with slopes and without


def modules(d=3, cap=CAP, levels=LEVELS, feat=2, **kw):
    import permutohedral_encoding_amd as pe
    from permutohedral_encoding_amd import _native

    class Instrumented(_native.EncodingWrapper):
        pass

    torch.manual_seed(5)
    sig = np.geomspace(1.0, 1e-3, levels)
    native, python = (pe.PermutoEncoding(d, cap, levels, feat, sig, **kw) for _ in range(2))
    with torch.no_grad():
        native.lattice_values.uniform_(-1, 1)
    python.load_state_dict(native.state_dict())
    python.lattice.__class__ = Instrumented
    return native, python


def close(a, b):
    # sums of the same terms in another order, 2^-24 each
    assert torch.isfinite(a).all() and (a - b).norm() <= 1e-6 * b.norm()


def sdf_pass(m, pts, up, q, g, window=None, between=None):
    m.lattice_values.grad = None
    p, u = pts.clone().requires_grad_(True), up.clone(memory_format=torch.preserve_format).requires_grad_(True)
    out = m(p, window)
    if between is not None:
        with torch.no_grad():
            between(m, p)
    normal, = torch.autograd.grad(out, p, u, create_graph=True)
    torch.autograd.backward([out, normal], [g, q])
    table = m.table_grad.grad if m.sparse_table_grad else m.lattice_values.grad
    return [t.detach().clone() for t in (out, normal, p.grad, u.grad, table)]


@pytest.fixture(scope="module")
def inputs():
    torch.manual_seed(6)
    pts = torch.rand(N, 3, device="cuda")
    return pts, lambda m: (torch.randn(N, m.output_dims(), device="cuda"), torch.randn(N, 3, device="cuda"), torch.randn(N, m.output_dims(), device="cuda"))


def keeps_slopes(m, pts):
    """Whether a forward holds more memory than its result and what autograd keeps of the call (the points are given)."""
    with torch.no_grad():
        m(pts[:1])  # (makes the 16-bit copy of the table, if there is one)
    before = torch.cuda.memory_allocated()
    out = m(pts.clone().requires_grad_(True))
    slopes = 4 * m.nr_levels * m.nr_feat_per_level * pts.numel()
    return torch.cuda.memory_allocated() - before > out.numel() * 4 + pts.numel() * 4 + slopes // 2


@pytest.mark.parametrize("kw,rows", [({}, True), ({}, False), (dict(contiguous_output=True, concat_points=True), True), (dict(sparse_table_grad=True), True),
                                     (dict(lattice_half_precision=torch.bfloat16), False)])
def test_module_keeps_slopes_and_agrees_with_the_gathering_path(inputs, kw, rows):
    pts, draw = inputs
    native, python = modules(**kw)
    assert keeps_slopes(native, pts) and not keeps_slopes(python, pts)
    up, q, g = draw(native)
    up = up if rows else up.t().contiguous().t()
    window = torch.tensor([1, 0.5, 1, 0, 1, 1, 0.25, 1.0])
    a, b = (sdf_pass(m, pts, up, q, g, window) for m in (native, python))
    assert torch.equal(a[0], b[0])
    for x, y in zip(a[1:], b[1:]):
        close(x, y)


@pytest.mark.parametrize("what", ["table", "data", "other_memory", "positions", "shift", "window", "hooks", "cap"])
def test_slopes_of_changed_inputs_are_not_used(inputs, monkeypatch, what):
    """Where an input changes in place, or is given other memory, between the passes the gathering kernels run, as in the autograd
    functions: the same bits.  And nothing is kept beside what hooks on saved tensors see, nor over the cap on scratch memory."""
    from permutohedral_encoding_amd import _native
    pts, draw = inputs
    native, python = modules()
    up, q, g = draw(native)
    window = torch.ones(LEVELS, device="cuda")

    def between(m, p):
        if what == "table":
            m.lattice_values.mul_(0.5)
        elif what == "data":  # (the version counter does not see the write: the program says so)
            m.lattice_values.data.mul_(0.5)
            torch.autograd.graph.increment_version(m.lattice_values)
        elif what == "other_memory":
            m.lattice_values.data = 0.5 * m.lattice_values.data
        elif what == "positions":
            p.mul_(0.5)
        elif what == "shift":
            m.random_shift_per_level.add_(1.0)
        elif what == "window":
            window.copy_(torch.linspace(0.1, 1.0, LEVELS))
    if what == "cap":
        monkeypatch.setattr(_native, "MAX_WORKSPACE_BYTES", 1 << 20)
    results = []
    for m in (native, python):
        window.fill_(1.0)
        if what == "hooks":
            with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
                results.append(sdf_pass(m, pts, up, q, g, window))
        else:
            results.append(sdf_pass(m, pts, up, q, g, window, between))
    for x, y in zip(*[r[:4] for r in results]):
        assert torch.equal(x, y)


def test_slopes_are_freed_with_the_graph_and_travel_through_a_captured_graph(inputs):
    pts, draw = inputs
    native, _ = modules()
    up, q, g = draw(native)
    sdf_pass(native, pts, up, q, g)
    native.lattice_values.grad = None
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    out = native(pts.clone().requires_grad_(True))
    del out
    assert torch.cuda.memory_allocated() == before  # dropped without a backward
    static = pts.clone()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        sdf_pass(native, static, up, q, g)
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    native.lattice_values.grad = None
    with torch.cuda.graph(graph):
        captured = sdf_pass(native, static, up, q, g)
    for replay in range(3):
        static.copy_(torch.rand_like(pts))
        graph.replay()
        got = [t.clone() for t in captured]
        want = sdf_pass(native, static, up, q, g)
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(got[:4], want[:4])), replay
        assert torch.allclose(got[4], want[4], rtol=1e-4, atol=1e-6 * want[4].abs().max().item()), replay


@pytest.fixture
def little_memory():
    """-> f(left): lets this process take `left` more bytes from the device (what it has cached is released first)."""
    # (large blocks that earlier tests have left in the cache go too: what the test itself allocates would be cut from them, and what is left
    # of such a block serves requests that are meant to find no memory)
    gc.collect()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()

    def limit(left):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + left) / torch.cuda.get_device_properties(0).total_memory)
    yield limit
    torch.cuda.set_per_process_memory_fraction(1.0)


def test_slopes_are_given_back_where_memory_runs_short(inputs, little_memory):
    """A tensor that fits only in the place of the slopes (11.6 MB) is allocated, and the passes over the graph then gather: the bits of the
    autograd functions."""
    pts, draw = inputs
    native, python = modules()
    up, q, g = draw(native)

    def next_layer(m, p):
        little_memory(16 << 20)
        big = torch.empty(22 << 20, dtype=torch.uint8, device="cuda")  # noqa: F841
        torch.cuda.set_per_process_memory_fraction(1.0)
    a, b = sdf_pass(native, pts, up, q, g, between=next_layer), sdf_pass(python, pts, up, q, g)
    for x, y in zip(a[:4], b[:4]):
        assert torch.equal(x, y)
    assert keeps_slopes(native, pts)  # the next forward keeps them again


@pytest.mark.parametrize("rows", [False, True])
def test_a_forward_that_fits_without_slopes_does_not_fail_for_them(little_memory, rows):
    """64 MB of result, 193 MB of slopes, and room for one of them; in rows the forward writes through an array of the result's size."""
    n = 1 << 20
    native, _ = modules(contiguous_output=rows)
    pts = torch.rand(n, 3, device="cuda").requires_grad_(True)
    with torch.no_grad():
        want = native(pts)
    little_memory((200 << 20) + (rows << 26))
    out = native(pts)
    assert torch.equal(out, want)


def test_slopes_take_a_bounded_share_of_the_memory(inputs, little_memory):
    """A sixteenth of what the process may use: here room for the slopes of a few forwards and a half."""
    pts, _ = inputs
    native, _ = modules()
    torch.cuda.empty_cache()
    slopes, reserved = 4 * LEVELS * 2 * pts.numel(), torch.cuda.memory_reserved()
    few = 1 + reserved // (5 * slopes)  # (so many that there is no shortage: less than three quarters of the limit are taken)
    little_memory(16 * (2 * few + 1) * slopes // 2 - reserved)
    outs = []
    for _ in range(few):
        assert keeps_slopes(native, pts)
        outs.append(native(pts.clone().requires_grad_(True)))
    assert not keeps_slopes(native, pts)
    outs.pop()
    assert keeps_slopes(native, pts)


# just above the sizes that gather with two features: the product of points, levels and dimensions, and the gathers on a large table ... and
# where four and eight features keep slopes
GEOMETRIES = [(2, 2, 320001, 5, 1 << 12), (3, 2, 22060, 17, 1 << 19), (5, 2, 106667, 6, 1000), (8, 2, 100001, 4, 1 << 12), (2, 4, 70001, 8, 1 << 18),
              (7, 4, 50001, 4, 1 << 18), (4, 8, 80001, 4, 1 << 18)]


@pytest.mark.parametrize("d,feat,n,levels,cap", GEOMETRIES)
@pytest.mark.parametrize("layout", ["rows", "padded", "level_major", "broadcast", "every_other", "odd_stride"])
def test_module_with_slopes_in_other_geometries_and_layouts(d, feat, n, levels, cap, layout):
    """Values, position gradients, what comes back through them and both table gradients, of every layout an upstream gradient arrives in."""
    native, python = modules(d, cap, levels, feat)
    pts = torch.rand(n, d, device="cuda")
    assert keeps_slopes(native, pts) and (feat != 2 or not keeps_slopes(native, pts[:-2]))
    cols = native.output_dims()
    g = torch.randn(n, cols, device="cuda")
    up = {"rows": lambda: g, "padded": lambda: torch.nn.functional.pad(g, (0, 4))[:, :cols], "level_major": lambda: g.t().contiguous().t(),
          "broadcast": lambda: torch.randn(1, 1, device="cuda").expand(n, cols), "every_other": lambda: torch.randn(2 * n, cols, device="cuda")[::2],
          "odd_stride": lambda: torch.nn.functional.pad(g, (0, 1))[:, :cols]}[layout]()
    q = torch.randn(n, d, device="cuda")
    results = []
    for m in (native, python):
        p, u = pts.clone().requires_grad_(True), up.detach()
        if layout != "broadcast":
            u = u.requires_grad_(True)
        m.lattice_values.grad = u.grad = None
        out = m(p)
        normal, = torch.autograd.grad(out, p, u, create_graph=True)
        torch.autograd.backward([out, normal], [up.detach(), q])
        results.append([out, normal, p.grad, m.lattice_values.grad] + ([u.grad] if u.requires_grad else []))
    assert torch.equal(results[0][0], results[1][0])
    for x, y in zip(*[r[1:] for r in results]):
        close(x.detach(), y.detach())


def test_slopes_serve_every_pass_over_a_kept_graph(inputs):
    """retain_graph: the same bits again, after which the graph is freed; two sets of normals in one pass, each differentiated."""
    pts, draw = inputs
    native, python = modules()
    up, q, g = draw(native)
    p = pts.clone().requires_grad_(True)
    out = native(p)
    grads = [torch.autograd.grad(out, p, up, retain_graph=keep)[0] for keep in (True, True, False)]
    assert torch.equal(grads[0], grads[1]) and torch.equal(grads[0], grads[2])
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out, p, up)
    ups, qs = [up, torch.randn_like(up)], [q, torch.randn_like(q)]
    results = []
    for m in (native, python):
        m.lattice_values.grad = None
        p, us = pts.clone().requires_grad_(True), [u.clone().requires_grad_(True) for u in ups]
        out = m(p)
        normals = [torch.autograd.grad(out, p, u, create_graph=True)[0] for u in us]
        torch.autograd.backward([out] + normals, [g] + qs, retain_graph=True)
        first = [t.clone() for t in (p.grad, us[0].grad, us[1].grad, m.lattice_values.grad)]
        torch.autograd.backward([out] + normals, [g] + qs)
        results.append([n.detach() for n in normals] + first + [p.grad / 2, us[0].grad / 2, us[1].grad / 2, m.lattice_values.grad / 2])
    for x, y in zip(*results):
        close(x, y)


@pytest.mark.parametrize("where", ["forward", "backward", "thread"])
def test_slopes_across_streams_and_threads(inputs, where):
    """Forward on a side stream, backward called from one, backward from another thread."""
    import threading
    pts, draw = inputs
    native, python = modules()
    up, q, g = draw(native)
    want = sdf_pass(python, pts, up, q, g)
    p, u = pts.clone().requires_grad_(True), up.clone().requires_grad_(True)
    main, side = torch.cuda.current_stream(), torch.cuda.Stream()
    native.lattice_values.grad = None

    def forward():
        return native(p)

    def backward(out):
        normal, = torch.autograd.grad(out, p, u, create_graph=True)
        torch.autograd.backward([out, normal], [g, q])
        return normal
    side.wait_stream(main)
    if where == "forward":
        with torch.cuda.stream(side):
            out = forward()
        main.wait_stream(side)
        normal = backward(out)
    elif where == "backward":
        out = forward()
        side.wait_stream(main)
        with torch.cuda.stream(side):
            normal = backward(out)
    else:
        out, results = forward(), []
        worker = threading.Thread(target=lambda: results.append(backward(out)))
        worker.start()
        worker.join()
        normal, = results
    torch.cuda.synchronize()
    assert torch.equal(out, want[0])
    for x, y in zip((normal, p.grad, u.grad, native.lattice_values.grad), want[1:]):
        close(x.detach(), y)


def test_hooks_on_saved_tensors_are_looked_at_under_the_interpreters_lock():
    """Forwards of several threads under the same hooks leave their reference counts as they were."""
    import sys
    import threading
    native, _ = modules(levels=2, cap=1 << 18)
    pts = torch.rand(9000, 3, device="cuda").requires_grad_(True)

    def pack(t):
        return t

    def unpack(t):
        return t

    def forwards():
        with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
            for _ in range(300):
                native(pts)
    before = sys.getrefcount(pack), sys.getrefcount(unpack)
    workers = [threading.Thread(target=forwards) for _ in range(4)]
    for w in workers:
        w.start()
    for w in workers:
        w.join()
    torch.cuda.synchronize()
    del workers
    gc.collect()
    assert (sys.getrefcount(pack), sys.getrefcount(unpack)) == before
