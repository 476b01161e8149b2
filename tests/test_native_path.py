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
