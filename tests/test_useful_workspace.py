"""What a table gradient asks for beside its workspace: lists of late adds only where they are used and pay, else the slack of narrower bins alone."""
import numpy as np
import pytest
import torch

from permutohedral_encoding_amd import _native


def lists(d, n, pair_levels):
    return 12 * (d + 1) * n * pair_levels


def useful(*geometry):
    return _native.lib().penc_scatter_useful_bytes(*geometry)


def test_lists_are_asked_for_where_they_are_used():
    assert useful(3, 2, 1 << 20, 24, 1 << 18) > lists(3, 1 << 20, 24)
    assert useful(3, 4, 1 << 18, 16, 1 << 18) > lists(3, 1 << 18, 32)
    assert useful(3, 8, 1 << 18, 16, 1 << 18) == 0                        # four pairs of features write every slot in parts
    assert useful(2, 2, 1 << 18, 24, 1 << 18) > lists(2, 1 << 18, 24) and useful(2, 2, (1 << 18) + 1, 24, 1 << 18) == 0
    assert useful(3, 2, 1 << 15, 24, 1 << 18) == 0                        # the sorted groups serve it
    assert useful(3, 8, 1 << 18, 16, 1 << 20) > lists(3, 1 << 18, 64)     # cleared in the scatter, whatever the number of features


@pytest.mark.parametrize("d,feat,n,levels,cap", [(2, 4, (1 << 18) + 3, 16, 1 << 16), (3, 2, 1 << 20, 24, 1 << 16), (8, 2, 1 << 18, 16, 1 << 16), (3, 2, 1 << 19, 24, 4097)])
def test_narrow_bins_are_not_lost_with_the_lists(d, feat, n, levels, cap):
    """A few percent on top of the workspace, whether or not a few hundred MB could be had."""
    pairs = levels * feat // 2
    plain = _native.lib().penc_scatter_workspace_bytes(d, n, pairs, cap, pairs)
    assert 0 < useful(d, feat, n, levels, cap) < 0.15 * plain < 0.15 * 1.6 * lists(d, n, pairs)


def test_never_more_than_the_most_and_nothing_for_what_is_refused():
    lib = _native.lib()
    for d in range(2, 9):
        for feat in (2, 4, 8):
            for n in (1000, 30011, 1 << 18, 1 << 20):
                for levels, cap in ((1, 700), (16, 1 << 14), (24, 100003), (16, 1 << 18), (24, (1 << 19) - 1), (20, 1 << 21), (4, 1 << 24), (2, 1 << 26)):
                    assert useful(d, feat, n, levels, cap) <= lib.penc_scatter_extra_bytes(d, n, levels * feat // 2, cap)
    assert useful(1, 2, 1000, 4, 16) == useful(3, 3, 1 << 20, 24, 1 << 18) == useful(3, 2, 0, 4, 16) == useful(3, 2, 10, 0, 16) == useful(3, 2, 10, 4, 0) == 0


@pytest.mark.gpu
def test_a_cap_between_the_two_keeps_the_narrow_bins():
    import permutohedral_encoding_amd as pe
    d, n, levels, cap = 3, 1 << 19, 24, 1 << 16
    plain, slack = _native.lib().penc_scatter_workspace_bytes(d, n, levels, cap, levels), useful(d, 2, n, levels, cap)
    m = pe.PermutoEncoding(d, cap, levels, 2, np.geomspace(1.0, 1e-3, levels))
    pos, g = torch.rand(n, d, device="cuda"), torch.randn(n, 2 * levels, device="cuda")

    def peak(limit):
        before, _native.MAX_WORKSPACE_BYTES = _native.MAX_WORKSPACE_BYTES, limit
        try:
            m.lattice_values.grad = None
            out = m(pos)
            torch.cuda.synchronize()
            torch.cuda.reset_peak_memory_stats()
            held = torch.cuda.memory_allocated()
            out.backward(g)
            torch.cuda.synchronize()
            return torch.cuda.max_memory_allocated() - held, m.lattice_values.grad.clone()
        finally:
            _native.MAX_WORKSPACE_BYTES = before

    grad_bytes = m.lattice_values.numel() * 4
    most, want = peak(None)
    at_the_cap, got = peak(plain + slack)
    below, without = peak(plain + slack - 1)
    assert most == at_the_cap >= plain + slack > below >= plain and most <= plain + slack + grad_bytes + (4 << 20)
    for other in (got, without):
        assert (other - want).norm() <= 1e-6 * want.norm()
