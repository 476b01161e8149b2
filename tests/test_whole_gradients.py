"""Table gradients that their reducers write whole: several pairs of features (masked levels too), records that segments have no room for, and points
without a place among ordinary ones."""
import numpy as np
import pytest
import torch

from permutohedral_encoding_amd import _native


@pytest.mark.gpu
@pytest.mark.parametrize("d,feat,levels,n,cap", [(3, 4, 16, 131075, 1 << 18), (5, 4, 12, 100003, 245759), (2, 4, 24, 1 << 18, (1 << 18) + 1), (4, 2, 24, 300007, 180225)])
def test_pairs_of_features_and_crowds(d, feat, levels, n, cap):
    import test_scatter_branches as branches
    assert _native.lib().penc_scatter_useful_bytes(d, feat, n, levels, cap) > levels * feat // 2 * n * (d + 1) * 12
    branches.test_scatter_with_more_workspace(d, feat, levels, n, cap)


@pytest.mark.gpu
@pytest.mark.parametrize("d,levels,n,cap", [(2, 24, 200003, 1 << 18), (3, 24, 131075, 1 << 18), (5, 20, 90001, 245759), (8, 16, 70001, 1 << 19), (3, 16, 200003, 1 << 14), (3, 16, 200003, 1 << 20)])
def test_points_without_a_place(d, levels, n, cap):
    """A coordinate that is not finite, or overflows, makes the gradient of the slots it is sent to NaN, at every live level, and of no other; with the bins of a
    whole gradient, narrow ones, and those of a large table."""
    from helpers import make_encoding
    rng = np.random.default_rng(d)
    lib, st = _native.lib(), torch.cuda.current_stream().cuda_stream
    enc, fp = make_encoding(d, np.geomspace(1.0, 1e-4, levels).astype(np.float32), (rng.standard_normal((levels, d)) * 10).astype(np.float32))
    torch.manual_seed(d)
    pos = torch.rand(n, d, device="cuda")
    bad = torch.arange(7, n, n // 5, device="cuda")
    payloads = torch.tensor([0x7FC00000, 0x7F800000, -8388608, 0x7F600000, 0x7FFFFFFF, -1], dtype=torch.int32, device="cuda").view(torch.float32)  # nan, inf, -inf, 3e38, nan of all bits, -nan
    without = pos.clone()
    pos[bad, torch.arange(len(bad), device="cuda") % d] = payloads[:len(bad)]
    window = torch.ones(levels, device="cuda")
    window[1] = 0.0
    up = torch.randn(n, 2 * levels, device="cuda")
    table = torch.zeros(levels, cap, 2, device="cuda")  # (not read by a table gradient)
    extra = lib.penc_scatter_useful_bytes(d, 2, n, levels, cap)
    assert extra > 0
    ws = torch.empty(lib.penc_scatter_workspace_bytes(d, n, levels, cap, levels) + extra, dtype=torch.uint8, device="cuda")

    def gradient(points, upstream):
        tg = torch.full((levels, cap, 2), 7.0, device="cuda")
        ws.fill_(0xAB)
        assert lib.penc_backward_rowmajor(d, 2, n, levels, cap, points.data_ptr(), table.data_ptr(), fp.m_scale_factor.data_ptr(), fp.m_random_shift_per_level.data_ptr(), window.data_ptr(),
                                          upstream.data_ptr(), 2 * levels, tg.data_ptr(), None, ws.data_ptr(), ws.numel(), st) == 0
        return tg

    ordinary = up.clone()
    ordinary[bad] = 0.0
    got, want, magnitude = gradient(pos, up), gradient(without, ordinary), gradient(without, ordinary.abs())
    slots = enc.simplex_debug(pos[bad].contiguous(), cap, gather_path=2)["slot"].long()
    # what is scaled there is not finite: 3e38 at the finer levels only (at the others such a point has slots of its own like any other)
    nowhere = ~torch.isfinite(pos[bad] * fp.m_scale_factor.view(levels, 1, d)).all(-1)
    mark = lambda which: torch.zeros(levels, cap, dtype=torch.int32, device="cuda").scatter_add_(
        1, slots.reshape(levels, -1), which[..., None].expand(-1, -1, d + 1).reshape(levels, -1).int()) > 0
    must, hit = mark(nowhere), mark(torch.ones_like(nowhere))
    assert torch.all(got[1] == 0.0)
    live = torch.arange(levels, device="cuda") != 1
    is_nan = torch.isnan(got[live])
    assert must[live].any(-1).all() and torch.all(is_nan.all(-1) | ~must[live]) and not torch.any(is_nan.any(-1) & ~hit[live])
    # A wave's sum over its lanes rounds up to 64 times, each of the groups its partial sum once, and the sum it is added to once, to 2^-24 of what they sum; the rest is
    # summed in fp64.  Both runs do, and a little is left for the order of what is not.
    groups = -(-n // 1024)
    off = (got - want).abs().masked_fill(hit[..., None], 0.0)
    assert torch.all(off[live] <= 4 * (groups + 64) * 2.0 ** -24 * magnitude[live].abs() + 1e-12)
