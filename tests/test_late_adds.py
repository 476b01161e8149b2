"""Table gradients of few bins that their reducers write whole, from a workspace with lists of late adds: whatever the gradient held, masked levels, what
segments have no room for, last bins and tables that are not full, bins of 2^10 to 2^13 slots, several pairs of features."""
import pytest

from permutohedral_encoding_amd import _native


@pytest.mark.gpu
@pytest.mark.parametrize("d,feat,levels,n,cap", [(3, 2, 24, 131075, 1 << 18), (2, 2, 17, 300007, (1 << 19) - 1), (4, 2, 24, 100003, 200001), (5, 2, 20, 90001, 245759),
                                                 (8, 2, 16, 70001, 1 << 19), (6, 2, 17, 60013, 1 << 18), (2, 4, 16, (1 << 18) + 3, 1 << 16), (3, 8, 8, 100003, 100001),
                                                 (3, 2, 24, (1 << 20) + 513, 1 << 15)])
def test_reducers_write_the_gradient(d, feat, levels, n, cap):
    import test_scatter_branches as branches
    pairs = levels * feat // 2
    assert _native.lib().penc_scatter_extra_bytes(d, n, pairs, cap) > pairs * n * (d + 1) * 12
    branches.test_scatter_with_more_workspace(d, feat, levels, n, cap)


def test_lists_are_offered_where_a_reducer_has_its_bin_to_itself():
    extra = _native.lib().penc_scatter_extra_bytes
    assert extra(3, 1 << 20, 24, 1 << 18) > 24 * 4 * (1 << 20) * 12
    assert extra(3, 1 << 20, 16, 1 << 18) > 16 * 4 * (1 << 20) * 12  # 512 wide bins of 8192 slots
    assert extra(4, 1 << 20, 8, 1 << 18) == 0                         # 256 of them, shared by reducers
    assert 0 < extra(3, 1 << 19, 16, 1 << 13) < 16 * 4 * (1 << 19) * 12  # narrow ones that are shared
