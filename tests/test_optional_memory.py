"""Memory that a call does better with and can do without: a call that is refused it gives the same results, and a card on which it was refused
is not asked for it, its cache released each time, by every call."""
import gc

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def room_for():
    """-> f(bytes): lets this process take that much more from the device (what it has cached is released first)."""
    # (what a test allocates before it sets the limit would be cut from large blocks that earlier tests have left in the cache, and what is left of
    # those would serve requests that are meant to find no memory)
    gc.collect()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()

    def limit(left):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + left) / torch.cuda.get_device_properties(0).total_memory)
    yield limit
    torch.cuda.set_per_process_memory_fraction(1.0)


def peak_of(call):
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = call()
    torch.cuda.synchronize()
    return out, torch.cuda.max_memory_allocated() - before


def refused_once(call, check, extra, room_for):
    """`call` with memory for everything, without `extra` bytes of it, and with it again."""
    want, peak = peak_of(call)
    retries = lambda: torch.cuda.memory_stats()["num_alloc_retries"]
    room_for(peak - extra // 2)
    before = retries()
    check(call(), want)
    assert retries() > before, "the sizes leave room for what is to be refused"
    after_one = retries()
    for _ in range(4):
        got = None
        got, taken = peak_of(call)
        check(got, want)
        assert taken <= peak - extra // 2
    assert retries() == after_one
    torch.cuda.set_per_process_memory_fraction(1.0)
    got = None
    got, taken = peak_of(call)
    check(got, want)
    assert taken == peak


def test_a_gradient_that_is_refused_its_lists(room_for):
    import permutohedral_encoding_amd as pe
    levels, cap, n = 16, 1 << 20, 100003
    m = pe.PermutoEncoding(3, cap, levels, 2, np.geomspace(1.0, 1e-3, levels))
    pos, g = torch.rand(n, 3, device="cuda"), torch.randn(n, 2 * levels, device="cuda")

    def call():
        m(pos).backward(g)
        grad, m.lattice_values.grad = m.lattice_values.grad, None
        return grad

    def check(got, want):
        assert (got - want).norm() <= 1e-6 * want.norm()
    refused_once(call, check, pe._native.lib().penc_scatter_extra_bytes(3, n, levels, cap), room_for)


@pytest.mark.parametrize("rows", [False, True])
def test_a_forward_that_is_refused_its_copy_in_cells(room_for, rows):
    import permutohedral_encoding_amd as pe
    levels, cap, n = 16, 1 << 18, 1 << 20
    m = pe.PermutoEncoding(3, cap, levels, 2, np.geomspace(1.0, 1e-3, levels), contiguous_output=rows)
    pos = torch.rand(n, 3, device="cuda")

    def call():
        with torch.no_grad():
            return m(pos)

    def check(got, want):  # (a column at a time: there is little memory)
        assert all(torch.equal(got[:, c], want[:, c]) for c in range(2 * levels))
    refused_once(call, check, pe._native.lib().penc_forward_cells_workspace_bytes(3, 2, n, levels, cap, 2 * levels if rows else 0), room_for)


def half_table(levels, cap):
    """-> (an encoding with a 16-bit table, its call on points enough for a copy in cells over a number of calls)"""
    import permutohedral_encoding_amd as pe
    m = pe.PermutoEncoding(3, cap, levels, 2, np.geomspace(1.0, 1e-3, levels), lattice_half_precision=torch.bfloat16)
    pos = torch.rand(pe._native.lib().penc_table_cells_points(2, cap, 2), 3, device="cuda")

    def call(of=1):
        with torch.no_grad():
            return m(pos[:len(pos) // of])
    return m, call


def test_a_table_that_is_refused_its_copy_in_cells(room_for):
    m, call = half_table(16, 1 << 20)
    want = call(8)
    room_for(60 << 20)  # a result of 8 MB, not a copy of 64 MB
    before = torch.cuda.memory_stats()["num_alloc_retries"]
    for _ in range(12):
        got = call(8)
        assert torch.equal(got, want) and m.lattice._cells is None
    assert torch.cuda.memory_stats()["num_alloc_retries"] == before + 1
    torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(call(8), want) and m.lattice._cells is not None


def test_a_copy_in_cells_keeps_to_the_workspace_cap(monkeypatch):
    """Some levels at a time through a smaller workspace, or, with no room for one, the copy in the table's order."""
    from permutohedral_encoding_amd import _native
    levels, cap = 16, 1 << 20
    m, call = half_table(levels, cap)
    slice_bytes = 4 * cap
    want = call()
    assert m.lattice._cells is not None
    for most, made in ((3 * slice_bytes + 300, True), (slice_bytes + 256, True), (slice_bytes + 255, False), (0, False)):
        m.invalidate_half_table()
        monkeypatch.setattr(_native, "MAX_WORKSPACE_BYTES", most)
        got, taken = peak_of(call)
        assert torch.equal(got, want) and (m.lattice._cells is not None) == made
        assert taken <= got.numel() * 4 + levels * slice_bytes + most


def test_slopes_are_not_given_back_for_memory_that_a_call_can_do_without(room_for):
    """A forward finds room for its result, but for its copy in cells only in the place of another graph's slopes."""
    import permutohedral_encoding_amd as pe
    levels, cap, n = 16, 1 << 18, 1 << 20
    m = pe.PermutoEncoding(3, cap, levels, 2, np.geomspace(1.0, 1e-3, levels))
    ballast = torch.empty(1 << 30, dtype=torch.uint8, device="cuda")  # noqa: F841  (slopes take a sixteenth of what the process may use)
    few, many = torch.rand(100003, 3, device="cuda").requires_grad_(True), torch.rand(n, 3, device="cuda")
    before = torch.cuda.memory_allocated()
    out = m(few)
    with_slopes = torch.cuda.memory_allocated()
    assert with_slopes - before - 4 * out.numel() > pe._native.lib().penc_forward_cells_workspace_bytes(3, 2, n, levels, cap, 0) > 0
    room_for(1 << 30)
    torch.empty(2 * levels, n, device="cuda")  # freed at once: the allocator has a place for the result
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (8 << 20)) / torch.cuda.get_device_properties(0).total_memory)
    with torch.no_grad():
        m(many)
    assert torch.cuda.memory_allocated() == with_slopes
