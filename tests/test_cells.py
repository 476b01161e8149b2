"""Tables in cells (csrc/penc_cells.hpp): a gather from a permuted copy reads the values of the table it was made from."""
import numpy as np
import pytest
import torch

CELLS = 0x100
HALF = {1: torch.float16, 2: torch.bfloat16}


def make_cells(table, pos_dim, fmt, workspace_levels=None):
    from permutohedral_encoding_amd import _native
    lib, (levels, cap, feat) = _native.lib(), table.shape
    source = 0 if table.dtype == torch.float32 else fmt
    cells = torch.full((levels, cap, feat), float("nan"), dtype=HALF[fmt], device="cuda")
    nbytes = lib.penc_table_cells_workspace_bytes(feat, levels, cap, fmt)
    if workspace_levels is not None:
        nbytes = workspace_levels * cap * feat * cells.element_size() + 256
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    assert lib.penc_table_cells(pos_dim, feat, levels, cap, table.data_ptr(), source, fmt, cells.data_ptr(), ws.data_ptr(), nbytes,
                                torch.cuda.current_stream().cuda_stream) == 0
    return cells


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [1, 2])
@pytest.mark.parametrize("feat", [2, 4, 8])
@pytest.mark.parametrize("d", range(2, 9))
def test_every_gather_from_cells_equals_the_gather_from_the_table(d, feat, fmt):
    """One line, two, less than a workgroup's lines, as many, a few workgroups'; levels one and several at a time through the workspace, a masked
    one; results bit for bit, from workgroups of 64 points and all levels and from launches a level at a time."""
    from helpers import make_encoding, random_problem, to_gpu
    from permutohedral_encoding_amd import _native
    line = 128 // (feat * 2)
    lib, st = _native.lib(), torch.cuda.current_stream().cuda_stream
    for cap, levels, n in ((line, 3, 100), (2 * line, 3, 65), (64 * line, 5, 1003), (128 * line, 5, 1003), (1 << 14, 5, 2001), (1 << 18, 24 // feat * 2, 30001)):
        p = random_problem(d, n, levels, cap, seed=d, sigma_range=(1.0, 1e-3), nr_feat=feat)
        p["window"][levels // 2] = 0.0
        _, fp = make_encoding(d, p["sigmas"], p["shift"], nr_feat=feat)
        table, pos, win, dpos, grad = (to_gpu(p[k]) for k in ("table", "pos", "window", "dpos", "grad"))
        plain = table.to(HALF[fmt])
        cells = make_cells(table, d, fmt, workspace_levels=2 if cap == 1 << 14 else None)
        assert torch.equal(cells, make_cells(plain, d, fmt))  # from a table already rounded
        assert torch.equal(cells.reshape(levels, -1, feat).float().sort(1).values, plain.reshape(levels, -1, feat).float().sort(1).values)
        sf, shift = fp.m_scale_factor.data_ptr(), fp.m_random_shift_per_level.data_ptr()
        cols = feat * levels
        rows = grad.reshape(cols, n).t().contiguous()
        ws = torch.empty(lib.penc_positions_workspace_bytes(d, n, levels) + 4 * cols * n + 1024, dtype=torch.uint8, device="cuda")

        def results(values, table_format):
            common = (d, feat, n, levels, cap, pos.data_ptr(), values.data_ptr(), table_format, sf, shift, win.data_ptr())
            out, as_rows, positions_grad = torch.empty(cols, n, device="cuda"), torch.empty(n, cols, device="cuda"), torch.empty(n, d, device="cuda")
            slopes = torch.zeros(levels * -(-n // 64) * 64 * d * feat, device="cuda")
            assert lib.penc_forward_half(*common, out.data_ptr(), 0, 1.0, st) == 0
            got = [out.clone()]
            for to_rows in (None, as_rows.data_ptr()):
                assert lib.penc_forward_slopes(*common, out.data_ptr(), to_rows, cols, slopes.data_ptr(), 0, 1.0, st) == 0
                got += [slopes.clone(), out.clone() if to_rows is None else as_rows]
            level_major = torch.empty(cols, n, device="cuda")
            assert lib.penc_backward_positions_rowmajor(*common, rows.data_ptr(), cols, level_major.data_ptr(), positions_grad.data_ptr(),
                                                        ws.data_ptr(), ws.numel(), st) == 0
            got.append(positions_grad)
            grad_grad = torch.empty(n, cols, device="cuda")
            assert lib.penc_grad_grad_rowmajor(*common, dpos.data_ptr(), grad_grad.data_ptr(), cols, 0, ws.data_ptr(), ws.numel(), st) == 0
            got.append(grad_grad)
            positions_grad2, grad_grad2 = torch.empty(n, d, device="cuda"), torch.empty(cols, n, device="cuda")
            assert lib.penc_backward_half(*common, grad.data_ptr(), 0, None, positions_grad2.data_ptr(), ws.data_ptr(), ws.numel(), st) == 0
            assert lib.penc_double_backward_from_positions_half(*common, dpos.data_ptr(), grad.data_ptr(), 0, None, grad_grad2.data_ptr(), 0,
                                                                ws.data_ptr(), ws.numel(), st) == 0
            got += [positions_grad2, grad_grad2]
            return got

        for k, (want, got) in enumerate(zip(results(plain, fmt), results(cells, fmt | CELLS))):
            assert torch.equal(want, got), (cap, levels, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [1, 2])
def test_conversion_rounds_as_torch_does(fmt):
    """Ties, subnormals, overflow, infinities, NaN, signed zeros: a line of them each."""
    bits = torch.cat([torch.arange(0, 1 << 32, 65521, dtype=torch.int64), torch.tensor([0x7F800000, 0xFF800000, 0x7FC00000, 0x7F800001, 0x80000000, 0x33000000,
                      0x33000001, 0x387FE000, 0x477FF000, 0x477FEFFF, 0x3F808000, 0x3F818000, 0x7F7FFFFF])])
    bits = torch.cat([bits, bits[: (1 << 17) - len(bits) % (1 << 17)]])
    values = bits.to(torch.int32).view(torch.float32)[: 1 << 17].reshape(1, 1 << 16, 2).cuda()
    plain, cells = values.to(HALF[fmt]), make_cells(values, 3, fmt)
    as_bits = lambda t: torch.where(torch.isnan(t), torch.full_like(t, float("nan")), t).view(torch.int16).reshape(-1).sort().values
    assert torch.equal(as_bits(plain), as_bits(cells))


def test_cells_are_refused_where_they_are_not_possible():
    import ctypes
    from permutohedral_encoding_amd import _native
    lib, p = _native.lib(), ctypes.c_void_p(1 << 20)
    assert lib.penc_table_cells_workspace_bytes(2, 4, 32, 1) > 0 and lib.penc_table_cells_workspace_bytes(8, 4, 8, 2) > 0
    for feat, cap, fmt in ((2, 16, 1), (2, 64, 0), (2, 1000, 2), (8, 4, 1), (3, 64, 1), (2, 64, 3), (2, 64, 1 | CELLS)):
        assert lib.penc_table_cells_workspace_bytes(feat, 4, cap, fmt) == 0 and lib.penc_table_cells_points(feat, cap, fmt) == -1
        assert lib.penc_table_cells(3, feat, 4, cap, p, 0, fmt, p, p, 1 << 20, None) != 0
    for cap, fmt in ((16, 1), (1000, 2), (64, 0)):  # neither is a table said to be in cells
        assert lib.penc_forward_slopes(3, 2, 10, 4, cap, p, p, fmt | CELLS, p, p, p, p, None, 0, p, 0, 1.0, None) == 9
        assert lib.penc_forward_half(3, 2, 10, 4, cap, p, p, fmt | CELLS, p, p, p, p, 0, 1.0, None) == 9
    assert lib.penc_table_cells(3, 2, 4, 64, p, 1, 2, p, p, 1 << 20, None) == 9
    assert lib.penc_table_cells(3, 2, 4, 64, None, 0, 1, p, p, 1 << 20, None) == 1
    assert lib.penc_table_cells(3, 2, 4, 64, p, 0, 1, ctypes.c_void_p((1 << 20) + 8), p, 1 << 20, None) == 5
    assert lib.penc_table_cells(3, 2, 4, 64, p, 0, 1, p, p, 64, None) == 8
    for feat, cap, bad in ((8, 64, 9), (2, 8, 9), (2, 1000, 9)):
        assert lib.penc_forward_cells(3, feat, 10, 4, cap, p, p, p, p, p, p, None, 0, None, 0, 1.0, p, 1 << 20, None) == bad
    assert lib.penc_forward_cells(3, 2, 10, 4, 64, p, None, p, p, p, p, None, 0, None, 0, 1.0, p, 1 << 20, None) == 1
    assert lib.penc_forward_cells(3, 2, 10, 4, 64, p, p, p, p, p, p, None, 0, None, 0, 1.0, p, 64, None) == 8
    assert lib.penc_forward_cells(3, 2, 10, 4, 64, p, p, p, p, p, p, p, 7, None, 0, 1.0, p, 1 << 20, None) == 2  # rows of seven floats


def test_where_a_forward_goes_by_way_of_cells():
    from permutohedral_encoding_amd import _native
    serves = lambda *geometry: _native.lib().penc_forward_cells_workspace_bytes(*geometry) > 0
    assert serves(3, 2, 1 << 20, 24, 1 << 18, 0) and serves(3, 2, 1 << 20, 24, 1 << 18, 48) and not serves(3, 8, 1 << 20, 24, 1 << 14, 0)
    assert not serves(8, 2, 1 << 20, 24, 1 << 18, 0) and not serves(3, 2, 1 << 20, 24, 1 << 19, 0) and not serves(3, 2, 1 << 20, 24, 200000, 0)
    assert not serves(3, 2, 1 << 18, 24, 1 << 14, 0) and not serves(3, 2, 1 << 20, 24, 1 << 12, 0)
    assert serves(3, 2, 1 << 20, 24, 1 << 14, 0) and not serves(3, 2, 1 << 20, 24, 1 << 14, 48)  # rows without a transpose


def test_from_how_many_points_a_16_bit_table_is_laid_out_in_cells():
    """Where a first pass on a new table takes as long either way: a third of a slice in points, half a million from 1.5 MiB on, a 28th of a slice."""
    from permutohedral_encoding_amd import _native
    points = _native.lib().penc_table_cells_points
    assert points(2, 1 << 14, 2) == (1 << 16) // 3 and points(2, 1 << 13, 2) == -1 and points(2, 1 << 18, 1) == (1 << 20) // 3
    assert points(2, 1 << 19, 2) == points(2, 1 << 20, 2) == points(4, 1 << 20, 2) == 1 << 19
    assert points(2, 1 << 22, 2) == (1 << 24) // 28 > 500003 and points(8, 1 << 22, 1) == (1 << 26) // 28


def test_cells_cover_the_lattice_once():
    """The rule of penc_cells.hpp in Python's integers: offsets with all residues, whichever they are, give a permutation.  (Those the library has are
    looked at in test_cells_of_neighbouring_lattice_points.)"""
    mul = 2531011
    for d in (2, 3, 5, 8):
        step = [(sum(mul ** (d - i) for i in range(d)) - ((d + 1) * mul ** (d - c) if c < d else 0)) % (1 << 32) for c in range(d + 1)]
        for line in (4, 8, 16, 32):
            offset, frontier = {0: 0}, [0]
            while frontier:  # breadth first over the steps
                frontier = [h for f in frontier for s in step for h in ((f + s) % (1 << 32), (f - s) % (1 << 32))
                            if h % line not in offset and offset.setdefault(h % line, h) == h]
            assert len(offset) == line
            cap = 64 * line
            slots = {((h - offset[h % line]) | (h % line)) % cap for h in range(cap)}
            assert slots == set(range(cap))


def hash_steps(d):
    """From one vertex of a simplex to the next: the hashes of the lattice's D+1 steps (penc_lattice.hpp: hash_step)."""
    mul = 2531011
    return [(sum(mul ** (d - i) for i in range(d)) - ((d + 1) * mul ** (d - c) if c < d else 0)) % (1 << 32) for c in range(d + 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("feat", [2, 4, 8])
@pytest.mark.parametrize("d", range(2, 9))
def test_cells_of_neighbouring_lattice_points(d, feat):
    """The offsets the library ships, from a table whose slots hold their own number: they make a permutation, and bring the vertices of a simplex onto
    as few lines as penc_cells.hpp says."""
    line = 64 // feat
    cap = 4096 * line
    numbers = torch.zeros(1, cap, feat, dtype=torch.int16)
    numbers[0, :, 0], numbers[0, :, 1] = (torch.arange(cap) & 0xFFFF).to(torch.int16), (torch.arange(cap) >> 16).to(torch.int16)
    cells = make_cells(numbers.view(torch.float16).cuda(), d, 1).view(torch.int16).cpu().numpy()[0].astype(np.int64)
    slot = ((cells[:, 0] & 0xFFFF) | (cells[:, 1] << 16)).reshape(-1, line)  # of each place of a line
    assert np.array_equal(np.sort(slot.reshape(-1)), np.arange(cap))
    offsets = (slot - line * np.arange(cap // line)[:, None]) % cap
    assert (offsets == offsets[0]).all() and np.array_equal(offsets[0] % line, np.arange(line))  # one lattice vector for each residue
    rng, steps = np.random.default_rng(d), np.array(hash_steps(d))
    order = np.argsort(rng.random((20000, d + 1)), axis=1)[:, :d]
    vertices = np.concatenate([np.zeros((20000, 1), np.int64), np.cumsum(steps[order], axis=1)], axis=1)
    vertices = (vertices + rng.integers(0, cap, (20000, 1))) % cap
    lines = np.sort((vertices - offsets[0][vertices % line]) % cap // line, axis=1)
    mean = (1 + (lines[:, 1:] != lines[:, :-1]).sum(axis=1)).mean()
    want = {2: (1.36, 1.5, 1.75), 3: (2.03, 2.23, 2.57), 4: (2.83, 3.11, 3.6), 5: (3.86, 4.35, 4.56), 6: (4.85, 5.2, 5.9), 7: (5.74, 6.29, 6.8), 8: (6.98, 7.4, 7.77)}
    assert mean <= want[d][(2, 4, 8).index(feat)] + 0.05  # (the mean of 20000 is within 0.03 of that of all at four standard errors)


@pytest.mark.gpu
@pytest.mark.parametrize("d,feat,cap,dtype", [(3, 2, 1 << 16, torch.bfloat16), (2, 4, 1 << 14, torch.float16), (5, 8, 1 << 12, torch.bfloat16)])
def test_module_gathers_from_cells_once_enough_points_were_gathered(d, feat, cap, dtype):
    """Results are those of the table in its own order throughout: before, at and after the call that makes the copy, in both derivatives, after
    an in-place change, in a graph captured before the copy was made, and where its making is refused."""
    import permutohedral_encoding_amd as pe
    from permutohedral_encoding_amd import _native
    levels = 6
    line = _native.lib().penc_table_cells_points(feat, cap, _native.TABLE_FORMATS[dtype])
    assert line > 0
    m = pe.PermutoEncoding(d, cap, levels, feat, np.geomspace(1.0, 1e-3, levels), lattice_half_precision=dtype)
    plain = pe.PermutoEncoding(d, cap, levels, feat, np.geomspace(1.0, 1e-3, levels))  # of the rounded values, gathered in fp32
    plain.load_state_dict(m.state_dict())

    def follow():
        with torch.no_grad():
            plain.lattice_values.copy_(m.lattice_values.to(dtype).float())
    follow()
    few, many = torch.rand(line // 2, d, device="cuda"), torch.rand(line, d, device="cuda")
    with torch.no_grad():
        assert torch.equal(m(few), plain(few)) and m.lattice._cells is None
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            m(few[:100])
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            captured = m(many)  # enough by now, but not while a graph is captured
        assert m.lattice._cells is None
        assert torch.equal(m(few), plain(few)) and m.lattice._cells is not None
        assert torch.equal(m(many), plain(many)) and torch.equal(m(many[:1]), plain(many[:1]))
        for _ in range(2):
            captured.zero_()
            graph.replay()
            assert torch.equal(captured, plain(many))

        m.lattice_values.mul_(0.5)
        follow()
        assert torch.equal(m(many), plain(many)) and m.lattice._cells is not None and m.lattice._half_copy is None

    def derivatives(enc, pos):
        pos = pos.clone().requires_grad_(True)
        out = enc(pos)
        normal, = torch.autograd.grad(out, pos, torch.ones_like(out).requires_grad_(True), create_graph=True)
        enc.lattice_values.grad = None
        (normal * pos.detach()).sum().backward()
        return out.detach(), normal.detach(), enc.lattice_values.grad
    for pos in (few, many):
        for a, b in zip(derivatives(m, pos), derivatives(plain, pos)):
            assert (a - b).norm() <= 1e-6 * b.norm()

    # a table in training: four times the points before the next version is laid out
    with torch.no_grad():
        m.lattice_values.mul_(2.0)
    follow()
    assert torch.equal(m(many).detach(), plain(many).detach()) and m.lattice._cells is None
    for _ in range(3):
        m(many)
    assert m.lattice._cells is not None and torch.equal(m(many).detach(), plain(many).detach())

    # no memory for it: the copy in the table's own order serves
    m.invalidate_half_table()

    class Refusing:
        def __getattr__(self, name):
            return getattr(_native_bridge, name)

        def table_in_cells(self, *args):
            raise torch.cuda.OutOfMemoryError("refused")
    _native_bridge, _native._bridge = _native._bridge, Refusing()
    try:
        with torch.no_grad():
            assert torch.equal(m(many), plain(many)) and m.lattice._cells is None
    finally:
        _native._bridge = _native_bridge


@pytest.mark.gpu
@pytest.mark.parametrize("feat", [2, 4])
@pytest.mark.parametrize("d", range(2, 9))
def test_forward_by_way_of_cells_equals_the_forward(d, feat):
    """Levels that are chosen for the copy and levels that are not in one call, a masked one among them, fewer levels than dies and more, one line,
    part of a workgroup's and several workgroups' lines, a batch of one point and one that ends in the middle of a wave; level by level, in rows,
    with and without slopes."""
    from helpers import make_encoding, random_problem, to_gpu
    from permutohedral_encoding_amd import _native
    lib, st = _native.lib(), torch.cuda.current_stream().cuda_stream
    line, kinds = 128 // (4 * feat), set()
    for cap, levels, n, finest in ((line, 2, 1, 1e-3), (4 * line, 3, 65, 1e-3), (1 << 14, 6, 5003, 1e-4), (1 << 16, 19, 3001, 1e-4)):
        p = random_problem(d, n, levels, cap, seed=d, sigma_range=(1.0, finest), nr_feat=feat)
        p["window"][levels // 3] = 0.0
        _, fp = make_encoding(d, p["sigmas"], p["shift"], nr_feat=feat)
        table, pos, win = to_gpu(p["table"]), to_gpu(p["pos"]), to_gpu(p["window"])
        cols, slope_floats = feat * levels, levels * -(-n // 64) * 64 * d * feat
        nbytes = 512 + cap * feat * 4 * levels
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        common = (d, feat, n, levels, cap, pos.data_ptr(), table.data_ptr())
        geometry = (fp.m_scale_factor.data_ptr(), fp.m_random_shift_per_level.data_ptr(), win.data_ptr())
        want, kept = torch.empty(cols, n, device="cuda"), torch.zeros(slope_floats, device="cuda")
        assert lib.penc_forward_slopes(*common, 0, *geometry, want.data_ptr(), None, 0, kept.data_ptr(), 0, 1.0, st) == 0
        for as_rows in (False, True):
            for keep in (False, True):
                out, rows, slopes = torch.zeros(cols, n, device="cuda"), torch.zeros(n, cols, device="cuda"), torch.zeros(slope_floats, device="cuda")
                assert lib.penc_forward_cells(*common, *geometry, out.data_ptr(), rows.data_ptr() if as_rows else None, cols,
                                              slopes.data_ptr() if keep else None, 0, 1.0, ws.data_ptr(), nbytes, st) == 0
                assert torch.equal(rows.t() if as_rows else out, want)
                assert not keep or torch.equal(slopes, kept)
                first = (ws.data_ptr() + 255) // 256 * 256 - ws.data_ptr()
                chosen = ws[first:first + 4 * levels].view(torch.int32)
                assert chosen[levels // 3] == 0
                kinds.update(chosen.tolist())
    assert kinds == {0, 1}


@pytest.mark.gpu
def test_copy_made_on_one_stream_is_waited_for_on_another():
    """The copy is made in the middle of a program, behind what its stream has to do; a call on another stream that finds it made waits for it."""
    import permutohedral_encoding_amd as pe
    m = pe.PermutoEncoding(3, 1 << 20, 12, 2, np.geomspace(1.0, 1e-3, 12), lattice_half_precision=torch.bfloat16)
    line = pe._native.lib().penc_table_cells_points(2, 1 << 20, 2)
    few, many = torch.rand(1000, 3, device="cuda"), torch.rand(line, 3, device="cuda")
    work = torch.randn(4096, 4096, device="cuda")
    side = torch.cuda.Stream()
    with torch.no_grad():
        want = m(few)
        torch.cuda.synchronize()
        for _ in range(20):
            work = (work @ work).clamp(-1, 1)
        m(many)
        assert m.lattice._cells[4] == [None]  # (the default stream's: the event is recorded when one is needed, and kept)
        with torch.cuda.stream(side):
            got = m(few)
            event, = m.lattice._cells[4]
            again = m(few)
    torch.cuda.synchronize()
    assert event is not None and m.lattice._cells[4] == [event] and torch.equal(got, want) and torch.equal(again, want)


def busy(work, times=20):
    for _ in range(times):
        work = (work @ work).clamp(-1, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("captured", [False, True])
def test_cells_are_made_of_the_table_where_its_16_bit_copy_is_not_filled_yet(captured):
    """The 16-bit copy waits for what its stream has to do, or for the first replay of the graph that makes it, when a call on another stream gathers
    enough for cells: they hold the table's values all the same, then and later."""
    import permutohedral_encoding_amd as pe
    levels, cap = 12, 1 << 20
    m = pe.PermutoEncoding(3, cap, levels, 2, np.geomspace(1.0, 1e-3, levels), lattice_half_precision=torch.bfloat16)
    plain = pe.PermutoEncoding(3, cap, levels, 2, np.geomspace(1.0, 1e-3, levels))
    plain.load_state_dict(m.state_dict())
    few, many = torch.rand(1000, 3, device="cuda"), torch.rand(pe._native.lib().penc_table_cells_points(2, cap, 2), 3, device="cuda")
    work, side, graph = torch.randn(4096, 4096, device="cuda"), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.no_grad():
        plain.lattice_values.copy_(plain.lattice_values.bfloat16().float())
        want_few, want_many = plain(few), plain(many)
        plain(few[:10])
        torch.cuda.synchronize()
        if captured:
            with torch.cuda.graph(graph):
                first = m(few)
        else:
            with torch.cuda.stream(side):
                busy(work)
                first = m(few)
        got = m(many)
        assert m.lattice._cells is not None
        torch.cuda.synchronize()
        if captured:
            graph.replay()
        assert torch.equal(got, want_many) and torch.equal(first, want_few) and torch.equal(m(few), want_few)


@pytest.mark.gpu
def test_a_16_bit_copy_made_on_one_stream_is_waited_for_on_another():
    import permutohedral_encoding_amd as pe
    m = pe.PermutoEncoding(3, 1 << 20, 12, 2, np.geomspace(1.0, 1e-3, 12), lattice_half_precision=torch.float16)
    few = torch.rand(1000, 3, device="cuda")
    work, side = torch.randn(4096, 4096, device="cuda"), torch.cuda.Stream()
    with torch.no_grad():
        want = m(few)
        m.invalidate_half_table()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            busy(work)
            m(few)
        got = m(few)  # beside the other stream's work, but for the copy
        again = m(few)
    torch.cuda.synchronize()
    assert m.lattice._half_copy[3] == side.cuda_stream and torch.equal(got, want) and torch.equal(again, want)


@pytest.mark.gpu
@pytest.mark.parametrize("captured", ["not", "on its stream", "on another"])
def test_the_copy_in_the_tables_order_goes_once_there_are_cells(captured):
    """One 16-bit copy of a table in the end, as ever, unless a graph has been captured with the first one."""
    import permutohedral_encoding_amd as pe
    levels, cap = 6, 1 << 20
    m = pe.PermutoEncoding(3, cap, levels, 2, np.geomspace(1.0, 1e-3, levels), lattice_half_precision=torch.bfloat16)
    few, many = torch.rand(1000, 3, device="cuda"), torch.rand(pe._native.lib().penc_table_cells_points(2, cap, 2), 3, device="cuda")
    before, side, graph = torch.cuda.memory_allocated(), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.no_grad():
        with torch.cuda.stream(side if captured == "on its stream" else torch.cuda.current_stream()):
            want = m(few)
        torch.cuda.synchronize()
        if captured != "not":
            with torch.cuda.graph(graph, stream=side):
                got = m(few)
        m(many)
        assert m.lattice._cells is not None and (m.lattice._half_copy is None) == (captured == "not")
        if captured == "not":
            assert torch.cuda.memory_allocated() - before <= 2 * m.lattice_values.numel() + 4 * want.numel() + 4096
        else:
            torch.empty(m.lattice_values.numel(), dtype=torch.bfloat16, device="cuda").fill_(7.0)
            got.zero_()
            graph.replay()
            assert torch.equal(got, want)
        assert torch.equal(m(few), want)


@pytest.mark.gpu
def test_no_cells_are_made_for_a_call_that_would_not_gather_from_them():
    """A window that requires a gradient is for the autograd functions, which gather from the copy in the table's order."""
    import permutohedral_encoding_amd as pe
    levels, cap = 6, 1 << 16
    m = pe.PermutoEncoding(3, cap, levels, 2, np.geomspace(1.0, 1e-3, levels), lattice_half_precision=torch.bfloat16)
    m.lattice_values.requires_grad_(False)
    many = torch.rand(pe._native.lib().penc_table_cells_points(2, cap, 2), 3, device="cuda")
    window = torch.ones(levels, device="cuda", requires_grad=True)
    with torch.no_grad():
        want = m(many, window)
    m.invalidate_half_table()
    got = m(many, window)
    assert m.lattice._cells is None and m.lattice._half_copy is not None and torch.equal(got.detach(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("points", [1000, 1 << 19])
def test_a_wrapper_that_keeps_copies_can_be_copied(points):
    """As it could when the 16-bit copy was a tensor alone: (1000 points: in the table's order, else in cells)"""
    import copy
    import permutohedral_encoding_amd as pe
    m = pe.PermutoEncoding(3, 1 << 16, 12, 2, np.geomspace(1.0, 1e-3, 12), lattice_half_precision=torch.bfloat16)
    pos = torch.rand(points, 3, device="cuda")
    with torch.no_grad():
        want = m(pos)
        assert (m.lattice._cells is None) == (points == 1000)
        other = copy.deepcopy(m.lattice)
        assert other.half_table == torch.bfloat16 and other._half_copy is None and other._cells is None
        assert torch.equal(other.encode(m.lattice_values, pos, m.anneal_window), want)
        assert torch.equal(copy.deepcopy(m)(pos), want) and torch.equal(m(pos), want)


@pytest.mark.gpu
def test_positions_that_are_no_tensor_are_refused_as_ever():
    import permutohedral_encoding_amd as pe
    m = pe.PermutoEncoding(3, 1 << 16, 4, 2, np.geomspace(1.0, 1e-3, 4), lattice_half_precision=torch.bfloat16)
    for bad in ([[0.0, 0.0, 0.0]], np.zeros((4, 3), np.float32), 1.0):
        with pytest.raises(ValueError, match="must be a torch.Tensor"):
            m(bad)
    with pytest.raises(ValueError, match="should have 2 dimensions"):
        m(torch.rand(3, device="cuda"))


@pytest.mark.gpu
@pytest.mark.parametrize("cells", [False, True])
def test_a_capture_waits_for_a_copy_made_on_another_stream(cells):
    """A graph captured and replayed while the stream that makes the copy is busy with other things."""
    import permutohedral_encoding_amd as pe
    m = pe.PermutoEncoding(3, 1 << 20, 12, 2, np.geomspace(1.0, 1e-3, 12), lattice_half_precision=torch.bfloat16)
    few, many = torch.rand(1000, 3, device="cuda"), torch.rand(pe._native.lib().penc_table_cells_points(2, 1 << 20, 2), 3, device="cuda")
    work, side, graph = torch.randn(4096, 4096, device="cuda"), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.no_grad():
        want = m(few)
        m.invalidate_half_table()
        torch.cuda.synchronize()
        busy(work)
        m(many if cells else few)
        with torch.cuda.stream(side):
            graph.capture_begin()
            got = m(few)
            graph.capture_end()
            graph.replay()
        side.synchronize()
        assert (m.lattice._cells is not None) == cells and m.lattice._captured is None and torch.equal(got, want)
        for _ in range(2):
            got.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("cells", [False, True])
def test_a_capture_on_a_stream_the_default_stream_waits_for(cells):
    """No event can be recorded on the default stream, which made the copy, while such a stream is captured: the graph makes its own."""
    import ctypes
    import permutohedral_encoding_amd as pe
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipStreamCreate.argtypes = [ctypes.POINTER(ctypes.c_void_p)]
    hip.hipStreamDestroy.argtypes = [ctypes.c_void_p]
    m = pe.PermutoEncoding(3, 1 << 16, 6, 2, np.geomspace(1.0, 1e-3, 6), lattice_half_precision=torch.bfloat16)
    few, many = torch.rand(1000, 3, device="cuda"), torch.rand(pe._native.lib().penc_table_cells_points(2, 1 << 16, 2), 3, device="cuda")
    handle = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(handle)) == 0
    stream, graph = torch.cuda.ExternalStream(handle.value), torch.cuda.CUDAGraph()
    with torch.no_grad():
        want = m(many if cells else few)[:1000]
        points = many[:1000].contiguous() if cells else few
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            graph.capture_begin()
            got = m(points)
            graph.capture_end()
        assert (m.lattice._cells is not None) == cells and m.lattice._captured is not None
        for _ in range(3):
            got.zero_()
            torch.cuda.synchronize()
            with torch.cuda.stream(stream):
                graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, want) and torch.equal(m(points), want)
    del graph, got
    torch.cuda.synchronize()
    assert hip.hipStreamDestroy(handle) == 0


@pytest.mark.gpu
def test_a_16_bit_copy_that_a_capture_makes_is_that_captures_alone():
    """Neither a call outside, before the graph has run, nor another graph reads it; the calls of one capture share it."""
    import permutohedral_encoding_amd as pe
    m = pe.PermutoEncoding(3, 1 << 16, 6, 2, np.geomspace(1.0, 1e-3, 6), lattice_half_precision=torch.bfloat16)
    few, other = torch.rand(1000, 3, device="cuda"), torch.rand(1000, 3, device="cuda")
    with torch.no_grad():
        want, want_other = m(few), m(other)
        first, second = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
        m.invalidate_half_table()
        torch.cuda.synchronize()
        with torch.cuda.graph(first):
            a = m(few)
            made = m.lattice._captured[1]
            b = m(other)
            assert m.lattice._captured[1] is made
        assert m.lattice._half_copy is None
        with torch.cuda.graph(second):
            c = m(few)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.graph(torch.cuda.CUDAGraph()):  # (never run) a stream that takes part in a capture begun on another
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                m(few)
            torch.cuda.current_stream().wait_stream(side)
        third = torch.cuda.CUDAGraph()
        with torch.cuda.graph(third):
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                d = m(few)
            torch.cuda.current_stream().wait_stream(side)
        assert torch.equal(m(few), want)
        for graph, outs, wants in ((second, (c,), (want,)), (third, (d,), (want,)), (first, (a, b), (want, want_other))):
            for _ in range(3):
                for out in outs:
                    out.zero_()
                graph.replay()
                torch.cuda.synchronize()
                assert all(torch.equal(x, y) for x, y in zip(outs, wants))


@pytest.mark.gpu
@pytest.mark.parametrize("feat", [2, 4, 8])
def test_cells_of_a_table_that_does_not_begin_at_a_slot(feat):
    """A view into flattened parameters, one float into them: its 16-bit copy has always served, and so do the cells made of it."""
    import permutohedral_encoding_amd as pe
    levels, cap = 4, 1 << 14
    m = pe.PermutoEncoding(3, cap, levels, feat, np.geomspace(1.0, 1e-3, levels), lattice_half_precision=torch.bfloat16)
    flat = torch.randn(m.lattice_values.numel() + 1, device="cuda")
    m.lattice_values = torch.nn.Parameter(flat[1:].view(levels, cap, feat))
    many = torch.rand(pe._native.lib().penc_table_cells_points(feat, cap, 2), 3, device="cuda")
    with torch.no_grad():
        few = m(many[:100])
        assert m.lattice._cells is None
        m.invalidate_half_table()
        got = m(many)
    assert m.lattice._cells is not None and torch.equal(got[:100], few)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [False, True])
def test_forward_by_way_of_cells_keeps_to_the_workspace_cap(monkeypatch, rows):
    import permutohedral_encoding_amd as pe
    from permutohedral_encoding_amd import _native
    levels, cap, n = 16, 1 << 18, 1 << 20
    m = pe.PermutoEncoding(3, cap, levels, 2, np.geomspace(1.0, 1e-3, levels), contiguous_output=rows)
    assert _native.lib().penc_forward_cells_workspace_bytes(3, 2, n, levels, cap, 2 * levels if rows else 0) > m.lattice_values.numel() * 4
    pos = torch.rand(n, 3, device="cuda")

    def taken():
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        with torch.no_grad():
            out = m(pos)
        return out, torch.cuda.max_memory_allocated() - before

    want, free = taken()
    monkeypatch.setattr(_native, "MAX_WORKSPACE_BYTES", m.lattice_values.numel() * 4)
    got, capped = taken()
    assert torch.equal(got, want) and capped <= free - m.lattice_values.numel() * 4
