"""Branches of the table gradient that depend on the size of the table or on the layout of the upstream gradient, at the sizes where they
can go wrong."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("d,n,cap", [(3, 17 * 8192 + 777, 1 << 22), (3, 17 * 8192 + 777, 1 << 21), (2, 140001, (1 << 22) - 5), (5, 133001, 1 << 22),
                                     (8, 131201, 1 << 22), (4, 130001, (1 << 22) + 1), (4, 16 * 8192 + 1025, 1 << 22)])
def test_hundreds_of_bins(d, n, cap):
    """More than 256 bins (workgroups of 1024 threads; at 2^21 slots, 256 bins, of 512), a remainder in the last tile, bins of 2^14 slots.
    A third of a group's points, behind the tile by which the workgroup decides to stream, sit in one simplex: their records crowd a few
    segments up to the last place, so that four segments together hold more records than a reducer's registers take at a time, and the rest
    goes straight into the gradient.  First and second order against the oracle, at the first, a middle and the last level."""
    from helpers import assert_sum_close, gpu_input, make_encoding, random_problem, scatter_plan, to_gpu
    from oracle import api as orc
    rng = np.random.default_rng(d)
    levels = 24
    group, n_groups, bins, places = scatter_plan(d, n, levels, cap)
    threads = 1024 if bins > 256 else 512
    at = np.arange(n) % group
    crowd = (at >= group // 2) & (at < group // 2 + 1024)
    # several tiles, the crowded ones not the first; their records do not fit the segments; those of a wave's four are more than six
    # (up to 64 places: three) to a lane
    assert group == 4096 and group >= 4 * threads and 1024 > places and places <= 128 and n_groups >= 32
    assert 4 * places > 64 * (3 if places <= 64 else 6) or (d, cap) in [(5, 1 << 22), (4, 1 << 22)]
    p = random_problem(d, n, levels, 1, seed=60 + d, sigma_range=(2e-3, 1e-3))
    p["pos"] = np.where(crowd[:, None], (0.61 + 1e-7 * rng.standard_normal((n, d))).astype(np.float32), p["pos"])
    sf = orc.scale_factors(d, p["sigmas"])
    enc, _ = make_encoding(d, p["sigmas"], p["shift"])
    inp = gpu_input(p, need_pos_grad=False)
    inp.m_lattice_values = torch.zeros(levels, cap, 2, device="cuda")  # the table gradient does not read the table
    tg, _ = enc.backward(inp, to_gpu(p["grad"]))
    tg2, _ = enc.double_backward_from_positions(inp, to_gpu(p["dpos"]), to_gpu(p["grad"]))
    for level in (0, 11, levels - 1):
        one = slice(level, level + 1)
        args = (p["pos"], sf[one], p["shift"][one], p["window"][one])
        want = orc.backward_table(*args, p["grad"][one], cap, want_abs=True)
        assert_sum_close(tg[level].cpu().numpy()[None], want["grad64"], want["abs64"], 1e-4, f"first order, level {level}")
        want = orc.double_backward(p["pos"], np.zeros((1, cap, 2), np.float32), sf[one], p["shift"][one], p["window"][one], p["dpos"], p["grad"][one], want_abs=True)
        assert_sum_close(tg2[level].cpu().numpy()[None], want["grad64"], want["abs64"], 1e-4, f"second order, level {level}")


@pytest.mark.parametrize("d,n,cap", [(2, 17 * 8192 + 777, 1 << 19), (3, 17 * 8192 + 777, 1 << 18), (4, 130001, 200001), (5, 133001, 1 << 18), (8, 131201, 1 << 18)])
def test_segments_of_few_bins_run_over(d, n, cap):
    """At most 64 bins: tiles whose records all fit their segments take turns with tiles whose do not.  Of every group, 1024 points behind the tile
    by which it decides to stream sit in one simplex, and the rest of the group fills what their segments have left; the last tile ends early, and from
    non-powers of two slots are remainders.  First and second order against the oracle."""
    from helpers import assert_sum_close, gpu_input, make_encoding, random_problem, scatter_plan, to_gpu
    from oracle import api as orc
    rng = np.random.default_rng(d)
    levels = 24
    group, _, bins, places = scatter_plan(d, n, levels, cap)
    at = np.arange(n) % group
    crowd = (at >= group // 2) & (at < group // 2 + 1024)
    assert group == 4096 and bins <= 64 and n % 512 != 0
    assert 1024 + (group - 1024) * (d + 1) // bins > places
    p = random_problem(d, n, levels, 1, seed=80 + d, sigma_range=(2e-3, 1e-3))
    p["pos"] = np.where(crowd[:, None], (0.61 + 1e-7 * rng.standard_normal((n, d))).astype(np.float32), p["pos"])
    sf = orc.scale_factors(d, p["sigmas"])
    enc, _ = make_encoding(d, p["sigmas"], p["shift"])
    inp = gpu_input(p, need_pos_grad=False)
    inp.m_lattice_values = torch.zeros(levels, cap, 2, device="cuda")  # the table gradient does not read the table
    tg, _ = enc.backward(inp, to_gpu(p["grad"]))
    tg2, _ = enc.double_backward_from_positions(inp, to_gpu(p["dpos"]), to_gpu(p["grad"]))
    for level in (0, levels - 1):
        one = slice(level, level + 1)
        args = (p["pos"], sf[one], p["shift"][one], p["window"][one])
        want = orc.backward_table(*args, p["grad"][one], cap, want_abs=True)
        assert_sum_close(tg[level].cpu().numpy()[None], want["grad64"], want["abs64"], 1e-4, f"first order, level {level}")
        want = orc.double_backward(p["pos"], np.zeros((1, cap, 2), np.float32), sf[one], p["shift"][one], p["window"][one], p["dpos"], p["grad"][one], want_abs=True)
        assert_sum_close(tg2[level].cpu().numpy()[None], want["grad64"], want["abs64"], 1e-4, f"second order, level {level}")


@pytest.mark.parametrize("d,levels,n,cap", [(3, 24, (1 << 20) + 5, 1 << 17), (4, 24, (1 << 20) + 5, 1 << 18), (5, 24, (1 << 20) + 12345, 1 << 12)])
def test_rows_take_other_groups_of_points_than_level_major_gradients(d, levels, n, cap):
    """Groups of eight tiles from rows (of sixteen from five dimensions on), of sixteen from [L][F][N], at a size that has both, give the
    same sums."""
    from helpers import make_encoding, scatter_plan
    from permutohedral_encoding_amd import _native
    assert scatter_plan(d, n, levels, cap)[0] == 16 * 512  # (level-major)
    rng = np.random.default_rng(d)
    _, fp = make_encoding(d, np.geomspace(1.0, 1e-4, levels).astype(np.float32), (rng.standard_normal((levels, d)) * 10).astype(np.float32))
    pos, window = torch.rand(n, d, device="cuda"), torch.ones(levels, device="cuda")
    rows = torch.randn(n, 2 * levels, device="cuda")
    lib, st = _native.lib(), torch.cuda.current_stream().cuda_stream
    ws = torch.empty(lib.penc_scatter_workspace_bytes(d, n, levels, cap, 0), dtype=torch.uint8, device="cuda")
    out = []
    for given, stride in ((rows, 2 * levels), (rows.t().contiguous(), 0), (rows.abs().t().contiguous(), 0)):
        tg = torch.empty(levels, cap, 2, device="cuda")
        params = (pos.data_ptr(), None, fp.m_scale_factor.data_ptr(), fp.m_random_shift_per_level.data_ptr(), window.data_ptr(), given.data_ptr())
        if stride:
            rc = lib.penc_backward_rowmajor(d, 2, n, levels, cap, *params, stride, tg.data_ptr(), None, ws.data_ptr(), ws.numel(), st)
        else:
            rc = lib.penc_backward(d, 2, n, levels, cap, *params, tg.data_ptr(), None, ws.data_ptr(), ws.numel(), st)
        assert rc == 0
        out.append(tg)
    # the weights are not negative: the third is the sum of magnitudes.  Each of up to 257 groups rounds its partial sum, and the sum it is
    # added to, to 2^-24 of that
    assert torch.all((out[0] - out[1]).abs() <= 2 * 2 * 257 * 2.0 ** -24 * out[2] + 1e-30)


@pytest.mark.parametrize("d,feat,levels,n,cap", [(3, 2, 24, 17 * 8192 + 777, 1 << 22), (2, 4, 12, 200003, (1 << 22) - 6), (4, 2, 24, 130001, (1 << 22) + 2),
                                                 (3, 2, 6, 300001, 1 << 12), (2, 4, 16, (1 << 18) + 3, 1 << 16), (5, 2, 16, 100003, 50001),
                                                 (8, 2, 8, 65537, 1 << 18), (4, 2, 5, 120001, 1 << 14), (3, 2, 3, 60001, 700),
                                                 (8, 2, 8, 131201, 1 << 22), (3, 2, 24, 17 * 8192 + 777, 1 << 20), (3, 2, 5, (1 << 19) + 3, (1 << 21) + 8192),
                                                 (3, 2, 19, 95077, 1 << 21), (6, 2, 17, 60013, 600002), (8, 2, 24, 25003, 1 << 20),
                                                 (2, 2, 24, 700001, 1 << 20), (3, 2, 24, 700001, (1 << 21) + 8192),
                                                 (3, 2, 8, 200003, 1 << 14), (2, 2, 12, 300007, 30001), (2, 2, 21, 100003, 1342081), (2, 2, 21, 800003, 1342081)])
def test_scatter_with_more_workspace(d, feat, levels, n, cap):
    """Large tables: with lists of deferred adds in the workspace the scatter clears the gradient (in rows of workgroups that do nothing else, for
    16 M points times levels in shares of all), whatever it held, masked levels too, and what would go straight into it follows later: column sums of the
    coarse levels, and what segments have no room for (a third of the points sit in one simplex).  Small tables: bins of 2^10 to 2^12 slots, the
    last one not full, tables of less than one bin, summed by one workgroup or by several.  Both orders, rows and level-major, against the call without the extra bytes."""
    from helpers import make_encoding
    from permutohedral_encoding_amd import _native
    rng = np.random.default_rng(d)
    lib, st = _native.lib(), torch.cuda.current_stream().cuda_stream
    _, fp = make_encoding(d, np.geomspace(1.0, 1e-3, levels).astype(np.float32), (rng.standard_normal((levels, d)) * 10).astype(np.float32), nr_feat=feat)
    torch.manual_seed(d)
    pos = torch.rand(n, d, device="cuda")
    crowd = (torch.arange(n, device="cuda") % 4096 >= 2048) & (torch.arange(n, device="cuda") % 4096 < 3400)
    pos[crowd] = 0.61 + 1e-7 * torch.randn(int(crowd.sum()), d, device="cuda")
    window = torch.ones(levels, device="cuda")
    window[1] = 0.0
    rows, q = torch.randn(n, feat * levels, device="cuda"), torch.randn(n, d, device="cuda")
    pairs = levels * feat // 2
    table = torch.zeros(levels, cap, feat, device="cuda")  # (not read by a table gradient)
    plain, lists = lib.penc_scatter_workspace_bytes(d, n, pairs, cap, pairs), lib.penc_scatter_extra_bytes(d, n, pairs, cap)
    assert lists > (pairs * n * (d + 1) * 12 if cap * pairs >= 1 << 23 and cap > 1 << 19 else 0)
    ws = torch.empty(plain + lists, dtype=torch.uint8, device="cuda")

    def gradient(size, order, as_rows, up):
        up = up.contiguous() if as_rows else up.t().contiguous()
        tg = torch.full((levels, cap, feat), float("nan"), device="cuda")
        ws.fill_(0xAB)
        common = (pos.data_ptr(), table.data_ptr(), fp.m_scale_factor.data_ptr(), fp.m_random_shift_per_level.data_ptr(), window.data_ptr())
        end = (tg.data_ptr(), None)
        if order == 1:
            rc = (lib.penc_backward_rowmajor(d, feat, n, levels, cap, *common, up.data_ptr(), feat * levels, *end, ws.data_ptr(), size, st) if as_rows else
                  lib.penc_backward(d, feat, n, levels, cap, *common, up.data_ptr(), *end, ws.data_ptr(), size, st))
        elif as_rows:
            rc = lib.penc_double_backward_from_positions_rowmajor(d, feat, n, levels, cap, *common, q.data_ptr(), up.data_ptr(), feat * levels, *end, 0,
                                                                  ws.data_ptr(), size, st)
        else:
            rc = lib.penc_double_backward_from_positions(d, feat, n, levels, cap, *common, q.data_ptr(), up.data_ptr(), *end, 0, ws.data_ptr(), size, st)
        assert rc == 0
        return tg

    # Weights of the first order are not negative but for 2^-24 of rounding, so their sum with |gradient| is that of magnitudes.  A slot's groups round their partial sums, and what
    # these are added to, to 2^-24 of that: all but the slots of the crowd's simplex (a few more where its 1e-7 reach over a face), whose
    # contributions are added one by one.
    magnitude = gradient(plain, 1, False, rows.abs()).abs()
    each, one_by_one = -(-n // 4096), int(crowd.sum())
    want = gradient(plain, 1, False, rows)
    for as_rows in (False, True):
        got = gradient(plain + lists, 1, as_rows, rows)
        assert torch.all(got[1] == 0.0) and not torch.any(torch.isnan(got))
        off = (got - want).abs()
        assert torch.all(off <= 4 * (each + one_by_one) * 2.0 ** -24 * magnitude + 1e-12)
        assert int((off > 4 * each * 2.0 ** -24 * magnitude + 1e-12).sum()) <= levels * feat * 4 * (d + 1)
    for as_rows in (False, True):
        got, want = gradient(plain + lists, 2, as_rows, rows).double(), gradient(plain, 2, as_rows, rows).double()
        assert torch.all(got[1] == 0.0)
        # 2-norm, level by level: the two round the same sums in another order, those of the crowd's slots at random and `one_by_one` times
        for level in range(levels):
            assert (got[level] - want[level]).norm() <= 4 * one_by_one ** 0.5 * 2.0 ** -24 * (want[level].norm() + want[level].abs().max() * (d + 1) ** 0.5)
