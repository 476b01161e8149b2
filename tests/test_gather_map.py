"""The gathering kernels under every map of workgroups to (tile, row of levels): segments per die or not, rows of one or
two levels, remainders of tiles, rows and segments; forward and grad-grad bit for bit, position gradient within its bound (of
all levels of a block of points on the small tables of the first test, by groups of levels in the second)."""
import numpy as np
import pytest

from helpers import gpu_input, make_encoding, random_problem, to_gpu

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
orc = pytest.importorskip("oracle.api")


# d, n, levels, capacity, features, concat: one tile; fewer levels than dies; levels that do not divide the segments; single levels with
# three and with eight rounds; pairs with more and with fewer rows than dies; a slice too large for segments
@pytest.mark.parametrize("d,n,levels,cap,feat,concat", [(3, 1, 24, 1 << 10, 2, True), (3, 255, 7, 1 << 10, 2, False), (2, 513, 9, 1000, 4, True),
                                                        (6, 12001, 13, 1 << 11, 2, False), (5, 150001, 15, 1 << 11, 2, False),
                                                        (3, 131075, 19, 1 << 12, 2, True), (4, 300001, 8, 1 << 10, 2, False),
                                                        (3, 3000, 8, (1 << 20) + 1, 4, False)])
def test_every_level_and_point_is_reached_once(d, n, levels, cap, feat, concat):
    p = random_problem(d, n, levels, cap, seed=70 + d, sigma_range=(1.0, 1e-3), nr_feat=feat)
    p["window"][levels // 2] = 0.0
    enc, _ = make_encoding(d, p["sigmas"], p["shift"], concat_points=concat, nr_feat=feat)
    inp = gpu_input(p, need_table_grad=False)
    sf = orc.scale_factors(d, p["sigmas"])
    want = orc.forward(p["pos"], p["table"], sf, p["shift"], p["window"], concat_points=concat)
    assert np.array_equal(enc.forward(inp).cpu().numpy(), want)
    grad = np.concatenate([p["grad"], np.zeros((want.shape[0] - levels, feat, n), np.float32)])
    _, pg = enc.backward(inp, to_gpu(grad))
    wp = orc.backward_pos(p["pos"], p["table"], sf, p["shift"], p["window"], p["grad"])
    assert np.all(np.abs(pg.cpu().numpy() - wp["grad64"]) <= 1e-6 * wp["abs64"] + 1e-30)
    _, ggs = enc.double_backward_from_positions(inp, to_gpu(p["dpos"]), to_gpu(grad), want_lattice_values_grad=False)
    wd = orc.double_backward(p["pos"], p["table"], sf, p["shift"], p["window"], p["dpos"], p["grad"], concat_points=concat, want32=False, want64=False)
    assert np.array_equal(ggs.cpu().numpy(), wd["ggs"])


# d, n, levels, capacity, features: tables and batches beyond what the kernels that keep all levels of a block of points take, so that
# the position gradient gathers by groups of levels.  More and fewer groups than dies, a single one, a launch too large and a slice too
# large for segments
@pytest.mark.parametrize("d,n,levels,cap,feat", [(3, 30011, 17, 1 << 17, 2), (2, 60001, 9, 1 << 18, 2), (3, 200003, 2, 1 << 20, 2),
                                                 (3, 350003, 48, 1 << 15, 2), (3, 100003, 4, (1 << 20) + 1, 4)])
def test_position_gradient_of_every_group_and_point(d, n, levels, cap, feat):
    p = random_problem(d, n, levels, cap, seed=170 + d, sigma_range=(1.0, 1e-3), nr_feat=feat)
    enc, _ = make_encoding(d, p["sigmas"], p["shift"], nr_feat=feat)
    sf = orc.scale_factors(d, p["sigmas"])
    for masked in (None, levels // 2):
        if masked is not None:
            p["window"][masked] = 0.0
        _, pg = enc.backward(gpu_input(p, need_table_grad=False), to_gpu(p["grad"]))
        wp = orc.backward_pos(p["pos"], p["table"], sf, p["shift"], p["window"], p["grad"])
        assert np.all(np.abs(pg.cpu().numpy() - wp["grad64"]) <= 1e-6 * wp["abs64"] + 1e-30)
