"""The scatter's way to a point's simplex (a sorting network over the residuals, vertices in cyclic order) against the oracle:
the slots and weights it gives the vertices, bit for bit, over the forms it accepts."""
import numpy as np
import pytest
import torch

from helpers import make_encoding, to_gpu
from oracle import api as orc

pytestmark = pytest.mark.gpu

FIRST_ORDER, BOTH_ORDERS = 2, 3


def check(enc, pos, sf, shift, capacity):
    want = orc.simplex(pos, sf, shift, capacity)
    for routine in (FIRST_ORDER, BOTH_ORDERS):
        got = enc.simplex_debug(to_gpu(pos), capacity, gather_path=routine)
        weights, slots = got["barycentric"].cpu().numpy(), got["slot"].cpu().numpy()
        assert np.array_equal(weights, want["bary"]), routine
        # first order, D + 1 a power of two: two equal residuals leave open which vertex has the weight 0 between them
        open_vertices = (weights == 0) if routine == FIRST_ORDER and pos.shape[1] in (3, 7) else np.zeros_like(weights, bool)
        assert np.array_equal(slots[~open_vertices], want["slot"][~open_vertices]), routine
        assert slots.min() >= 0 and slots.max() < capacity


# what the key's lower word has to carry: all 32 bits of the hash (not a power of two, more than 2^28 slots), fewer, one slot
@pytest.mark.parametrize("capacity", [1, 1 << 18, 1 << 28, 1 << 29, 100003, (1 << 30) - 1])
@pytest.mark.parametrize("d", [2, 3, 4, 5, 6, 7, 8])
def test_slots_and_weights(d, capacity):
    rng = np.random.default_rng(100 * d)
    levels, n = min(10, ((1 << 31) - 1) // (2 * capacity)), 4001
    sigmas = np.geomspace(1e-4, 1.0, levels).astype(np.float32)  # residuals of fine levels tie often: coordinates of 10^4, exact to 10^-3
    shift = (rng.standard_normal((levels, d)) * 10).astype(np.float32)
    pos = rng.uniform(-1, 1, (n, d)).astype(np.float32)
    pos[1::2] = np.round(pos[1::2] * 8) / 8  # several equal coordinates
    enc, _ = make_encoding(d, sigmas, shift)
    check(enc, pos, orc.scale_factors(d, sigmas), shift, capacity)


@pytest.mark.parametrize("d", [2, 3, 4, 5, 6, 7, 8])
def test_points_on_ties_and_faces(d):
    rng = np.random.default_rng(d)
    pos = (rng.integers(-40, 41, size=(20000, d)) * 0.25).astype(np.float32)
    pos[:200, 1:] = 0.0
    pos[:200, 0] = (np.arange(200) - 100) * 0.25 * (d + 1)
    pos[200:210] = 0.0
    pos[210:220] = -0.0
    pos[220:230] = 1e-42  # subnormal
    pos[230:240] = -1e-30
    sf, shift = np.ones((1, d), np.float32), np.zeros((1, d), np.float32)
    enc, fp = make_encoding(d, np.ones(1, np.float32), shift)
    fp.m_scale_factor = torch.ones((1, d), device="cuda")
    check(enc, pos, sf, shift, 1 << 16)


@pytest.mark.parametrize("d", [2, 3, 4, 5, 6, 7, 8])
def test_weights_of_points_without_a_place(d):
    """A coordinate that is not finite, or overflows, gives weights that are NaN, as every other pass does, and slots within the table."""
    rng = np.random.default_rng(d)
    pos = rng.uniform(-1, 1, (4 * d + 100, d)).astype(np.float32)
    for i in range(d):
        pos[4 * i:4 * i + 4, i] = [np.nan, np.inf, -np.inf, 3e38]
    levels, capacity = 2, 100003
    shift = np.zeros((levels, d), np.float32)
    enc, _ = make_encoding(d, np.array([1e-2, 1e-4], np.float32), shift)
    for routine in (FIRST_ORDER, BOTH_ORDERS):
        got = enc.simplex_debug(to_gpu(pos), capacity, gather_path=routine)
        weights, slots = got["barycentric"].cpu().numpy(), got["slot"].cpu().numpy()
        bad = np.isnan(weights)
        print(d, routine, weights.shape)
        assert bad.all(-1)[:, :4 * d].all() and not bad[:, 4 * d:].any()
        assert slots.min() >= 0 and slots.max() < capacity
