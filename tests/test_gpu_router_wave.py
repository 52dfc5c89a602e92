"""ROUTER_SEL on one wave per token against the oracle: every expert count to
64, every top_k to 8, ties, logits far below the maximum, and a NaN."""
import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu


def run(flh, gpu, lg, K, norm):
    n, E = lg.shape
    dl = flh.DeviceBuffer.from_array(lg, gpu)
    di, dg = flh.DeviceBuffer(4 * n * K), flh.DeviceBuffer(4 * n * K)
    flh.router_sel(dl, n, E, K, norm, 1.5, di, dg, gpu)
    return di.download(np.uint32, n * K, gpu).reshape(n, K), dg.download(np.float32, n * K, gpu).reshape(n, K)


@pytest.mark.parametrize("E,K", [(1, 1), (2, 2), (7, 3), (8, 2), (8, 8), (9, 1), (31, 8), (33, 4), (60, 4), (63, 6), (64, 8)])
def test_router_wave(flh, orc, gpu, E, K):
    say("router wave", E, K)
    rng = np.random.default_rng(E * 10 + K)
    lg = rng.standard_normal((12, E)).astype(np.float32)
    lg[1] = 0.25                                       # all equal: experts in ascending order
    lg[2] = np.round(lg[2])                            # ties
    lg[3] *= 60                                        # weights that underflow to 0
    lg[4] = -np.inf
    lg[4, E // 2] = 1.0                                # one expert left, the others at weight 0
    for norm in (0, 1):
        ids, gates = run(flh, gpu, lg, K, norm)
        for t in range(lg.shape[0]):
            wi, wg = orc.router_sel(lg[t], K, norm, 1.5)
            assert len(set(ids[t])) == K, t
            # equal logits may not change places (t = 1, 2, 4); weights one expf
            # rounding apart may
            same = np.array_equal(ids[t], wi)
            assert same or (t not in (1, 2, 4) and np.allclose(lg[t][ids[t]], lg[t][wi], rtol=0, atol=1e-6)), t
            assert np.allclose(gates[t], wg, rtol=2e-6, atol=0), t


def test_router_wave_nan(flh, orc, gpu):
    """A NaN logit makes every weight NaN: nothing beats -1, expert 0 is chosen
    each time with that weight, as the reference's scan does."""
    lg = np.random.default_rng(3).standard_normal((2, 16)).astype(np.float32)
    lg[1, 5] = np.nan
    ids, gates = run(flh, gpu, lg, 3, 0)
    wi, wg = orc.router_sel(lg[1], 3, 0, 1.5)
    assert np.array_equal(ids[1], wi) and np.array_equal(gates[1], wg)
