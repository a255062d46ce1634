"""The Normal-Wishart draw at the edges of its 16 x 16 tiles.

Every number of tiles (1 to 8), with a last tile that is full, one column
short and one column wide, against the FP64 oracle.  Tolerance: the draw is
FP64 throughout; K rounding steps of 1.1e-16 amplified by the conditioning of
X (below 1e3 here) stay below 128 * 1.1e-16 * 1e3 = 1.4e-11.
"""
import numpy as np
import pytest

import oracle as O
from _gpu_helpers import SEED, announce, gpu_cond_normal_wishart, spd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 80, 96, 97, 112, 113, 127, 128])
def test_draw_at_tile_edges(K):
    announce("Normal-Wishart draw K=%d" % K)
    rng = np.random.default_rng(K)
    N = 40 + 7 * K
    U = rng.standard_normal((N, K)) * 0.7 + 0.2
    T, mu0 = spd(rng, K, 1.0), rng.standard_normal(K) * 0.1
    mu, Lam = gpu_cond_normal_wishart(U, mu0, 2.0, T, K + 2.0, SEED, 5, 1)
    mur, Lamr = O.cond_normal_wishart(U, mu0, 2.0, T, K + 2.0, SEED, 5, 1)
    assert np.linalg.norm(mu - mur) <= 1.4e-11 * np.linalg.norm(mur)
    assert np.linalg.norm(Lam - Lamr) <= 1.4e-11 * np.linalg.norm(Lamr)
    np.testing.assert_array_equal(Lam, Lam.T)


@pytest.mark.parametrize("K", [5, 20, 64, 100])
def test_draw_of_an_indefinite_scale_fails(K):
    announce("Normal-Wishart draw of an indefinite scale, K=%d" % K)
    rng = np.random.default_rng(K)
    T = np.eye(K)
    T[K // 2, K // 2] = -1e6
    with pytest.raises(RuntimeError, match="not positive definite"):
        gpu_cond_normal_wishart(rng.standard_normal((200, K)), np.zeros(K), 2.0, T, K + 2.0, SEED, 0, 0)
