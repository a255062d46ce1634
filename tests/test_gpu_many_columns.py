"""The Normal-Wishart draw of K > 64 around the column count from which its
statistics take more work-groups, against the FP64 oracle.

Tolerance: sums of 32768 terms in sequence (the oracle's) are off by at most
32768 x 1.1e-16 = 3.6e-12 of the terms' size, the draw's K rounding steps by
1.4e-14, amplified by the conditioning of X (below 3: independent columns, many
more than K): 1.1e-11."""
import numpy as np
import pytest

import oracle as O
from _gpu_helpers import SEED, announce, gpu_cond_normal_wishart, spd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,N", [(65, 8193), (65, 32767), (65, 32768), (128, 32801)])
def test_draw_of_many_columns(K, N):
    announce("Normal-Wishart draw K=%d N=%d" % (K, N))
    rng = np.random.default_rng(K + N)
    U = rng.standard_normal((N, K)) * 0.7 + 0.2
    T, mu0 = spd(rng, K, 1.0), rng.standard_normal(K) * 0.1
    mu, Lam = gpu_cond_normal_wishart(U, mu0, 2.0, T, K + 2.0, SEED, 5, 1)
    mur, Lamr = O.cond_normal_wishart(U, mu0, 2.0, T, K + 2.0, SEED, 5, 1)
    assert np.linalg.norm(mu - mur) <= 1.1e-11 * np.linalg.norm(mur)
    assert np.linalg.norm(Lam - Lamr) <= 1.1e-11 * np.linalg.norm(Lamr)
