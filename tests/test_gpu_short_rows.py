"""K in (16, 32], some thousand short rows: which of the sampler's ways takes
them depends on the rows and on the longest one.  Against the FP64 oracle on
identical FP32 inputs and draws, tolerance 1e-4 per row (the split-BF16
samplers' own)."""
import numpy as np
import pytest

import oracle as O
from _gpu_helpers import SEED, announce, f32, gpu_sample_latents, row_rel_err, spd
from macau_amd import _lib

pytestmark = pytest.mark.gpu


# N rows of at most `most` nonzeros: both sides of most = N / 12 (four a wave up
# to there, a work-group's four above), of 3000 and of 12000 rows
@pytest.mark.parametrize("N,most,K,nother", [
    (3000, 5, 32, 1), (3001, 250, 17, 1), (3001, 251, 32, 2), (6007, 64, 20, 1), (6007, 65, 32, 4), (12000, 3, 31, 1),
    (12000, 1000, 32, 1), (12000, 1001, 24, 1), (12001, 33, 32, 3)])
def test_short_rows(N, most, K, nother):
    announce("short rows N=%d most=%d K=%d other=%d" % (N, most, K, nother))
    rng = np.random.default_rng(N + most)
    nb = 500
    deg = rng.integers(0, min(most, 30) + 1, N)
    deg[rng.integers(0, N)] = most
    r = np.repeat(np.arange(N), deg)
    idx = np.stack([r] + [rng.integers(0, nb, len(r)) for _ in range(nother)], 1).astype(np.int32)
    modes, mean, _ = O.tensor_rows(idx, rng.standard_normal(len(r)), [N] + [nb] * nother)
    others = [f32(0.5 * rng.standard_normal((nb, K))) for _ in range(nother)]
    Lam, mu = f32(spd(rng, K, 2.0)), f32(rng.standard_normal(K))
    ref = O.sample_latents(K, modes[0], mean, others, 3.0, mu, Lam, SEED, 2, 0)
    got = gpu_sample_latents(K, modes[0], mean, others, 3.0, mu, Lam, SEED, 2, 0, _lib.SAMPLER_BATCHED)
    e = row_rel_err(got, ref)
    print("short rows: row err %.3e" % e)
    assert e < 1e-4
