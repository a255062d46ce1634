"""The K <= 32 samplers' ways of sharing rows out (pairs a wave; four rows a
wave; four, two or one a work-group; segments of heavy rows) against the FP64
oracle on identical FP32 inputs and draws.

Tolerance 1e-4 per row, the split-BF16 samplers' own: two parts keep 2^-17 of a
factor, a well-conditioned row (Lambda >= I here) multiplies that by the few
tens of its condition number."""
import numpy as np
import pytest

import oracle as O
from _gpu_helpers import SEED, announce, f32, gpu_sample_latents, row_rel_err, spd
from macau_amd import _lib

pytestmark = pytest.mark.gpu

TOL = 1e-4


# rows at the edges of each way; K at the edges of the 4-column steps; one, two
# and four other modes; nonzeros at the blocks' edges and above a segment
@pytest.mark.parametrize("N,K,nother", [
    (1, 17, 1), (3, 32, 1), (5, 20, 2), (511, 31, 1), (512, 32, 1), (513, 32, 2), (1024, 18, 1), (1025, 32, 4),
    (1203, 25, 3), (12000, 32, 1), (12001, 32, 1), (12003, 29, 2), (1, 1, 1), (3, 4, 1), (301, 5, 2), (8193, 10, 1),
    (8195, 16, 1), (700, 13, 4)])
def test_rows_per_wave(N, K, nother):
    announce("rows per wave N=%d K=%d other=%d" % (N, K, nother))
    rng = np.random.default_rng(N + K)
    nb = 400
    edges = [0, 1, 31, 32, 33, 63, 64, 65, 128, 129, 2048, 2049, 4100]
    deg = np.array([edges[i % len(edges)] if i < 2 * len(edges) else int(rng.integers(0, 12)) for i in range(N)])
    rng.shuffle(deg)
    r = np.repeat(np.arange(N), deg)
    idx = np.stack([r] + [rng.integers(0, nb, len(r)) for _ in range(nother)], 1).astype(np.int32)
    vals = rng.standard_normal(len(r))
    if nother == 1:
        modes, mean, _ = O.matrix_rows(idx[:, 0], idx[:, 1], vals, N, nb)
    else:
        modes, mean, _ = O.tensor_rows(idx, vals, [N] + [nb] * nother)
    others = [f32(0.5 * rng.standard_normal((nb, K))) for _ in range(nother)]
    Lam, mu = f32(spd(rng, K, 2.0)), f32(rng.standard_normal(K))
    ref = O.sample_latents(K, modes[0], mean, others, 3.0, mu, Lam, SEED, 2, 0)
    got = gpu_sample_latents(K, modes[0], mean, others, 3.0, mu, Lam, SEED, 2, 0, _lib.SAMPLER_BATCHED)
    e = row_rel_err(got, ref)
    print("rows per wave: row err %.3e" % e)
    assert e < TOL
