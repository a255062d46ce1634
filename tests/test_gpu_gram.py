"""The link-matrix updates on F's non-empty columns against the FP64 oracle.

After one iteration the oracle updates the prior from the device's own factors
(FP32 values, exact inputs for both), so only FP64 arithmetic is compared.

Univariate sweep: 1e-8 relative, FP64 rounding (1e-16) through a few hundred
sequential updates of well-conditioned sums, with a margin of 1e4.  Block CG: both
stop at a relative residual of 1e-6 after the same number of iterations up to
one; a solution's error is at most the residual times the condition number of
F^T F + lambda_beta I, which stays below 10 here: 1e-5."""
import numpy as np
import pytest

import oracle as O
from _gpu_helpers import SEED, GpuModel, announce, rel_err
from macau_amd import _lib

pytestmark = pytest.mark.gpu


def _side(rng, N, n, nempty, per, kind):
    """n columns with about `per` entries among n + nempty, at random places."""
    nfeat = n + nempty
    cols = np.sort(rng.permutation(nfeat)[:n])
    fr = np.concatenate([rng.choice(N, min(per, N), replace=False) for _ in range(n)])
    fc = np.repeat(cols, min(per, N))
    if kind == "repeated":
        fr, fc = np.concatenate([fr, fr[::3]]), np.concatenate([fc, fc[::3]])
    fv = np.ones(len(fr)) if kind == "ones" else rng.standard_normal(len(fr))
    order = rng.permutation(len(fr))
    return fr[order].astype(np.int32), fc[order].astype(np.int32), fv[order], nfeat


def _model(rng, N, K, graph, add):
    ncol = 30
    r, c = np.nonzero(rng.random((N, ncol)) < 0.1)
    m = GpuModel(2, K, 5.0)
    m.data(np.stack([r, c], 1), rng.standard_normal(len(r)), [N, ncol])
    add(m)
    m.prior()
    m.setup(3, 3, SEED, _lib.SAMPLER_PLAIN_FP32 if K > 32 else _lib.SAMPLER_BATCHED, graph=graph)
    m.iterate(1)
    return m


# n at the edges of the 64-wide steps and the 16-wide tiles; N on both sides of
# the 16-row step and of the residuals' LDS form; kinds of F; 1000 x 3 entries
# stays on the walk over the entries
@pytest.mark.parametrize("N,n,nempty,per,K,kind", [
    (50, 1, 0, 20, 3, "ones"), (333, 15, 3, 40, 8, "values"), (333, 16, 0, 40, 10, "repeated"),
    (1000, 63, 200, 100, 16, "values"), (1000, 64, 0, 100, 17, "ones"), (1000, 65, 5, 300, 32, "repeated"),
    (2000, 300, 1000, 300, 40, "values"), (19500, 129, 7, 500, 5, "ones"), (2000, 1000, 0, 3, 8, "values")])
def test_univariate_sweep_on_columns(N, n, nempty, per, K, kind):
    announce("univariate sweep N=%d n=%d empty=%d per=%d K=%d %s" % (N, n, nempty, per, K, kind))
    rng = np.random.default_rng(N + n + K)
    fr, fc, fv, nfeat = _side(rng, N, n, nempty, per, kind)
    m = _model(rng, N, K, False,
               lambda m: m.one_prior((fr, fc, None if kind == "ones" else fv, N, nfeat), lambda_beta=2.0))
    F, Ft = O.csr_pair(fr, fc, fv, N, nfeat)
    colsq = np.bincount(fc, weights=fv ** 2, minlength=nfeat)
    _, _, beta, _, lb = O.macau_one_update_prior(
        m.latents(0, N), F, Ft, colsq, np.zeros(K), np.full(K, 10.0), np.zeros((nfeat, K)), np.zeros((N, K)),
        np.full(K, 2.0), SEED, 0, 0)
    e = rel_err(m.link(0, nfeat), beta)
    lbg = _lib.lib().macau_get_link_lambda(m.h, 0)
    print("sweep on columns: beta err %.3e, lambda_beta %.12f vs %.12f" % (e, lbg, lb.mean()))
    assert e < 1e-8
    assert abs(lbg - lb.mean()) < 1e-8 * lb.mean()


# non-empty columns at the tiles' edges, 127 and 128 empty ones (the second
# replaces them), F's products (300 x 1, 2100) and its Gram matrix, K at the
# 16-wide tiles' edges and above 32 (never replaced)
@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("N,n,nempty,per,K,kind", [
    (50, 1, 128, 20, 3, "ones"), (333, 15, 128, 10, 8, "values"), (333, 16, 127, 10, 10, "repeated"),
    (1000, 63, 200, 30, 16, "values"), (1000, 64, 5000, 30, 17, "ones"), (1000, 65, 300, 30, 31, "repeated"),
    (2000, 300, 1000, 20, 32, "values"), (2000, 300, 500, 1, 32, "ones"), (3000, 2100, 700, 8, 32, "ones"),
    (3000, 2100, 700, 8, 20, "values"), (1000, 100, 400, 20, 40, "ones")])
def test_block_cg_on_columns(N, n, nempty, per, K, kind, graph):
    announce("block CG N=%d n=%d empty=%d per=%d K=%d %s graph=%d" % (N, n, nempty, per, K, kind, graph))
    rng = np.random.default_rng(N + n + K)
    fr, fc, fv, nfeat = _side(rng, N, n, nempty, per, kind)
    lb0 = 5.0 * per
    m = _model(rng, N, K, graph,
               lambda m: m.prior(side=(fr, fc, None if kind == "ones" else fv, N, nfeat), lambda_beta=lb0, tol=1e-6))
    F, Ft = O.csr_pair(fr, fc, fv, N, nfeat)
    mu, Lam, beta, _, lb, it = O.macau_update_prior(m.latents(0, N), F, Ft, np.zeros((nfeat, K)), np.zeros((N, K)), lb0,
                                                    SEED, 0, tol=1e-6)
    e = rel_err(m.link(0, nfeat), beta)
    itg = _lib.lib().macau_get_last_cg_iters(m.h, 0)
    print("CG on columns: beta err %.3e, iterations %d vs %d" % (e, itg, it))
    assert e < 1e-5
    assert abs(itg - it) <= 1
    assert abs(_lib.lib().macau_get_link_lambda(m.h, 0) - lb) < 1e-5 * lb
