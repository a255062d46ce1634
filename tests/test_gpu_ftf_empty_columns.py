"""The F^T F branch where most columns of F are empty (enumerated fingerprints,
the frequent ones first): the solve through the eigendecomposition against the
solve through Cholesky, same data and draws.

Tolerance: both are backward stable, so beta differs by at most a few n eps
times the conditioning (d_max + lambda) / lambda, below 1e5 here:
2000 x 1.1e-16 x 1e5 = 2.2e-8 (on empty columns both are y / lambda)."""
import numpy as np
import pytest

from _gpu_helpers import GpuModel, announce
from macau_amd import _lib

pytestmark = pytest.mark.gpu


def _fingerprints(rng, N, nf, per):
    w = np.arange(1, nf + 1) ** -1.5
    k = np.unique(np.repeat(np.arange(N), 8 * per) * nf + rng.choice(nf, 8 * per * N, p=w / w.sum()))
    r, f = k // nf, k % nf
    keep = np.arange(len(k)) - np.searchsorted(r, np.arange(N))[r] < per
    return r[keep], f[keep]


# seeds 2 and 4: eigenvectors that are not orthogonal on the empty columns when
# all columns are decomposed (beta off by 7e-3 and 1e-2)
@pytest.mark.parametrize("seed,N,nf,K,values", [(2, 15000, 2000, 32, False), (4, 15000, 2000, 32, False),
                                                (4, 15000, 2000, 70, True), (1, 300, 200, 5, True)])
def test_spectral_solve_with_empty_columns(seed, N, nf, K, values, monkeypatch):
    announce("F^T F with empty columns seed=%d nf=%d K=%d" % (seed, nf, K))
    rng = np.random.default_rng(seed)
    fr, fc = _fingerprints(rng, N, nf, min(60, nf // 10))
    fv = rng.uniform(0.5, 1.5, len(fr)) if values else None
    r = np.repeat(np.arange(N), 4)
    c = rng.integers(0, 100, len(r))
    y = rng.standard_normal(len(r)) + 3
    beta = []
    for solver in ("spectral", "cholesky"):
        monkeypatch.setenv("MACAU_AMD_FTF_SOLVER", solver)
        m = GpuModel(2, K, 4.0)
        m.data(np.stack([r, c], 1), y, [N, 100], np.stack([r[:50], c[:50]], 1), y[:50])
        m.prior((fr, fc, fv, N, nf), 5.0, 1e-6, 10000)
        m.prior()
        m.setup(2, 50, seed, _lib.SAMPLER_BATCHED)
        assert _lib.lib().macau_get_ftf_solver(m.h, 0) == (2 if solver == "spectral" else 1)
        m.iterate(1)
        beta.append(m.link(0, nf))
    empty = np.setdiff1d(np.arange(nf), fc)
    assert len(empty) > nf // 4
    e = [np.linalg.norm(beta[0][s] - beta[1][s]) / np.linalg.norm(beta[1][s]) for s in (fc, empty)]
    print("beta: used columns %.1e, empty ones %.1e" % tuple(e))
    assert e[0] < 2.2e-8 and e[1] < 1e-13


# equal columns among the non-empty ones make a null space too; without a shift
# of the decomposed matrix the eigenvectors of these two were not orthogonal there
@pytest.mark.parametrize("seed,nf", [(18, 1872), (29, 1921)])
def test_equal_columns_keep_the_spectral_solve(seed, nf, monkeypatch):
    announce("F^T F with equal columns seed=%d nf=%d" % (seed, nf))
    rng = np.random.default_rng(seed)
    assert rng.integers(800, 2000) == nf
    N, K = 12000, 8
    fr, fc = _fingerprints(rng, N, nf, 60)
    r = np.arange(N)
    beta = []
    for solver in ("spectral", "cholesky"):
        monkeypatch.setenv("MACAU_AMD_FTF_SOLVER", solver)
        m = GpuModel(2, K, 4.0)
        m.data(np.stack([r, r % 20], 1), np.sin(r), [N, 20], np.stack([r[:50], r[:50] % 20], 1), np.sin(r[:50]))
        m.prior((fr, fc, None, N, nf), 5.0, 1e-6, 10000)
        m.prior()
        m.setup(2, 50, 1, _lib.SAMPLER_BATCHED)
        assert _lib.lib().macau_get_ftf_solver(m.h, 0) == (2 if solver == "spectral" else 1)
        m.iterate(1)
        beta.append(m.link(0, nf))
    e = np.linalg.norm(beta[0] - beta[1]) / np.linalg.norm(beta[1])
    print("beta: %.1e" % e)
    assert e < 2.2e-8
