"""Tuned launch shapes belong to the kernels they were measured on: K <= 16 and
K in (16, 32] share a padded size but not their kernels, and above K = 64 the
caps count work-groups of eight waves."""
import numpy as np
import pytest

from _gpu_helpers import SEED, GpuModel, announce, power_law_rows, row_rel_err
from macau_amd import _lib
from macau_amd._lib import check, ptr

pytestmark = pytest.mark.gpu

NROW, NCOL = 900, 700


def _model(K):
    rng = np.random.default_rng(78)
    r, c, y = power_law_rows(rng, NROW, NCOL, 20000, heavy=(700, 650))
    m = GpuModel(2, K, "adaptive")
    m.data(np.stack([r, c], 1), y, [NROW, NCOL], np.stack([r[:100], c[:100]], 1), y[:100])
    m.prior()
    m.prior()
    m.setup(2, 6, SEED, _lib.SAMPLER_BATCHED)
    return m


def _knobs(m, mode):
    k = np.zeros(4, dtype=np.int32)
    tuned = _lib.lib().macau_get_tuning(m.h, mode, ptr(k))
    assert tuned in (0, 1), _lib.last_error()
    return tuned, k.tolist()


def test_a_shape_is_found_for_its_own_kernels_only(tmp_path, monkeypatch):
    announce("tuned shapes of K = 10 and K = 32")
    rec = str(tmp_path / "tune.txt")
    m = _model(10)
    check(_lib.lib().macau_autotune(m.h, 1, rec.encode(), None, None))
    monkeypatch.setenv("MACAU_AMD_TUNE_CACHE", rec)
    assert [_knobs(_model(K), 0)[0] for K in (16, 17, 32)] == [1, 0, 0]


def test_caps_above_64_are_honoured_and_reported(tmp_path, monkeypatch):
    announce("caps at K = 70")
    monkeypatch.setenv("MACAU_AMD_TUNE_DISABLE", "1")
    a = _model(70)
    assert _knobs(a, 0) == (0, [2048, 256, 256, 16384])
    rec = str(tmp_path / "tune.txt")
    check(_lib.lib().macau_autotune(a.h, 1, rec.encode(), None, None))
    # segments of 256 nonzeros, three work-groups for the light rows, one for the heavy ones
    out = []
    for ln in open(rec).read().splitlines():
        f = ln.split()
        out.append(" ".join(f[:6] + ["256", "3", "1", "8"] + f[10:]))
    open(rec, "w").write("\n".join(out) + "\n")
    monkeypatch.delenv("MACAU_AMD_TUNE_DISABLE")
    monkeypatch.setenv("MACAU_AMD_TUNE_CACHE", rec)
    b = _model(70)
    assert _knobs(b, 0) == (1, [256, 3, 1, 8])
    a.iterate(3)
    b.iterate(3)
    for mode, n in ((0, NROW), (1, NCOL)):
        assert row_rel_err(b.latents(mode, n), a.latents(mode, n)) < 1e-5
    assert abs(a.alpha() - b.alpha()) <= 1e-6 * a.alpha()


def test_caps_beyond_the_limit_are_cut(tmp_path, monkeypatch):
    """A table's caps reach the kernels at most as large as what the partial sums'
    slots are sized for (36000 rows are 18000 pairs, the largest cap 16384)."""
    announce("caps beyond the limit")
    rng = np.random.default_rng(5)
    N = 36000
    r, c, y = np.arange(N), rng.integers(0, 50, N), rng.standard_normal(N)

    def model():
        m = GpuModel(2, 10, "adaptive")
        m.data(np.stack([c, r], 1), y, [50, N], np.stack([c[:50], r[:50]], 1), y[:50])
        m.prior()
        m.prior()
        m.setup(2, 6, SEED, _lib.SAMPLER_BATCHED)
        return m

    monkeypatch.setenv("MACAU_AMD_TUNE_DISABLE", "1")
    a = model()
    rec = str(tmp_path / "tune.txt")
    check(_lib.lib().macau_autotune(a.h, 1, rec.encode(), None, None))
    lines = [" ".join(ln.split()[:6] + ["2048", "16384", "4096", "16384"]) for ln in open(rec).read().splitlines()]
    open(rec, "w").write("\n".join(lines).replace(" 16384 4096 ", " 1000000 1000000 ") + "\n")
    monkeypatch.delenv("MACAU_AMD_TUNE_DISABLE")
    monkeypatch.setenv("MACAU_AMD_TUNE_CACHE", rec)
    b = model()
    a.iterate(2)
    b.iterate(2)
    assert row_rel_err(b.latents(1, N), a.latents(1, N)) < 1e-5
    assert abs(a.alpha() - b.alpha()) <= 1e-6 * a.alpha()
