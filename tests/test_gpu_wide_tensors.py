"""The K > 64 sampler on matrices and tensors with one to four other modes,
rows below and above a segment, against the FP64 oracle on identical FP32
inputs and draws.

Which component blocks are compiled depends on K and on the number of other
modes, so K stands at the edges of the 16-component blocks.  Device memory is
left full of NaN first, and the same rows are sampled at K = 128 before: what a
kernel reads without anyone having written it then shows.

Tolerance 1e-4 per row, the split-BF16 samplers' own (three parts keep 24 bits
of a factor here; Lambda >= 2 I)."""
import ctypes

import numpy as np
import pytest

import oracle as O
from _gpu_helpers import SEED, announce, f32, gpu_sample_latents, row_rel_err, spd
from macau_amd import _lib


pytestmark = pytest.mark.gpu

TOL = 1e-4


def _leave_nan(nbytes):
    """Allocate nbytes of device memory, fill it with NaN and give it back."""
    _lib.lib()
    hip = ctypes.CDLL("libamdhip64.so.7")  # the copy that the library is linked to
    p = ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(nbytes)) == 0
    assert hip.hipMemset(p, 0xFF, ctypes.c_size_t(nbytes)) == 0
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipFree(p) == 0


# rows at the edges of the ways they are shared out: eight, four, two waves a row,
# one, and a wave's second row
@pytest.mark.parametrize("N,K,nother", [
    (1, 128, 1), (255, 65, 1), (256, 97, 2), (257, 128, 1), (300, 80, 4), (511, 100, 1), (512, 128, 3), (513, 81, 1),
    (1023, 112, 1), (1024, 66, 2), (1025, 128, 1), (2049, 113, 1)])
def test_wide_rows_per_wave(N, K, nother):
    announce("wide rows N=%d K=%d other=%d" % (N, K, nother))
    rng = np.random.default_rng(N + K)
    nb = 400
    edges = [2049, 1, 31, 32, 33, 63, 64, 65, 128, 255, 256, 257, 2048, 0]
    deg = np.array([edges[i % len(edges)] if i < 2 * len(edges) else int(rng.integers(0, 12)) for i in range(N)])
    rng.shuffle(deg)
    r = np.repeat(np.arange(N), deg)
    idx = np.stack([r] + [rng.integers(0, nb, len(r)) for _ in range(nother)], 1).astype(np.int32)
    modes, mean, _ = O.tensor_rows(idx, rng.standard_normal(len(r)), [N] + [nb] * nother)
    others = [f32(0.7 * rng.standard_normal((nb, K))) for _ in range(nother)]
    Lam, mu = f32(spd(rng, K, 2.0)), f32(rng.standard_normal(K))
    ref = O.sample_latents(K, modes[0], mean, others, 3.0, mu, Lam, SEED, 2, 0)
    got = gpu_sample_latents(K, modes[0], mean, others, 3.0, mu, Lam, SEED, 2, 0, _lib.SAMPLER_BATCHED)
    e = row_rel_err(got, ref)
    print("wide rows: row err %.3e" % e)
    assert e < TOL


@pytest.mark.parametrize("nother", [1, 2, 3, 4])
@pytest.mark.parametrize("K", [65, 80, 81, 97, 112, 113])
def test_wide_tensor_rows(K, nother):
    announce("wide tensor K=%d other=%d" % (K, nother))
    rng = np.random.default_rng(100 * K + nother)
    nb = 300
    deg = np.array([2048, 2049, 4100, 0, 1, 31, 33, 64, 700, 5000, 12, 3])
    N = len(deg)
    r = np.repeat(np.arange(N), deg)
    idx = np.stack([r] + [rng.integers(0, nb, len(r)) for _ in range(nother)], 1).astype(np.int32)
    vals = rng.standard_normal(len(r))
    # matrices too as tensors' rows: cells may repeat
    modes, mean, _ = O.tensor_rows(idx, vals, [N] + [nb] * nother)

    def sample(k, it):
        others = [f32(0.7 * rng.standard_normal((nb, k))) for _ in range(nother)]
        Lam, mu = f32(spd(rng, k, 2.0)), f32(rng.standard_normal(k))
        return others, Lam, mu, gpu_sample_latents(k, modes[0], mean, others, 3.0, mu, Lam, SEED, it, 0,
                                                   _lib.SAMPLER_BATCHED)

    nseg = int(np.sum((deg[deg > 2048] + 2047) // 2048))
    _leave_nan(nseg * (128 * 128 + 64) * 4)
    sample(128, 1)
    others, Lam, mu, got = sample(K, 2)
    ref = O.sample_latents(K, modes[0], mean, others, 3.0, mu, Lam, SEED, 2, 0)
    e = row_rel_err(got, ref)
    print("wide tensor: row err %.3e" % e)
    assert e < TOL
