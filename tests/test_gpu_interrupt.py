"""Ctrl-C during macau_run: where the host takes part in every iteration (block
CG), the chain stops after the current one."""
import os
import signal
import threading
import time

import numpy as np
import pytest

from _gpu_helpers import SEED, GpuModel, announce
from macau_amd import _lib
from macau_amd._lib import check

pytestmark = pytest.mark.gpu


def test_interrupt_stops_a_block_cg_chain_after_the_current_iteration():
    announce("Ctrl-C in a block CG chain")
    L = _lib.lib()
    rng = np.random.default_rng(8)
    N, nc, nf = 20000, 100, 60000
    r = np.repeat(np.arange(N), 4)
    c = rng.integers(0, nc, len(r))
    y = rng.standard_normal(len(r))
    key = np.unique(np.repeat(np.arange(N), 40) * nf + rng.integers(0, nf, 40 * N))
    m = GpuModel(2, 32, 2.0)
    m.data(np.stack([r, c], 1), y, [N, nc], np.stack([r[:50], c[:50]], 1), y[:50])
    m.prior((key // nf, key % nf, None, N, nf), lambda_beta=0.01, tol=1e-12)
    m.prior()
    m.setup(20, 20, SEED, _lib.SAMPLER_BATCHED)  # a look at the state every ten of 40 iterations
    m.iterate(4)
    seen = []

    def interrupt():
        end = time.monotonic() + 60
        # macau_run starts over: the count falls back to 0, then grows
        while not 1 <= L.macau_get_iteration(m.h) <= 3 and time.monotonic() < end:
            time.sleep(0.0005)
        seen.append(L.macau_get_iteration(m.h))
        os.kill(os.getpid(), signal.SIGINT)

    old = signal.getsignal(signal.SIGINT)
    thread = threading.Thread(target=interrupt)
    try:
        t0 = time.monotonic()
        thread.start()
        check(L.macau_run(m.h))
        thread.join()
    finally:
        signal.signal(signal.SIGINT, old)
    done = L.macau_get_iteration(m.h)
    print("%.0f ms, Ctrl-C at iteration %d, stopped after %d" % (1e3 * (time.monotonic() - t0), seen[0], done))
    # the one under way, and one more should the signal come late
    assert 1 <= seen[0] <= done <= seen[0] + 2
