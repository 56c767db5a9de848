"""Downloads (fivonagi_collect): a state that has not been stepped comes back
bit for bit, through the small path, the ring of staging slots (fewer and more
chunks than slots, a ragged last one) and from two host threads at once; and
step targets written by a launch, several calls in a row on a batch."""
import threading

import numpy as np
import pytest

import fivonagi_amd as fa
from fivonagi_amd import workloads as wl

pytestmark = pytest.mark.gpu


def problem(nx, ny, seed):
    rng = np.random.default_rng(seed)
    p = wl.gauss_pulse(nx, ny)
    p.q0_f64 = 1e-3 * rng.standard_normal((3, ny, nx))
    p.q0 = p.q0_f64.astype(np.float32)
    return p


# 3 fields of 4 or 8 bytes: below, just past and well past 4 MiB, past 16 MiB
@pytest.mark.parametrize("nx,ny", [(8, 8), (683, 512), (701, 509), (1333, 1051), (2049, 1027)])
@pytest.mark.parametrize("fp64", [False, True])
def test_collect_returns_the_state(nx, ny, fp64):
    print(f"[collect] {nx}x{ny} fp64 {fp64}", flush=True)
    probs = [problem(nx, ny, s) for s in (1, 2)]
    ctxs = [fa.Context(p, fp64=fp64) for p in probs]
    got = [None, None]

    def work(k):
        for _ in range(3):
            got[k] = ctxs[k].collect(0)[0]

    threads = [threading.Thread(target=work, args=(k,)) for k in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k, p in enumerate(probs):
        assert np.array_equal(got[k], p.q0_f64 if fp64 else p.q0)
        ctxs[k].close()


def test_targets_of_consecutive_calls():
    probs = [wl.gauss_pulse(64 + 9 * k, 40 + 5 * k, sigma_cells=4.0) for k in range(3)]
    with fa.Context(probs) as a, fa.Context(probs) as b:
        a.step(13)
        for n in (1, 0, 4, 8):
            b.step(n)
        b.enqueue(2)
        b.enqueue(1)
        b.sync()
        a.step(3)
        for k in range(3):
            (qa, sa), (qb, sb) = a.collect(k), b.collect(k)
            assert np.array_equal(qa, qb) and sa == sb and sa["n_accepted"] == 16
