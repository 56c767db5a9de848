"""A Taylor instance that an imaginary eigenvalue stops: its state is the one the
failing attempt read, ghost cells at that attempt's time, however many attempts
the run launched after it."""
import numpy as np
import pytest

import fivonagi_amd as fa
from fivonagi_amd import workloads as wl

pytestmark = pytest.mark.gpu


def stopped(eta, theta, moving):
    """A Taylor problem whose first attempt fails (a cell at five times the
    speed of sound) and whose initial ghost cells are not the closed form."""
    p = wl.taylor(eta, theta=theta, moving=moving)
    q = p.q0_f64.copy()
    q[:, :2] = q[:, -2:] = q[:, :, :2] = q[:, :, -2:] = 0.0
    q[1, p.ny // 2, p.nx // 2] = 5.0
    return fa.Problem(p.nx, p.ny, p.dx, p.dy, p.beta, p.delta, q, dt0=p.dt0, T0=p.T0, bc=p.bc,
                      taylor=p.taylor, moving=p.moving)


@pytest.mark.parametrize("fp64", [False, True])
@pytest.mark.parametrize("attempts", [1, 4, 7, 40, 320])
def test_ghost_cells_after_an_error(attempts, fp64):
    good = wl.taylor(1, theta=np.pi / 8)
    probs = [stopped(1, 0.0, False), good, stopped(2, np.pi / 16, True)]
    print(f"[stop] {attempts} attempts fp64 {fp64}", flush=True)
    with fa.Context(probs, fp64=fp64) as ctx:
        ctx.enqueue(attempts)
        assert ctx.sync() == fa.ERR_EIGEN
        got = [ctx.collect(k)[0] for k in range(3)]
        assert ctx.info(1)["n_accepted"] == attempts
    with fa.Context(good, fp64=fp64) as ctx:
        ctx.step(attempts)
        assert np.array_equal(ctx.collect(0)[0], got[1])
    for k in (0, 2):
        p, q = probs[k], got[k]
        t, cs, sn = p.taylor, np.cos(p.taylor["theta"]), np.sin(p.taylor["theta"])
        x = np.arange(p.nx)[None, :] * p.dx
        y = (np.arange(p.ny)[:, None] - t["jc"]) * p.dy + t["yoff"]
        r = t["rhoa"] * np.tanh(t["c"] * (x * cs + y * sn - p.T0))
        want = np.stack([r, r * cs, r * sn])
        want[:, 2:-2, 2:-2] = p.q0_f64[:, 2:-2, 2:-2]
        # a few roundings of the closed form's argument, which is O(100)
        tol = (1e-12 if fp64 else 1e-4) * abs(t["rhoa"])
        ghost = np.ones((p.ny, p.nx), bool)
        ghost[2:-2, 2:-2] = False
        assert np.abs(q - want)[:, ghost].max() <= tol
        assert np.array_equal(q[:, ~ghost], want.astype(q.dtype)[:, ~ghost])
