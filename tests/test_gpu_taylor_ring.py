"""Ghost rings and data collection made beside the step: runs of several
attempts per call (one graph) against the same attempts launched one by one,
where both are launches of their own, bit for bit -- states, counts and
measurement grids, with rejected attempts, a moving window, a batch whose
instances finish at different times, both precisions, and a run that ends in a
rejected attempt."""
import numpy as np
import pytest

import fivonagi_amd as fa
from fivonagi_amd import workloads as wl

pytestmark = pytest.mark.gpu


def taylor_at(T, eta, theta, dt0=0.005, moving=True):
    p = wl.taylor(eta, theta=theta, moving=moving)
    t = p.taylor
    x = np.arange(p.nx)[None, :] * p.dx
    y = (np.arange(p.ny)[:, None] - t["jc"]) * p.dy + t["yoff"]
    cs, sn = np.cos(theta), np.sin(theta)
    r = t["rhoa"] * np.tanh(t["c"] * (x * cs + y * sn - T))
    return fa.Problem(p.nx, p.ny, p.dx, p.dy, p.beta, p.delta, np.stack([r, r * cs, r * sn]),
                      cfl_wish=p.cfl_wish, dt0=dt0, T0=T, bc=p.bc, taylor=t, moving=p.moving)


def everything(ctx):
    return [(ctx.collect(k), ctx.measure(k), ctx.info(k)) for k in range(len(ctx.problems))]


def compare(a, b, counts=True):
    for ((qa, sa), ma, ia), ((qb, sb), mb, ib) in zip(a, b):
        assert np.array_equal(qa, qb)
        assert np.array_equal(ma, mb)
        assert sa == sb and (ia["md_x"], ia["md_y"]) == (ib["md_x"], ib["md_y"])


@pytest.mark.parametrize("fp64", [False, True])
def test_one_graph_equals_single_launches(fp64):
    # dt0 far above the limit: the first attempts are rejected
    probs = [taylor_at(5.9, 1, 0.0, dt0=0.9), taylor_at(5.9, 2, np.pi / 8),
             taylor_at(0.05, 1, np.pi / 16, moving=False),
             wl.hifu(nx=96, ny=190)]
    n = 40
    out = []
    for single in (False, True):
        print(f"[ring] fp64 {fp64} single {single}", flush=True)
        with fa.Context(probs, fp64=fp64) as ctx:
            for k, p in enumerate(probs[:3]):
                ctx.set_collect(k, **wl.taylor_collect(p, fp64))
            ctx.set_collect(3, **wl.hifu_collect(probs[3]))
            if single:
                for _ in range(n):
                    ctx.enqueue(1)
            else:
                ctx.enqueue(n)
            ctx.sync()
            out.append(everything(ctx))
    assert out[0][0][2]["n_rejected"] > 0 and out[0][1][2]["md_x"] > 0
    compare(*out)


def test_frames_end_at_their_own_times():
    """Instances of different resolution in frames: each alone gives the batch's
    result (its attempts past the frame's end do not run)."""
    probs = [taylor_at(5.0, e, 0.0) for e in (1, 2)]
    res = []
    for group in ([0, 1], [0], [1]):
        with fa.Context([probs[k] for k in group]) as ctx:
            for i, k in enumerate(group):
                ctx.set_collect(i, **wl.taylor_collect(probs[k]))
            for T in (5.5, 6.5, 7.5):
                ctx.step_until(T)
            res.append(everything(ctx))
    compare(res[0], res[1] + res[2])


def test_run_that_ends_in_a_rejected_attempt():
    """The state after a rejected last attempt holds the ghost cells that
    attempt read."""
    p = taylor_at(5.0, 1, 0.0, dt0=0.9, moving=False)
    with fa.Context(p) as ctx:
        ctx.enqueue(1)
        ctx.sync()
        assert ctx.info(0)["n_rejected"] == 1
        q, _ = ctx.collect(0)
    t = p.taylor
    x = np.arange(p.nx)[None, :] * p.dx
    r = t["rhoa"] * np.tanh(t["c"] * (x - p.T0)) * np.ones((p.ny, 1))
    ghost = np.ones((p.ny, p.nx), bool)
    ghost[2:-2, 2:-2] = False
    # the closed form in FP32 (a few ulp of its scale)
    assert np.abs(q[0][ghost] - r[ghost]).max() <= 4e-7 * abs(t["rhoa"])
    assert np.array_equal(q[:, 2:-2, 2:-2], p.q0[:, 2:-2, 2:-2])
