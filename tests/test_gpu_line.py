"""evh_run on a 1-D grid, one kernel per step, against the same steps taken one
by one through the staged kernels (evh_step): q, w, evo, s, times and stops
bit for bit.  A block of the kernel takes 252 cells, and rows above 4096 such
pieces give a block several."""
import numpy as np
import pytest

from evora_amd import hydro, ics

pytestmark = pytest.mark.gpu


def _state(p, seed=5):
    q = ics.sod(p)
    x = np.arange(p.nx)
    r = np.random.default_rng(seed).uniform(-1, 1, (4, p.nx))
    q[0, 0, :, 0] *= 1 + 1e-2 * r[0]
    for i in range(3):  # the shear and a velocity on both sides of zero
        q[0, 0, :, 1 + i] = q[0, 0, :, 0] * (0.3 * r[1 + i] + 0.2 * np.sin(0.01 * x + i))
    q[..., 4] += 0.5 * (q[..., 1:4] ** 2).sum(-1) / q[..., 0]
    return q


def _steps(h, n, t=0.0, tend=1e99):
    go, dt, done = True, 0.0, 0
    while go and done < n:
        t, dt, go = h.step(t, tend)
        done += 1
    return t, dt, done


@pytest.mark.parametrize("n,solver,limiter,bound,kw", [
    (2, 2, 1, 1, {}), (2, 1, 2, 2, {}), (3, 2, 3, 3, {}), (249, 2, 2, 2, {}), (250, 2, 1, 3, {}), (251, 1, 1, 1, {}),
    (252, 2, 3, 2, {}), (253, 1, 3, 3, {}), (254, 2, 2, 1, {}), (505, 2, 1, 3, {}), (1000, 2, 1, 1, {}),
    (1000, 1, 2, 2, {"secondorder": False}), (777, 2, 1, 2, {"dualenergy": True, "de_thresh": 0.1}),
    (1100003, 2, 2, 3, {}),
])
def test_line_equals_staged_steps(n, solver, limiter, bound, kw):
    p = ics.sod_params(n, solver=solver, limiter=limiter, boundtype=bound, cfl=0.4, **kw)
    q0 = _state(p)
    many, few = (70, 9) if n < 10**6 else (3, 3)
    out = []
    for drive in (hydro.Hydro.run, _steps):
        with hydro.Hydro(p) as h:
            h.upload_q(q0)
            a = drive(h, many)
            mid = (h.download_q(), h.download_w(), *h.download_evo_s())
            tend = a[0] + 2.5 * a[1]
            b = drive(h, few, a[0], tend)
            assert b[0] == tend and b[2] == 3, b
            c = drive(h, 3, b[0])
            out.append((a, b, c, *mid, h.download_q(), h.download_w(), *h.download_evo_s()))
    for x, y in zip(*out):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("what", ["upload", "unstable", "dt", "face"])
def test_line_stops_as_staged_steps_do(what):
    p = ics.sod_params(300, cfl=-0.4 if what == "dt" else 0.4)
    q0 = _state(p)
    bad = q0.copy()
    if what == "upload":
        bad[0, 0, 100, 4] = -1.0
    elif what == "unstable":  # a near vacuum left behind: the pressure turns negative in the run
        p.cfl = 4.0
    elif what == "face":  # a density that is no number gives no wave speeds
        bad[0, 0, 100, 0] = np.nan
    got = []
    for drive in (hydro.Hydro.run, _steps):
        with hydro.Hydro(p) as h:
            h.upload_q(bad)
            with pytest.raises(hydro.EvoraError) as e:
                drive(h, 500)
            got.append((e.value.code, e.value.message))
            if what in ("upload", "face"):
                h.upload_q(q0)
                got[-1] += drive(h, 5)
    assert got[0] == got[1], got


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_line_corrects_the_first_state_once(seed):
    """Dual energy, with an entropy that gives twice the pressure of E: the
    corrected E is back under the threshold, so that a second correction would
    take p from it.  Runs of one step (2 asked for, the end within the first)
    and of four."""
    n = 4000
    p = ics.sod_params(n, solver=2, limiter=1, boundtype=2, cfl=0.4, dualenergy=True, de_thresh=0.1)
    r = np.random.default_rng(seed).uniform(-0.1, 0.1, (2, 1, 1, n))
    rho, u = 1 + r[0], 2 + r[1]
    kin = 0.5 * rho * u * u  # kin / E = 1 / 1.1, just over the threshold of 0.9
    q = ics.prim_to_q(p.derive(), rho, u, 0 * u, 0 * u, 2.0 / 3.0 * 0.1 * kin)
    q[..., 5] *= 2
    out = []
    for drive in (hydro.Hydro.run, _steps):
        got = []
        for steps, tend in ((2, 1e-9), (4, 1e99)):
            with hydro.Hydro(p) as h:
                h.upload_q(q)
                a = drive(h, steps, 0.0, tend)
                got += [a, h.download_q(), h.download_w(), *h.download_evo_s()]
        out.append(got)
    assert out[0][0][2] == 1
    for x, y in zip(*out):
        assert np.array_equal(x, y)
