"""evh_run, whose steps take dt, t and the end of the run on the device, against
the same steps taken one by one through evh_step (each with its own read of
the limits): the same states, times and limits bit for bit, the same number
of steps, the same stops; over more steps than one batch of launches, in runs
that end early, after errors, and continued afterwards."""
import time

import numpy as np
import pytest

from evora_amd import hydro, ics
from evora_amd.params import HydroParams

pytestmark = pytest.mark.gpu


def _case(name):
    if name == "kh2d":
        p = HydroParams(nx=70, ny=45, nz=1, solver=2, limiter=2, boundtype=2, cfl=0.4, atomic=False, tend=1e30)
        return p, ics.kh_reference(p)
    if name == "conduction":
        p = ics.conduction_params(12)
        return p, ics.conduction_blob(p)
    if name == "conduction2d":
        p = ics.conduction_params(18, nz=1)
        return p, ics.conduction_blob(p)
    if name == "no_hydro":
        p = ics.conduction_params(12, hydro=False)
        return p, ics.conduction_blob(p)
    if name == "jeans":  # power-of-two sides: every kernel of the step is the library's
        p = ics.jeans_params(16)
        return p, ics.jeans(p, jeans_length=2.0)
    if name == "jeans_hipfft":
        p = ics.jeans_params(12)
        return p, ics.jeans(p, jeans_length=2.0)
    if name == "jeans_conduction":
        p = ics.jeans_params(16, conduction=True, simplekappa=True)
        return p, ics.jeans(p, jeans_length=2.0)
    p = ics.blast_params(20, solver=2, cfl=0.3)
    p.ny, p.nz = 13, 9
    return p, ics.blast_reference(p, p0=1e-2, r0=0.15)


def _run(h, n, t, tend):
    return h.run(n, t=t, tend=tend)


def _steps(h, n, t, tend):
    go, dt, done = True, 0.0, 0
    while go and done < n:
        t, dt, go = h.step(t, tend)
        done += 1
    h.synchronize()
    return t, dt, done


@pytest.mark.parametrize("precision,mode", [(hydro.FP64, hydro.MODE_FUSED), (hydro.FP64, hydro.MODE_FUSED_EXACT),
                                            (hydro.FP32_MIXED, hydro.MODE_FUSED)])
@pytest.mark.parametrize("name", ["blast", "kh2d", "conduction", "conduction2d", "no_hydro", "jeans", "jeans_hipfft",
                                  "jeans_conduction"])
def test_run_equals_steps(name, precision, mode):
    p, q0 = _case(name)
    out = []
    for drive in (_run, _steps):
        with hydro.Hydro(p, precision=precision, mode=mode) as h:
            h.upload_q(q0)
            a = drive(h, 3, 0.0, 1e30)
            b = drive(h, 70, a[0], 1e30)          # over one batch of launches
            tend = b[0] + 5.5 * b[1]
            c = drive(h, 200, b[0], tend)          # ends early, inside a batch
            assert c[0] == tend and c[2] < 200, c
            d = drive(h, 4, c[0], 1e30)            # and goes on from there
            out.append((a, b, c, d, h.download_q(), h.sums(), h.download_phi() if p.gravity else 0))
    for x, y in zip(*out):
        assert np.array_equal(x, y), name


@pytest.mark.parametrize("what", ["upload", "unstable", "dt"])
def test_run_stops_as_steps_do(what):
    """The stops of the driver loop: a negative pressure of the uploaded
    state, one in the run, a step that is not positive; the same code and
    message, and a context that runs on after an upload."""
    p = ics.blast_params(16, solver=2, cfl=0.4)
    bad = ics.blast_reference(p, p0=1e-2, r0=0.15)
    q0 = bad[:1, :1, :1] * np.linspace(1.0, 1.1, 16)[:, None, None, None] + np.zeros_like(bad)  # gas at rest, stable at any cfl
    if what == "upload":
        bad[5, 6, 7, 4] = -1.0
    elif what == "unstable":   # a time step beyond the scheme's stability: stops after some steps
        p.cfl = 0.95
        bad = ics.blast(p)
    else:
        p.cfl = -0.4
    got = []
    for drive in (_run, _steps):
        with hydro.Hydro(p) as h:
            h.upload_q(bad)
            with pytest.raises(hydro.EvoraError) as e:
                drive(h, 150, 0.0, 1e30)
            err = (e.value.code, e.value.message)
            if what == "dt":
                got.append((err,))
                continue
            h.upload_q(q0)
            t = drive(h, 5, 0.0, 1e30)
            got.append((err, t, h.download_q()))
    for x, y in zip(*got):
        assert np.array_equal(np.asarray(x, dtype=object), np.asarray(y, dtype=object)) if isinstance(x, tuple) \
            else np.array_equal(x, y), (x, y)


@pytest.mark.parametrize("precision,mode", [(hydro.FP64, hydro.MODE_FUSED), (hydro.FP64, hydro.MODE_FUSED_EXACT),
                                            (hydro.FP32_MIXED, hydro.MODE_FUSED)])
def test_run_without_hydro_takes_each_steps_own_potential(precision, mode):
    """Gravity and conduction without hydro: the potential's passes lead the
    step.  The first run of a context, one that ends with steps to spare, and
    one from another state after it: each step has the potential of its own
    state, and a step after the end forms none."""
    p = ics.conduction_params(16, hydro=False, gravity=True)
    q0 = 10 * ics.conduction_blob(p)
    q1 = ics.conduction_blob(p, seed=3)
    out = []
    for drive in (_run, _steps):
        with hydro.Hydro(p, precision=precision, mode=mode) as h:
            h.upload_q(q0)
            a = drive(h, 2, 0.0, 1e30)
            first = (h.download_q(), h.download_phi())
            b = drive(h, 100, a[0], a[0] + 2.5 * a[1])
            end = (h.download_q(), h.download_phi())
            h.upload_q(q1)
            c = drive(h, 2, 0.0, 1e30)
            out.append((a, b, c, *first, *end, h.download_q(), h.download_phi()))
    for x, y in zip(*out):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("name,steps", [("jeans", 1), ("jeans", 3), ("kh2d", 3)])
def test_run_to_an_output_time_launches_few_steps_beyond_it(name, steps):
    """A run asked for very many steps that ends after a few takes no longer
    than the steps one by one, but for its own start (half as long again).
    64 steps launched at once took 2.5 to 12 times as long."""
    if name == "jeans":
        p = ics.jeans_params(64)
        q0 = ics.jeans(p, jeans_length=2.0)
    else:
        p = HydroParams(nx=128, ny=128, nz=1, solver=2, limiter=2, boundtype=2, cfl=0.4, atomic=False, tend=1e30)
        q0 = ics.kh_reference(p)
    best = []
    for drive in (_run, _steps):
        with hydro.Hydro(p) as h:
            h.upload_q(q0)
            t, dt, _ = drive(h, 5, 0.0, 1e30)
            took = []
            for _ in range(20):
                h.synchronize()
                t0 = time.perf_counter()
                t, _, done = drive(h, 10**6, t, t + (steps - 0.5) * dt)
                h.synchronize()
                took.append(time.perf_counter() - t0)
                assert done == steps
            best.append(min(took))
    assert best[0] < 1.5 * best[1], best
