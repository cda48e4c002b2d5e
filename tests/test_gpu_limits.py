"""The limits a sweep leaves for the next step, in states that no step should
start from: the fast FP64 form takes most cells' CFL limit from q without the
primitive, and has to find every cell the primitive finds."""
import numpy as np
import pytest

from evora_amd import hydro, ics
from evora_amd.batch import Batch
from evora_amd.params import HydroParams

pytestmark = pytest.mark.gpu

L = np.longdouble
HOT = (13, 4)  # x, y of the cell that empties


def _hot_cell(nz, cfl=0.4, **kw):
    """Gas at rest with one hot, dense cell, which a step far beyond the CFL
    limit drains below zero, symmetrically, so that its momentum stays 0."""
    p = HydroParams(nx=24, ny=10, nz=nz, solver=2, limiter=1, boundtype=1, cfl=cfl, atomic=True, secondorder=False, **kw)
    one = np.ones((nz, 10, 24))
    rho, pres = one.copy(), one.copy()
    rho[nz // 2, HOT[1], HOT[0]], pres[nz // 2, HOT[1], HOT[0]] = 10.0, 100.0
    return p, ics.prim_to_q(p.derive(), rho, 0 * one, 0 * one, 0 * one, pres)


def _only_invalid(q, nz, sign_rho):
    """Whether the hot cell alone has no pressure, with E < 0 and rho of the given sign."""
    bad = np.argwhere(q[..., 4] - 0.5 * (q[..., 1:4] ** 2).sum(-1) / q[..., 0] <= 0).tolist()
    c = q[nz // 2, HOT[1], HOT[0]]
    return bad == [[nz // 2, HOT[1], HOT[0]]] and c[4] < 0 and sign_rho * c[0] > 0


# factor: of the CFL limit's dt; with a dual-energy threshold of 1 every cell
# of moving gas takes p from the entropy, and E < 0 at rest is the only stop
CASES = [(8, {}, 12.0, -1), (1, {}, 12.0, -1), (8, {"dualenergy": True, "de_thresh": 1.0}, 0.79, 1),
         (1, {"dualenergy": True, "de_thresh": 1.0}, 0.975, 1)]


@pytest.mark.parametrize("nz,kw,factor,sign_rho", CASES)
@pytest.mark.parametrize("mode", [hydro.MODE_FUSED, hydro.MODE_FUSED_EXACT])
def test_cell_without_pressure_is_found(nz, kw, factor, sign_rho, mode):
    p, q0 = _hot_cell(nz, **kw)
    with hydro.Hydro(p, mode=mode) as h:
        h.upload_q(q0)
        h.primitive()
        dt = factor * h.hydrostep(1e99) / p.cfl
        h.compevo(dt)
        h.sweep(dt)
        as_meant = _only_invalid(h.download_q(), nz, sign_rho)
        assert as_meant
        h.primitive()
        with pytest.raises(hydro.EvoraError) as e:
            h.hydrostep(1e99)
    assert e.value.code == 1 and e.value.cell == (HOT[0] + 1, HOT[1] + 1, nz // 2 + 1)


def test_cell_without_pressure_is_found_in_a_batch():
    nz, kw, factor, _ = CASES[0]
    p, q0 = _hot_cell(nz, cfl=factor)
    with Batch([p, p]) as b:
        b.upload_q(0, np.ones(q0.shape) * q0[0, 0, 0])
        b.upload_q(1, q0)
        with pytest.raises(hydro.EvoraError) as e:
            b.run(2, graph=False)
        assert e.value.code == 1 and e.value.box == 1 and e.value.cell == (HOT[0] + 1, HOT[1] + 1, nz // 2 + 1)
        assert b.times()[2].tolist() == [2, 1]


@pytest.mark.parametrize("where", [63, 64, 126, 127, 255, 300])
@pytest.mark.parametrize("precision,mode", [(hydro.FP64, hydro.MODE_FUSED), (hydro.FP64, hydro.MODE_FUSED_EXACT),
                                            (hydro.FP64, hydro.MODE_STAGED), (hydro.FP32_MIXED, hydro.MODE_FUSED)])
def test_cell_that_is_no_number_hides_no_limit(precision, mode, where):
    """The limits come from the fastest cell, the first one here, wherever in
    its wave or its block's other waves a density is no number."""
    p = ics.conduction_params(16, nx=128, ny=4, nz=4)
    one = np.ones((4, 4, 128))
    pres = one.copy()
    pres[0, 0, 0] = 100.0
    q = ics.prim_to_q(p.derive(), one, 0 * one, 0 * one, 0 * one, pres)
    got = []
    for w in (None, where):
        if w is not None:
            q.reshape(-1, 6)[w, 0] = np.nan
        with hydro.Hydro(p, precision=precision, mode=mode) as h:
            h.upload_q(q)
            h.primitive()
            h.bound()
            got.append((h.hydrostep(1e99), h.thermalstep(1e99)))
    assert got[0] == got[1]


def test_limit_of_the_fast_form_is_as_near_as_six_roundings():
    """The fast FP64 form's limit of a swept state against the same in 80 bits,
    over gas at rest and in subsonic motion.  A rounding of a value whose digits
    are spread over its binade is 2^-52 / sqrt(12) sqrt(3 / (8 ln 2)) = 4.7e-17
    rms; the limit and its product with cfl have, where the sound speed leads,
    those of the sum, the root, the division by dx, the quotient and the product,
    and half of two under the root: sqrt(5 + 2 / 4) = 2.35 of them."""
    err = []
    for nz in (4, 1):
        for atomic in (True, False):
            p = HydroParams(nx=16, ny=12, nz=nz, solver=2, limiter=1, boundtype=2, cfl=0.2, atomic=atomic)
            d = p.derive()
            with hydro.Hydro(p) as h:
                for seed in range(200):
                    r = np.random.default_rng(seed)
                    rho, pres = (r.uniform(0.7, 1.3, (nz, 12, 16)) * np.exp(r.uniform(-1, 1)) for _ in range(2))
                    v = r.uniform(-1, 1, (3, nz, 12, 16)) * np.sqrt(pres / rho) * (0.01, 0.5)[seed % 2]
                    h.upload_q(ics.prim_to_q(d, rho, *v, pres))
                    h.primitive()
                    dt = 0.2 * h.hydrostep(1e99)
                    h.compevo(dt)
                    h.sweep(dt)
                    q = h.download_q().astype(L)
                    h.primitive()
                    dt = h.hydrostep(1e99)
                    p80 = L(d.g1) * (q[..., 4] - (q[..., 1:4] ** 2).sum(-1) / (2 * q[..., 0]))
                    a = np.sqrt(L(d.g) * p80 / q[..., 0])
                    lim = min((L(dx) / (abs(q[..., 1 + i] / q[..., 0]) + a)).min() for i, dx in enumerate((d.dx, d.dy, d.dz)))
                    err.append(float(dt / (L(d.cfl) * lim) - 1))
    one = 2.0 ** -52 / np.sqrt(12) * np.sqrt(3 / (8 * np.log(2)))
    rms = float(np.sqrt(np.mean(np.square(err))))
    assert rms <= np.sqrt(5 + 2 / 4) * one, rms


@pytest.mark.parametrize("nz", [1, 4])
@pytest.mark.parametrize("scale", [1e154, 1e-152])
def test_limit_does_not_depend_on_the_unit_of_density(scale, nz):
    """Density and pressure in another unit leave every speed as it is: also
    where 2 rho E leaves the range of the type (rho p g, which the solvers
    form, does not)."""
    p = HydroParams(nx=20, ny=12, nz=nz, solver=2, limiter=1, boundtype=2, cfl=0.3, atomic=True)
    d = p.derive()
    r = np.random.default_rng(2)
    rho, pres = r.uniform(0.95, 1.0, (2, nz, 12, 20))
    v = r.uniform(-0.05, 0.05, (3, nz, 12, 20))
    got = []
    for unit in (1.0, scale):
        with hydro.Hydro(p) as h:
            h.upload_q(ics.prim_to_q(d, unit * rho, *v, unit * 0.7 * pres))
            h.primitive()
            dt = 0.2 * h.hydrostep(1e99)
            h.compevo(dt)
            h.sweep(dt)
            h.primitive()
            got.append(h.hydrostep(1e99))
    assert got[1] == pytest.approx(got[0], rel=1e-13)
