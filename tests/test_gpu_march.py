"""The launch shapes and the CFL limit of the march: FP32's 32 x 6 column tile
at its edges and with chunks from one plane to all of them, against the
16 x 8 tile bit for bit; the limit of a new state with one cell faster than
the rest, against the limit of the same state uploaded (formed from its
primitive); the potential's download over more than one buffer."""
import numpy as np
import pytest

from evora_amd import hydro, ics
from evora_amd.params import HydroParams

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,bound", [(31, 6, 3, 1), (32, 5, 2, 3), (32, 6, 4, 2), (64, 18, 5, 3), (96, 6, 9, 2), (63, 11, 7, 1),
                                            (256, 30, 3, 2)])
@pytest.mark.parametrize("solver,limiter", [(2, 1), (1, 2), (2, 3)])
def test_wide_tile_equals_the_other(nx, ny, nz, bound, solver, limiter):
    p = HydroParams(nx=nx, ny=ny, nz=nz, solver=solver, limiter=limiter, boundtype=bound, cfl=0.3, atomic=True)
    q = ics.random_smooth(p, seed=3)
    out = []
    for ty, zc in ((8, 0), (8, 1), (12, 0), (12, 1), (12, 2), (12, nz)):
        with hydro.Hydro(p, precision=hydro.FP32_MIXED) as h:
            h.set_tuning(tile_ty=ty, zchunk=zc)
            h.upload_q(q)
            t = h.run(4)
            out.append((t, h.download_q()))
    for t, s in out[1:]:
        assert t == out[0][0]
        assert np.array_equal(s, out[0][1])


@pytest.mark.parametrize("mode,precision,tol", [
    (hydro.MODE_FUSED_EXACT, hydro.FP64, 0.0),     # the same arithmetic
    (hydro.MODE_FUSED, hydro.FP64, 1e-14),         # one reciprocal for three, a few ulp
    # FP32 pressure at kin/E <= 0.93: 14 ulp of 1.2e-7, half of it in a, and the sum and quotients
    (hydro.MODE_FUSED, hydro.FP32_MIXED, 4e-6),
])
@pytest.mark.parametrize("nz", [1, 9])
@pytest.mark.parametrize("dual", [False, True])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("mach", [0.1, 8.0, 40.0])
def test_limit_of_a_new_state(mode, precision, tol, nz, dual, axis, mach):
    """One cell moves at up to Mach 40 (with dual energy its pressure comes
    from the entropy there), the rest at a tenth of its speed."""
    if nz == 1 and axis == 2:
        axis = 1
    p = HydroParams(nx=70, ny=26, nz=nz, solver=2, limiter=1, boundtype=2, cfl=0.05, atomic=True, dualenergy=dual,
                    de_thresh=0.01 if dual else 0.0)
    d = p.derive()
    rng = np.random.default_rng(1)
    shape = (nz, 26, 70)
    rho = 1 + 0.2 * rng.uniform(-1, 1, shape)
    pr = 1 + 0.2 * rng.uniform(-1, 1, shape)
    v = 0.05 * rng.uniform(-1, 1, (3,) + shape)
    at = (nz // 2, 17, 45)
    if mach > 1:
        v[axis][at] = -mach
    else:
        pr[at] = 100.0  # the fastest by its sound speed
    q = np.empty(shape + (6,))
    q[..., 0] = rho
    for i in range(3):
        q[..., 1 + i] = rho * v[i]
    q[..., 4] = pr / d.g1 + 0.5 * rho * (v ** 2).sum(0)
    q[..., 5] = pr / rho ** d.g1
    with hydro.Hydro(p, precision=precision, mode=mode) as h:
        h.upload_q(q)
        h.run(2)
        h.primitive()
        got = h.hydrostep()
        h.upload_q(h.download_q())
        h.primitive()
        want = h.hydrostep()
    assert abs(got / want - 1) <= tol, (got, want)


def test_potential_over_several_buffers():
    """A state that repeats along z has a potential that does: 2.3e6 cells are
    18 MB, and the download's buffers hold 16."""
    p = ics.jeans_params(128, nz=140)
    q = ics.jeans(ics.jeans_params(128, nz=70), jeans_length=2.0)
    with hydro.Hydro(p) as h:
        h.upload_q(np.concatenate([q, q]))
        h.gravpotential(1.0)
        phi = h.download_phi()
    scale = np.abs(phi).max()
    assert scale > 0
    assert np.abs(phi[:70] - phi[70:]).max() <= 1e-11 * scale  # log2(n) stages of a 2.3e6-point transform at 1e-16 each, the mode range 1e3
