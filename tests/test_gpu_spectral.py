"""The eigenbasis step of the solve (split and order-free FP64 forms) against
the FP64 form that sweeps all the way and is bit-exact to CalcEpotential.

Tolerance.  Both evaluate the same iterate in FP64.  A sweep rounds each cell
by about 2^-53 and the iteration forgets an error after about n^2 sweeps (n
the longest edge), so the swept potential is off by at most n^2 2^-53 relative
(65^2: 4.7e-13) and the transforms by far less: 1e-11 leaves a factor of twenty.  On
fully periodic boxes nothing damps the constant: q sweeps drift by up to q 2^-53.
The residual norm falls by about 5/n^2 a sweep, 1e-3 here, and its rounding is below
1e-9: the stop is the same sweep, or its neighbour where the norm meets the
threshold to that precision."""
import numpy as np
import pytest

from picard_amd import _lib, host

pytestmark = pytest.mark.gpu

FORMS = {"order_free": dict(order_free=True), "split": dict(precision=_lib.PICARD_FP32_SPLIT)}


def _solve(cfg, C, U=None, **kw):
    dom = host.Domain(cfg, max_particles=64, **kw)
    dom.calc_distance()
    dom.set_field(_lib.FIELD_C, C)
    dom.bc_potentials()
    if U is not None:
        dom.set_field(_lib.FIELD_U, U)
    n = dom.calc_epotential()
    out = dom.field(_lib.FIELD_U)
    dom.close()
    return n, out


def _case(dims, flow, **kw):
    cfg = host.Config(nx=dims[0], ny=dims[1], nz=dims[2], flow=flow, gmin=(-80.0,) * 3,
                      gmax=(80.0,) * 3, ppc=(0, 2, 0, 0, 0, 0, 0, 0), **kw)
    C = np.random.default_rng(sum(dims)).normal(size=tuple(v + 2 for v in dims[::-1])) * 1e-16
    if not any(flow):
        i = C[1:-1, 1:-1, 1:-1]
        i -= i.mean()
    return cfg, C


@pytest.mark.parametrize("form", ["order_free", "split"])
@pytest.mark.parametrize("dims,flow,kw", [
    ((16, 16, 16), (True, False, False), {}),
    ((15, 17, 33), (True, True, True), {}),
    ((65, 8, 31), (False, True, False), {}),              # past a tile of 64, odd periodic edge
    ((9, 64, 10), (True, False, True), {}),
    ((32, 12, 49), (False, False, True), {}),
    ((2, 3, 24), (True, True, True), {}),
    ((14, 22, 18), (True, True, False), dict(maxerr=1e-10)),
    ((12, 10, 14), (True, False, False), dict(maxerr=1e-30, maxit=700)),   # to the cap
    ((12, 10, 14), (False, False, False), dict(maxit=900)),
    ((24, 20, 16), (True, False, False), dict(maxit=150)),   # the rule ends before the solve does
    ((24, 20, 16), (True, False, False), dict(maxit=20)),
])
def test_solve_against_sweeps(dims, flow, kw, form):
    cfg, C = _case(dims, flow, **kw)
    q0, U0 = _solve(cfg, C)
    q1, U1 = _solve(cfg, C, **FORMS[form])
    print(f"[gpu-spectral] {form} {dims} {flow} {kw}: sweeps {q0}/{q1} "
          f"U {np.abs(U1 - U0).max() / np.abs(U0).max():.2e}", flush=True)
    if 2 * cfg.maxit + 1 <= 64 and form == "split":
        return                                             # FP32 sweeps throughout
    assert abs(q1 - q0) <= 1
    tol = 1e-11 if any(flow) else 1e-11 + 2.0 ** -53 * q0
    assert np.linalg.norm(U1 - U0) <= tol * np.linalg.norm(U0)


def test_start_from_any_potential():
    """A potential set by the caller, its halo not the image of its interior:
    the order-free form's first sweep reads it, as the reference's does."""
    cfg, C = _case((18, 14, 20), (True, False, False))
    U = np.random.default_rng(4).normal(size=C.shape)
    q0, U0 = _solve(cfg, C, U)
    q1, U1 = _solve(cfg, C, U, order_free=True)
    assert abs(q1 - q0) <= 1
    assert np.linalg.norm(U1 - U0) <= 1e-11 * np.linalg.norm(U0)


@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_non_finite_charge_is_swept(value):
    """A charge without a finite norm takes the sweeps: after few of them the
    cells it has not reached stay finite, the same ones as in the form that
    only sweeps."""
    cfg, C = _case((20, 20, 20), (True, True, True), maxit=4)
    C[3, 3, 3] = value
    q0, U0 = _solve(cfg, np.where(np.isfinite(C), C, 0.0))
    dom = host.Domain(cfg, max_particles=64, order_free=True)
    ref = host.Domain(cfg, max_particles=64)
    out = []
    for d in (ref, dom):
        d.set_field(_lib.FIELD_C, C)
        d.set_field(_lib.FIELD_U, U0)
        n = d.calc_epotential(maxit=40)
        out.append((n, np.isfinite(d.field(_lib.FIELD_U))))
        d.close()
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1])


def test_zero_charge_and_repeated_solves():
    cfg, C = _case((16, 12, 20), (True, False, False))
    dom = host.Domain(cfg, max_particles=64, order_free=True)
    dom.set_field(_lib.FIELD_C, np.zeros_like(C))
    assert dom.calc_epotential() == 0
    dom.calc_distance()
    got = []
    for scale in (1.0, 1e-3, 1.0):
        dom.set_field(_lib.FIELD_C, scale * C)
        dom.bc_potentials()
        got.append((dom.calc_epotential(), dom.field(_lib.FIELD_U)))
    dom.close()
    assert got[0][0] == got[2][0] and np.array_equal(got[0][1], got[2][1])


def _jacobi(U, b, dx, sweeps):
    """`sweeps` sweeps with fresh periodic images in y and z, and the residual
    norms of the last iterate and the one before it."""
    U = U.copy()

    def images():
        U[0], U[-1] = U[-2], U[1]
        U[:, 0], U[:, -1] = U[:, -2], U[:, 1]

    def residual():
        c = U[1:-1, 1:-1, 1:-1]
        lap = (U[1:-1, 1:-1, 2:] + U[1:-1, 1:-1, :-2] + U[1:-1, 2:, 1:-1] + U[1:-1, :-2, 1:-1] +
               U[2:, 1:-1, 1:-1] + U[:-2, 1:-1, 1:-1] - 6.0 * c) / dx ** 2
        return b - lap

    images()
    norms = [0.0, float(np.linalg.norm(residual()))]
    for _ in range(sweeps):
        U[1:-1, 1:-1, 1:-1] -= dx ** 2 / 6.0 * residual()
        images()
        norms = [norms[1], float(np.linalg.norm(residual()))]
    return U, norms


@pytest.mark.parametrize("dims,ppc,kw", [((8, 8, 8), 3, {}), ((17, 9, 33), 2, {}), ((33, 16, 10), 2, {}),
                                         ((16, 65, 8), 1, {}), ((65, 8, 12), 1, {}),
                                         ((15, 12, 14), 2, dict(maxit=40)),      # to the cap
                                         ((12, 10, 9), 2, dict(maxerr=1e-10))])
def test_ensemble_solve_is_the_jacobi_iterate(dims, ppc, kw):
    """Each simulation's potential is the iterate that sweeping in FP64 reaches
    (the tolerance of this file's other solves), and its sweep count the first at which
    the rule's norm passes, alone and beside another simulation."""
    from picard_amd import ensemble
    spec = ensemble.SimSpec(nx=dims[0], ny=dims[1], nz=dims[2], ppc=ppc, dx=10.0, density=5e6,
                            kelvin=1.2e5, drift=4e5, B=(1e-9, 0.0, 4e-9), seed=sum(dims), **kw)
    other = ensemble.SimSpec(nx=20, ny=11, nz=24, ppc=2, dx=8.0, density=8e6, kelvin=9e4, drift=5e5,
                             B=(0.0, 2e-9, 0.0), seed=5)
    got = []
    for mix in ([spec], [other, spec]):
        ens = ensemble.Ensemble.sized_for(mix, steps_room=4)
        slot = [ens.add(s) for s in mix][-1]
        ens.step()
        st = ens.status(slot)
        got.append((st.sweeps, st.noconv, ens.field(slot, _lib.FIELD_U), ens.field(slot, _lib.FIELD_C)))
        ens.close()
    assert got[0][0] == got[1][0] and np.array_equal(got[0][2], got[1][2])
    sweeps, noconv, U, C = got[0]
    d = ensemble.derive(spec)
    b = -C[1:-1, 1:-1, 1:-1] / (d.dV * 8.854187817e-12)
    U0 = np.zeros_like(U)
    U0[1:-1, 1:-1, 0], U0[1:-1, 1:-1, -1] = U[1:-1, 1:-1, 0], U[1:-1, 1:-1, -1]
    ref, (before, last) = _jacobi(U0, b, d.dxyz, sweeps)
    T = spec.maxerr * np.linalg.norm(b)
    i = (slice(1, -1),) * 3
    err = np.linalg.norm(U[i] - ref[i]) / np.linalg.norm(ref[i])
    print(f"[gpu-spectral] ensemble {dims}: {sweeps} sweeps, noconv {noconv}, {before / T:.9f} "
          f"{last / T:.9f}, U {err:.2e}", flush=True)
    assert err <= 1e-11
    if kw.get("maxit"):
        assert noconv == 1 and sweeps == 2 * kw["maxit"] + 1
    else:
        assert last <= T * (1 + 1e-8) and before > T * (1 - 1e-8)
