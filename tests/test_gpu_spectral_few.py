"""Solves of few sweeps, before and after ones of many in the same domain, and caps on both sides of the
shortest solve that leaves the split form's FP32 sweeps (maxit 33): every form's sweep count is the
oracle's, the reference-order form's potential its bits, the others' within FP64 rounding (1e-11, see
test_gpu_spectral.py) or, after FP32 sweeps, within the split form's stated 1e-5."""
import numpy as np
import pytest

import oracle
from picard_amd import _lib, host
from tests.pic_driver import oracle_grid

pytestmark = pytest.mark.gpu

FORMS = {"fp64": {}, "order_free": dict(order_free=True), "split": dict(precision=_lib.PICARD_FP32_SPLIT)}


def _setup(dims, flow):
    cfg = host.Config(nx=dims[0], ny=dims[1], nz=dims[2], flow=flow, gmin=(-60.0, -70.0, -80.0),
                      gmax=(60.0, 70.0, 80.0), ppc=(0, 2, 0, 0, 0, 0, 0, 0))
    rng = np.random.default_rng(sum(dims))
    shape = tuple(v + 2 for v in dims[::-1])
    C, U = rng.normal(size=shape) * 1e-16, rng.normal(size=shape)
    return cfg, C, U


def _images(U, flow):
    """The halo that the split form starts from: the interior's images across periodic boundaries."""
    U = U.copy()
    for axis, open_ in ((0, flow[2]), (1, flow[1]), (2, flow[0])):
        if not open_:
            a = np.moveaxis(U, axis, 0)
            a[0], a[-1] = a[-2].copy(), a[1].copy()
    return U


def _compare(form, cfg, dom, C, U, maxerr, maxit, fp32=False):
    dom.set_field(_lib.FIELD_C, C)
    dom.set_field(_lib.FIELD_U, U)
    n = dom.calc_epotential(maxerr=maxerr, maxit=maxit)
    got = dom.field(_lib.FIELD_U)
    ref = _images(U, cfg.flow) if form == "split" else U.copy()
    m, _ = oracle.calc_epotential(oracle_grid(cfg), ref, C, maxerr, maxit)
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    print(f"[gpu-spectral-few] {form} {maxerr} {maxit}: sweeps {n}, oracle {m}, U {err:.1e}", flush=True)
    assert n == m
    if form == "fp64":
        assert np.array_equal(got, ref)
    else:
        assert err <= (1e-5 if fp32 else 1e-11)


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("dims,flow", [((16, 12, 18), (True, False, False)), ((15, 17, 14), (True, True, True)),
                                       ((12, 14, 16), (False, False, True))])
def test_few_and_many_sweeps_in_turn(dims, flow, form):
    cfg, C, U = _setup(dims, flow)
    U *= 1e-3                                  # the charge's part of the residual, not the start's
    dom = host.Domain(cfg, max_particles=64, **FORMS[form])
    for maxerr in (0.5, 0.5, 0.2, 1e-4, 0.5, 0.05, 1e-4, 0.3, 0.3):
        _compare(form, cfg, dom, C, U, maxerr, 20000)
    dom.close()


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("maxit", [20, 31, 32, 33, 34])
def test_caps_about_the_shortest_step(maxit, form):
    cfg, C, U = _setup((24, 20, 16), (True, False, False))
    dom = host.Domain(cfg, max_particles=64, **FORMS[form])
    for _ in range(2):
        _compare(form, cfg, dom, C, _images(U, cfg.flow), 1e-8, maxit, fp32=maxit <= 32)
    dom.close()


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("flow", [(True, False, False), (False, False, False), (False, True, True)])
def test_no_sweep_at_all(flow, form):
    """Without charge the first test passes: the potential stays, and the split form's halo is its images."""
    cfg, C, U = _setup((7, 5, 6), flow)
    dom = host.Domain(cfg, max_particles=64, **FORMS[form])
    for _ in range(2):
        dom.set_field(_lib.FIELD_C, np.zeros_like(C))
        dom.set_field(_lib.FIELD_U, U)
        assert dom.calc_epotential(maxerr=1e-6, maxit=1000) == 0
        assert np.array_equal(dom.field(_lib.FIELD_U), _images(U, flow) if form == "split" else U)
    dom.close()
