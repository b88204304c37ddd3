"""The FP64 form's solve with several sweeps per launch against the oracle,
bit for bit: the sweeps round as the reference's do, and the stop test is
applied to the iterates it can end on, so the potential and the sweep count are
the oracle's.  Shapes at the edges of the tiles (rows of 64 and 128 cells, 2, 4 and
6 rows, boxes thinner than a tile's halo, periodic images of images), every flow
combination, caps that end inside a launch, and a start whose halo is not the
image of its interior."""
import numpy as np
import pytest

import oracle
from picard_amd import _lib, host
from tests.pic_driver import oracle_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,flow,kw", [
    ((16, 16, 16), (True, False, False), {}),
    ((63, 5, 4), (True, True, True), {}),
    ((64, 3, 2), (False, False, True), dict(maxit=3000)),               # thinner than the halo, periodic
    ((64, 33, 9), (False, True, False), dict(maxit=500)),
    ((2, 34, 31), (True, False, True), {}),
    ((9, 70, 66), (True, False, False), dict(maxit=200)),   # more tiles than resident blocks
    ((65, 6, 7), (True, False, False), {}),
    ((66, 5, 6), (False, True, True), dict(maxit=2000)),
    ((128, 9, 4), (True, True, False), dict(maxit=2000)),
    ((127, 4, 5), (False, False, True), dict(maxit=2000)),
    ((129, 4, 6), (True, False, True), dict(maxit=2000)),               # wider: one sweep per launch
    ((66, 97, 92), (True, False, False), dict(maxit=60)),  # tiles of six rows
    ((11, 41, 47), (True, False, True), dict(maxit=300)),  # of 3 x 3
    ((33, 66, 65), (False, True, False), dict(maxit=60)),  # of 5 x 4
    ((10, 86, 62), (True, False, False), dict(maxit=120)),              # of 6 x 4
    ((20, 18, 16), (True, False, False), dict(maxerr=1e-30, maxit=201)),
    ((20, 18, 16), (False, True, True), dict(maxit=120)),
])
def test_solve_is_the_oracles(dims, flow, kw):
    cfg = host.Config(nx=dims[0], ny=dims[1], nz=dims[2], flow=flow, gmin=(-60.0, -70.0, -80.0),
                      gmax=(60.0, 70.0, 80.0), ppc=(0, 2, 0, 0, 0, 0, 0, 0), **kw)
    rng = np.random.default_rng(sum(dims))
    shape = tuple(v + 2 for v in dims[::-1])
    C = rng.normal(size=shape) * 1e-16
    U = rng.normal(size=shape)                            # halo not the interior's image
    dom = host.Domain(cfg, max_particles=64)
    dom.set_field(_lib.FIELD_C, C)
    dom.set_field(_lib.FIELD_U, U)
    n = dom.calc_epotential()
    got = dom.field(_lib.FIELD_U)
    dom.close()
    ref = U.copy()
    m, _ = oracle.calc_epotential(oracle_grid(cfg), ref, C, cfg.maxerr, cfg.maxit)
    print(f"[gpu-jacobi-block] {dims} {flow} {kw}: sweeps {n}, oracle {m}", flush=True)
    assert n == m
    assert np.array_equal(got, ref)
