"""BCpotentials in the reference's order against the oracle, bit for bit, at the
edges of the face kernel's chunks: rows of 64, 128 and 192 cells and one more,
groups of 16 terms and their remainders, more than 64 face nodes along a row of lanes,
fewer rows than are staged at a time, every open dimension."""
import numpy as np
import pytest

import oracle
from picard_amd import _lib, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,flow", [
    ((2, 2, 2), (True, True, True)),
    ((15, 5, 4), (True, True, True)),
    ((16, 66, 3), (True, False, True)),
    ((17, 3, 65), (True, True, False)),
    ((63, 4, 9), (True, True, True)),
    ((64, 9, 5), (True, True, True)),
    ((65, 7, 6), (False, True, True)),
    ((128, 6, 5), (True, True, False)),
    ((129, 5, 4), (True, False, True)),
    ((192, 4, 3), (True, True, True)),
    ((193, 3, 4), (True, True, True)),
    ((33, 130, 2), (True, False, False)),
])
def test_face_sums_are_the_oracles(dims, flow):
    nx, ny, nz = dims
    cfg = host.Config(nx=nx, ny=ny, nz=nz, flow=flow, gmin=(-40.0, -50.0, -60.0),
                      gmax=(40.0, 50.0, 60.0), ppc=(0, 2, 0, 0, 0, 0, 0, 0))
    C = np.random.default_rng(nx * 100 + ny).normal(size=(nz + 2, ny + 2, nx + 2)) * 1e-16
    dom = host.Domain(cfg, max_particles=64)
    dom.calc_distance()
    D = dom.field(_lib.FIELD_D)
    out = []
    for q in (1.0, -3.0):                                 # a second call on other charge
        dom.set_field(_lib.FIELD_C, q * C)
        dom.bc_potentials()
        out.append(dom.field(_lib.FIELD_U))
    dom.close()
    g = oracle.Grid(nx, ny, nz, cfg.species, flow=flow, gmin=cfg.gmin, gmax=cfg.gmax)
    for q, U in zip((1.0, -3.0), out):
        print(f"[gpu-bcpot] {dims} {flow}", flush=True)
        assert np.array_equal(U, oracle.bc_potentials(g, q * C, D))
