"""Face potentials of the split form, mode by mode, against the sequential sums of the FP64
form on a random signed charge: edges of 2 and 3 cells, under, at and over the transforms'
tiles (16, 32, 64), every flow combination; and a distance table without the mirror symmetry, which
takes the FFT convolution, against its sum over cells.  Rounding: the transforms' error is bounded by some edge length
times 2^-53 of |C| |D| in the Euclidean norm; random signs leave a sum some 1 / sqrt(cells) of that of the
magnitudes, so 1e-12 of the greatest face value is above it by more than an order."""
import itertools

import numpy as np
import pytest

from picard_amd import _lib, host

pytestmark = pytest.mark.gpu

FLOWS = [f for f in itertools.product((False, True), repeat=3) if any(f)]


def _check(dims, flow):
    nx, ny, nz = dims
    cfg = host.Config(nx=nx, ny=ny, nz=nz, flow=flow, gmin=(-40.0, -50.0, -60.0), gmax=(40.0, 50.0, 60.0),
                      ppc=(0, 2, 0, 0, 0, 0, 0, 0))
    rng = np.random.default_rng(nx * 100 + ny + 7 * nz)
    C = rng.normal(size=(nz + 2, ny + 2, nx + 2)) * 1e-16
    U = []
    for prec in (_lib.PICARD_FP64, _lib.PICARD_FP32_SPLIT):
        dom = host.Domain(cfg, max_particles=16, precision=prec)
        dom.calc_distance()
        dom.set_field(_lib.FIELD_C, C)
        dom.bc_potentials()
        dom.bc_potentials()                                  # a second call has its tables
        U.append(dom.field(_lib.FIELD_U))
        dom.close()
    big = np.abs(U[0]).max()
    err = np.abs(U[1] - U[0]).max() / big
    print(f"[gpu-face-modes] {dims} {flow}: {err:.2e}", flush=True)
    assert big > 0
    assert err <= 1e-12


@pytest.mark.parametrize("flow", FLOWS)
@pytest.mark.parametrize("dims", [(2, 3, 2), (16, 8, 32), (17, 33, 9), (31, 15, 65)])
def test_faces(dims, flow):
    _check(dims, flow)


def test_x_faces_of_a_table_without_symmetry():
    """U(face node t') = sum over cells of C(n, t) D(n, t' - t): the split form's convolution."""
    nx, ny, nz = 12, 10, 9
    cfg = host.Config(nx=nx, ny=ny, nz=nz, flow=(True, False, False), gmin=(-40.0, -50.0, -60.0),
                      gmax=(40.0, 50.0, 60.0), ppc=(0, 2, 0, 0, 0, 0, 0, 0))
    rng = np.random.default_rng(3)
    C = rng.normal(size=(nz + 2, ny + 2, nx + 2)) * 1e-16
    dom = host.Domain(cfg, max_particles=16, precision=_lib.PICARD_FP32_SPLIT)
    dom.calc_distance()
    D = dom.field(_lib.FIELD_D)
    D = D * rng.uniform(0.5, 1.5, D.shape)
    dom.set_field(_lib.FIELD_D, D)
    dom.set_field(_lib.FIELD_C, C)
    dom.bc_potentials()
    U = dom.field(_lib.FIELD_U)
    dom.close()
    ref = np.zeros((2, nz, ny))
    for f in range(2):
        for n in range(1, nx + 1):
            o = nx + (n if f == 0 else n - nx - 1)
            for k in range(nz):
                for j in range(ny):
                    dk, dj = nz + k - np.arange(nz), ny + j - np.arange(ny)
                    ref[f, k, j] += (C[1:-1, 1:-1, n] * D[np.ix_(dk, dj, [o])][:, :, 0]).sum()
    ref /= 2.0 * 6.2831853071795864769252867665590 * 8.854187817e-12
    got = np.stack([U[1:-1, 1:-1, 0], U[1:-1, 1:-1, -1]])
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
