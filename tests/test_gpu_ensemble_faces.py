"""The ensemble's face potentials, formed mode by mode, against the plain sum over cells of
BCpotentials.f90:51-77 with CalcDistance's periodic images: odd and even axes, edges
under and over the transforms' tiles, a long axis (which has no basis and keeps the plain sum), and
several simulations at once.  The transforms' rounding is bounded in the Euclidean
norm by some edge length times 2^-53 of |C| |D|; 1e-12 of the greatest sum of |C| D is
above that for these boxes by two orders."""
import numpy as np
import pytest

from picard_amd import _lib, ensemble

pytestmark = pytest.mark.gpu


def _faces(spec, C):
    """Both faces [face][k][j] and the greatest sum of |C| D, without the factor."""
    ny, nz, nx, h = spec.ny, spec.nz, spec.nx, spec.dx
    j, k = np.arange(ny), np.arange(nz)
    out = np.zeros((2, nz, ny))
    big = np.zeros((2, nz, ny))
    Ci = C[1:-1, 1:-1, 1:-1]
    for ip in range(nx):
        for face, a in ((0, ip + 1), (1, nx - ip)):
            dy = [(j * h) ** 2, ((ny - j) * h) ** 2]
            dz = [(k * h) ** 2, ((nz - k) * h) ** 2]
            D = sum(1.0 / np.sqrt((a * h) ** 2 + dy[p][None, :] + dz[q][:, None])
                    for p in (0, 1) for q in (0, 1))
            for kk in range(nz):
                Dk = D[np.abs(k - kk)]                       # [kp][|dj|]
                for jj in range(ny):
                    w = Dk[:, np.abs(j - jj)]
                    out[face, kk, jj] += (Ci[:, :, ip] * w).sum()
                    big[face, kk, jj] += (np.abs(Ci[:, :, ip]) * w).sum()
    return out, big.max()


@pytest.mark.parametrize("boxes", [
    [(8, 8, 8)],
    [(17, 15, 9), (9, 16, 33), (33, 8, 11)],
    [(20, 13, 31), (1030, 8, 9)],
])
def test_face_sums(boxes):
    rho, T = 5e6, 116045.0
    specs = [ensemble.SimSpec(nx=b[0], ny=b[1], nz=b[2], ppc=3, dx=ensemble.debye_length(rho, T),
                              density=rho, kelvin=T, drift=4e5, B=(0.0, 0.0, 5e-9), seed=11 + q)
             for q, b in enumerate(boxes)]
    ens = ensemble.Ensemble.sized_for(specs, steps_room=4)
    slots = [ens.add(s) for s in specs]
    ens.step()
    for s, spec in zip(slots, specs):
        U, C = ens.field(s, _lib.FIELD_U), ens.field(s, _lib.FIELD_C)
        ref, big = _faces(spec, C)
        kappa = 1.0 / (2.0 * 6.2831853071795864769252867665590 * 8.854187817e-12)
        got = np.stack([U[1:-1, 1:-1, 0], U[1:-1, 1:-1, -1]])
        err = np.abs(got - kappa * ref).max() / (kappa * big)
        print(f"[gpu-ensemble-faces] {(spec.nx, spec.ny, spec.nz)}: {err:.2e}", flush=True)
        assert err <= 1e-12
    ens.close()
