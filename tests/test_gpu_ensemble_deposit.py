"""The ensemble's sort and deposit at particle counts off the chunks and blocks, several
simulations in one arena: after a step every particle is in its box, sits once (ids are distinct) and
the densities are those of the particles, formed here from the same FP32 weights in units of 2^-40
(whole numbers, so equal up to the last products' rounding, 1e-14)."""
import numpy as np
import pytest

from picard_amd import _lib, ensemble

pytestmark = pytest.mark.gpu


def _density(spec, rp, sp):
    n = np.array([spec.nx, spec.ny, spec.nz])
    xi = rp[:, :3] / spec.dx + 0.5 * n + 0.5                   # box centred on 0: xi = c + f
    f = (xi - np.floor(xi)).astype(np.float32)
    c = np.floor(xi).astype(np.int64)
    c[f >= 1.0] += 1
    f[f >= 1.0] = 0.0
    W = np.zeros((spec.nz + 2, spec.ny + 2, spec.nx + 2, 2), np.int64)
    one = np.float32(1.0)
    for o in range(8):
        b = [o & 1, (o >> 1) & 1, o >> 2]
        w = [f[:, d] if b[d] else one - f[:, d] for d in range(3)]
        units = ((w[0] * w[1] * w[2]).astype(np.float64) * 2.0 ** 40).astype(np.int64)
        np.add.at(W, (c[:, 2] + b[2], c[:, 1] + b[1], c[:, 0] + b[0], sp - 1), units)
    # guard folds: z and y periodic, x into the edge plane and cleared
    for ax in (0, 1):
        W = np.moveaxis(W, ax, 0)
        lo, hi = W[0] + W[-2], W[1] + W[-1]
        W[0], W[-2], W[1], W[-1] = lo, lo, hi, hi
        W = np.moveaxis(W, 0, ax)
    W[:, :, 1] += W[:, :, 0]
    W[:, :, -2] += W[:, :, -1]
    W[:, :, 0] = W[:, :, -1] = 0
    return W


@pytest.mark.parametrize("boxes", [
    [(8, 8, 8, 1)],
    [(9, 8, 11, 3), (8, 8, 8, 2), (24, 17, 10, 5), (13, 30, 9, 16)],
    [(40, 12, 9, 1), (8, 8, 8, 40)],
])
def test_densities_are_the_particles(boxes):
    rho, T = 5e6, 116045.0
    specs = [ensemble.SimSpec(nx=b[0], ny=b[1], nz=b[2], ppc=b[3], dx=ensemble.debye_length(rho, T),
                              density=rho, kelvin=T, drift=4e5, B=(0.0, 0.0, 5e-9), seed=5 + q)
             for q, b in enumerate(boxes)]
    ens = ensemble.Ensemble.sized_for(specs, steps_room=6)
    slots = [ens.add(s) for s in specs]
    for _ in range(3):
        ens.step()
    for s, spec in zip(slots, specs):
        rp, sp = ens.particles(s)
        assert np.unique(rp[:, 7]).size == len(rp)
        W = _density(spec, rp, sp)
        N = ens.field(s, _lib.FIELD_N)
        scale = N[W > 0].max() / W.max()
        err = np.abs(N - W * scale).max() / N.max()
        print(f"[gpu-ensemble-deposit] {boxes} {len(rp)} particles: {err:.1e}", flush=True)
        assert err <= 1e-14
    ens.close()
