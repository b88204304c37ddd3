"""The split form's deposit at counts off its chunks, rounds and blocks against the FP64
form's on the same particles.  Per particle the split weights differ by at most: the
offset's rounding, 2^-25 on each axis on both its corners (6 x 2^-25 over the eight corners),
that of 1 - f (another 6 x 2^-25), two products (4 x 2^-25), 16 x 2^-25 < 5e-7 of the
particle's unit in the sum over the corners; the flux adds the velocity's rounding, 2^-24.
Velocities are positive, so that sums of magnitudes bound the sums of errors."""
import numpy as np
import pytest

from picard_amd import _lib, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,dims", [(n, d) for n in (1, 7, 8, 9, 2047, 2049, 4095, 4097, 20011)
                                    for d in ((4, 3, 5), (37, 9, 6))]
                         + [((1 << 20) + 3, (37, 9, 6)), ((1 << 22) + 4099, (37, 9, 6))])
def test_deposit_counts(n, dims):
    half = tuple(5.0 * v for v in dims)
    cfg = host.Config(nx=dims[0], ny=dims[1], nz=dims[2], flow=(True, False, True),
                      gmin=tuple(-h for h in half), gmax=half, ppc=(0, 8, 0, 0, 0, 0, 0, 0))
    rng = np.random.default_rng(n + dims[0])
    rp = np.zeros((n, 8))
    rp[:, :3] = rng.uniform(-1.0, 1.0, (n, 3)) * half
    rp[:, 3:6] = rng.uniform(1e3, 4e5, (n, 3))
    sp = rng.integers(1, 3, n).astype(np.int32)
    out = []
    for prec in (_lib.PICARD_FP64, _lib.PICARD_FP32_SPLIT):
        dom = host.Domain(cfg, max_particles=n + 8, precision=prec)
        dom.append(rp, sp)
        dom.bc_outflow()
        dom.particles_transfer()
        assert dom.num_local == n
        dom.particles_gridify()
        N = dom.field(_lib.FIELD_N)
        dom.particles_gridify_all()
        assert np.array_equal(dom.field(_lib.FIELD_N), N)
        out.append((N, dom.field(_lib.FIELD_F)))
        dom.close()
    for a, b, tol in zip(out[0], out[1], (5e-7, 5e-7 + 2.0 ** -24)):
        err, size = np.abs(a - b).sum(), np.abs(a).sum()
        print(f"[gpu-split-deposit] n={n} {dims}: {err / size:.2e}", flush=True)
        assert err <= tol * size
