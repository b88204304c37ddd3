"""The order-free FP64 deposit at counts off its chunks and blocks, particles in any order,
buckets larger than a block and rows longer than its segments, against the oracle.  A weight is
rounded to 2^-49 of a particle's unit and the greatest node holds at least an eighth of one, so
the sums differ by less than 2^-46 = 1.5e-14 of the greatest a particle there, plus the reference
order's own rounding; 1e-12 is the form's stated bound."""
import numpy as np
import pytest

import oracle
from picard_amd import _lib, host
from tests.pic_driver import oracle_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 3, 4, 5, 1023, 1024, 1025, 30011])
@pytest.mark.parametrize("dims,species", [((3, 2, 4), 2), ((300, 4, 3), 3)])
def test_fixed_point_deposit(n, dims, species):
    half = tuple(5.0 * v for v in dims)
    ppc = (0, 2, 2, 0, 0, 0, 0, 0) if species == 3 else (0, 2, 0, 0, 0, 0, 0, 0)
    cfg = host.Config(nx=dims[0], ny=dims[1], nz=dims[2], flow=(True, False, True),
                      gmin=tuple(-h for h in half), gmax=half, ppc=ppc, species=species)
    rng = np.random.default_rng(n)
    rp = np.zeros((n, 8))
    rp[:, :3] = rng.uniform(-1.0, 1.0, (n, 3)) * half
    sp = rng.integers(1, species + 1, n).astype(np.int32)
    dom = host.Domain(cfg, max_particles=n + 8, order_free=True)
    if n:
        dom.append(rp, sp)
    N = []
    for _ in range(2):
        dom.particles_gridify()
        N.append(dom.field(_lib.FIELD_N))
    d = dom.d
    dom.close()
    N0, _, skipped = oracle.particles_gridify(oracle_grid(cfg), rp, sp, d.charge, d.n2p)
    assert skipped == 0
    assert np.array_equal(N[0], N[1])
    err = np.abs(N[0] - N0).max() / max(N0.max(), 1e-300)
    print(f"[gpu-dep-fixed] n={n} {dims}: {err:.1e}", flush=True)
    assert err <= 1e-12
