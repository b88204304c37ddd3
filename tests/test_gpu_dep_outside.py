"""Particles up to a cell below the grid's first node.  ParticlesGridify truncates towards zero, so they
count to the first cell with a remainder below zero: weights from -4 to 8, which the deposits
take as they are.  The order-free form rounds a weight to 2^-49 of a particle's unit, so a node that n
particles reach is off by less than n 2^-49 units, plus the reference order's own rounding of n 8 2^-53
a term; both are below n 2^-48, and the reference-order form is the oracle's bit for bit.  The order-free
form's sums are unsigned, so every node holds more particles inside than out here."""
import numpy as np
import pytest

import oracle
from picard_amd import _lib, host
from tests.pic_driver import oracle_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3000, 20_000, 300_000])
@pytest.mark.parametrize("axes", ["x", "yz", "xyz"])
def test_particles_below_the_first_node(n, axes):
    dims = (7, 5, 6)
    half = tuple(5.0 * v for v in dims)
    cfg = host.Config(nx=dims[0], ny=dims[1], nz=dims[2], flow=(True, False, True),
                      gmin=tuple(-h for h in half), gmax=half, ppc=(0, 2, 0, 0, 0, 0, 0, 0))
    rng = np.random.default_rng(n)
    rp = np.zeros((n, 8))
    rp[:, :3] = rng.uniform(-1.0, 1.0, (n, 3)) * half
    for q, a in enumerate("xyz"):
        if a in axes:
            out = rng.random(n) < 0.02
            rp[out, q] = -half[q] - 10.0 * rng.uniform(0.51, 1.49, int(out.sum()))
    sp = rng.integers(1, 3, n).astype(np.int32)
    N = {}
    for form in (False, True):
        dom = host.Domain(cfg, max_particles=n + 8, order_free=form)
        dom.append(rp, sp)
        dom.particles_gridify()
        N[form] = dom.field(_lib.FIELD_N)
        d = dom.d
        dom.close()
    N0, _, skipped = oracle.particles_gridify(oracle_grid(cfg), rp, sp, d.charge, d.n2p)
    assert skipped == 0 and N0.min() >= 0
    assert np.array_equal(N[False], N0)
    err = np.abs(N[True] - N0).max() / d.n2p[:2].max()
    print(f"[gpu-dep-outside] n={n} {axes}: {err:.1e} units", flush=True)
    assert err <= n * 2.0 ** -48
