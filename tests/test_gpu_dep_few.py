"""The order-free FP64 deposit on both sides of the line between one atomic per corner and particle and
bucketing first: integer sums, so the densities of a set of particles that the one form deposits are the
sums of its parts' that the other does, unit for unit, and both are the oracle's within
n 2^-49 of a particle's unit plus the reference order's own rounding, below n 2^-48."""
import numpy as np
import pytest

import oracle
from picard_amd import _lib, host
from tests.pic_driver import oracle_grid

pytestmark = pytest.mark.gpu


def _line(dims, species):
    buckets = species * np.prod([v + 1 for v in dims])
    return int(min(14 * buckets, 75000 + buckets // 4))


@pytest.mark.parametrize("dims", [(3, 2, 4), (9, 8, 7), (21, 20, 23)])
def test_both_sides_of_the_line(dims):
    half = tuple(5.0 * v for v in dims)
    cfg = host.Config(nx=dims[0], ny=dims[1], nz=dims[2], flow=(True, False, True),
                      gmin=tuple(-h for h in half), gmax=half, ppc=(0, 2, 0, 0, 0, 0, 0, 0))
    line = _line(dims, 2)
    n = line + 300
    rng = np.random.default_rng(n)
    rp = np.zeros((n, 8))
    rp[:, :3] = rng.uniform(-1.0, 1.0, (n, 3)) * half
    sp = rng.integers(1, 3, n).astype(np.int32)

    def deposit(a, b):
        dom = host.Domain(cfg, max_particles=b - a + 8, order_free=True)
        dom.append(rp[a:b], sp[a:b])
        dom.particles_gridify()
        N, d = dom.field(_lib.FIELD_N), dom.d
        dom.close()
        return np.rint(N / d.n2p[:2] * 2.0 ** 48), N, d

    whole, N, d = deposit(0, n)                       # bucketed
    parts = deposit(0, n // 2)[0] + deposit(n // 2, n)[0]       # each one atomic per corner
    below, Nb, _ = deposit(0, line - 1)
    above, Na, _ = deposit(0, line + 1)
    # N and its quotient are rounded by 2^-53 each: whole units come back below 2^51, as where few meet
    exact = np.abs(whole) < 2.0 ** 51
    assert np.array_equal(whole[exact], parts[exact])
    assert np.abs(whole - parts).max() <= np.abs(whole).max() * 2.0 ** -50
    for N1, m in ((N, n), (Nb, line - 1), (Na, line + 1)):
        N0, _, skipped = oracle.particles_gridify(oracle_grid(cfg), rp[:m], sp[:m], d.charge, d.n2p)
        assert skipped == 0
        assert np.abs(N1 - N0).max() <= m * 2.0 ** -48 * d.n2p[:2].max()


def test_particles_outside_are_counted():
    """Refused as before in the direct form too: particles beyond the arrays, the others deposited."""
    cfg = host.Config(nx=6, ny=5, nz=4, flow=(True, False, False), gmin=(-30.0, -25.0, -20.0),
                      gmax=(30.0, 25.0, 20.0), ppc=(0, 2, 0, 0, 0, 0, 0, 0))
    rp = np.zeros((5, 8))
    rp[1, 0], rp[3, 2] = 60.0, -55.0
    dom = host.Domain(cfg, max_particles=16, order_free=True)
    dom.append(rp, np.ones(5, np.int32))
    with pytest.raises(_lib.PicardError, match="2 particle"):
        dom.particles_gridify()
    assert abs(dom.field(_lib.FIELD_N).sum() / dom.d.n2p[0] - 3.0) < 1e-12
    dom.close()
