"""The reference-order deposit of few particles for the grid, by nodes, and of more, by rows: the
oracle's densities and charge bit for bit on both sides of the line, and with particles below the first node."""
import numpy as np
import pytest

import oracle
from picard_amd import _lib, host
from tests.pic_driver import oracle_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,species", [((3, 2, 4), 2), ((66, 5, 4), 2), ((13, 12, 14), 3)])
@pytest.mark.parametrize("flow", [(True, False, False), (False, True, True)])
def test_nodes_and_rows(dims, species, flow):
    half = tuple(5.0 * v for v in dims)
    ppc = (0, 2, 2, 0, 0, 0, 0, 0) if species == 3 else (0, 2, 0, 0, 0, 0, 0, 0)
    cfg = host.Config(nx=dims[0], ny=dims[1], nz=dims[2], flow=flow, gmin=tuple(-h for h in half),
                      gmax=half, ppc=ppc, species=species)
    line = -(-species * int(np.prod([v + 2 for v in dims])) // 3)       # from here on by rows
    rng = np.random.default_rng(line)
    rp = np.zeros((line + 7, 8))
    rp[:, :3] = rng.uniform(-1.0, 1.0, (line + 7, 3)) * half
    rp[::9, 0] = -half[0] - 10.0 * rng.uniform(0.51, 1.49, rp[::9].shape[0])
    rp[: line // 2, 1] = 0.3                                            # many to some nodes
    sp = rng.integers(1, species + 1, line + 7).astype(np.int32)
    for n in (1, line // 3, line - 1, line, line + 7):
        dom = host.Domain(cfg, max_particles=n + 8)
        dom.append(rp[:n], sp[:n])
        dom.particles_gridify()
        N, C, d = dom.field(_lib.FIELD_N), dom.field(_lib.FIELD_C), dom.d
        dom.close()
        N0, C0, skipped = oracle.particles_gridify(oracle_grid(cfg), rp[:n], sp[:n], d.charge, d.n2p)
        assert skipped == 0
        assert np.array_equal(N, N0) and np.array_equal(C, C0)
