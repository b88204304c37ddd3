"""The reference-order deposit at the edges of its blocks, bit for bit against the
oracle: rows of several segments, buckets of no particle, of more than a block's nodes can
share and of more than a block holds (one thread merges those), particles in every order,
three species, and no particle at all."""
import numpy as np
import pytest

import oracle
from picard_amd import _lib, host
from tests.pic_driver import oracle_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,n,heap,species", [
    ((5, 4, 3), 0, 0, 2),
    ((5, 4, 3), 1, 0, 2),
    ((2, 2, 2), 5000, 0, 2),             # columns of 400: a few nodes at a time
    ((62, 3, 4), 3000, 300, 2),          # one segment of 64 nodes
    ((63, 3, 4), 40000, 0, 2),           # two of 33 and 32
    ((150, 5, 2), 30000, 900, 3),
    ((9, 7, 8), 40, 1020, 2),            # about what a block holds
    ((9, 7, 8), 4000, 1025, 2),
    ((9, 7, 8), 4000, 6000, 2),
])
@pytest.mark.parametrize("flow", [(True, False, True)])
def test_gridify_is_the_oracles(dims, n, heap, species, flow):
    half = tuple(5.0 * v for v in dims)
    ppc = (0, 2, 2, 0, 0, 0, 0, 0) if species == 3 else (0, 2, 0, 0, 0, 0, 0, 0)
    cfg = host.Config(nx=dims[0], ny=dims[1], nz=dims[2], flow=flow, gmin=tuple(-h for h in half),
                      gmax=half, ppc=ppc, species=species)
    rng = np.random.default_rng(n + heap)
    rp = np.zeros((n + heap, 8))
    rp[:n, :3] = rng.uniform(-1.0, 1.0, (n, 3)) * half
    rp[n:, :3] = rng.uniform(0.5, 4.5, (heap, 3))        # of one cell and species
    rp[:, 3:6] = rng.normal(size=(n + heap, 3)) * 1e5
    sp = rng.integers(1, species + 1, n + heap).astype(np.int32)
    sp[n:] = 1
    order = rng.permutation(n + heap)
    rp, sp = np.ascontiguousarray(rp[order]), np.ascontiguousarray(sp[order])
    dom = host.Domain(cfg, max_particles=n + heap + 8)
    if n + heap:
        dom.append(rp, sp)
    dom.particles_gridify()
    N, C = dom.field(_lib.FIELD_N), dom.field(_lib.FIELD_C)
    dom.particles_gridify_all()
    Na = dom.field(_lib.FIELD_N)
    d = dom.d
    dom.close()
    N0, C0, skipped = oracle.particles_gridify(oracle_grid(cfg), rp, sp, d.charge, d.n2p)
    print(f"[gpu-dep-rows] {dims} n={n} heap={heap}: max {N0.max():.3g}", flush=True)
    assert skipped == 0
    assert np.array_equal(N, N0) and np.array_equal(C, C0)
    assert np.array_equal(Na, N0)
