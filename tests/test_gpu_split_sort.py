"""The split form's step, whose sort pushes, deletes and wraps on the way, against the
same phases called one by one (AdvancePosition as its own pass): every particle and the
densities bit for bit.  Boxes with fewer keys than the counted window and with many
windows, a time step that carries particles over rows and planes (keys far from their
block's), appended particles (not pushed), and particle counts off the block's size."""
import numpy as np
import pytest

from picard_amd import _lib, host

pytestmark = pytest.mark.gpu


def _rows(dom):
    rp, sp = dom.particles()
    a = np.column_stack([rp, sp])
    return a[np.lexsort(a.T)]


@pytest.mark.parametrize("dims,flow,ppc,speed", [
    ((2, 2, 3), (True, False, False), 1, 1.0),
    ((5, 4, 3), (False, True, False), 3, 20.0),
    ((16, 16, 16), (True, True, True), 5, 8.0),
    ((33, 18, 9), (True, False, True), 8, 40.0),
    ((40, 3, 37), (False, False, False), 4, 5.0),
])
def test_step_is_its_phases(dims, flow, ppc, speed):
    half = tuple(5.0 * v for v in dims)
    cfg = host.Config(nx=dims[0], ny=dims[1], nz=dims[2], flow=flow, gmin=tuple(-h for h in half),
                      gmax=half, ppc=(0, ppc, 0, 0, 0, 0, 0, 0), maxit=40)
    d = host.derive(cfg)
    d.dt *= speed
    cap = 8 * int(d.ppc[:2].sum() + 1) * int(np.prod([v + 2 for v in dims])) + 64
    rng = np.random.default_rng(sum(dims))
    extra = rng.uniform(-1.0, 1.0, (11, 8)) * 0.4
    extra[:, :3] *= half
    sp = np.ones(11, np.int32)
    out = []
    for fused in (True, False):
        dom = host.Domain(cfg, max_particles=cap, d=d, precision=_lib.PICARD_FP32_SPLIT)
        dom.calc_distance()
        dom.generate_initial(3)
        dom.generate_inflow(3, 1)
        if fused:
            st = dom.step((extra, sp))
            removed = st.removed
        else:
            dom.advance_position()
            dom.append(extra, sp)
            _, removed = dom.bc_outflow()
            dom.particles_transfer()
            dom.particles_gridify()
            dom.bc_potentials()
            dom.calc_epotential()
            dom.calc_efield()
            dom.bc_fields()
            dom.advance_velocity()
        out.append((removed, _rows(dom), dom.field(_lib.FIELD_N)))
        dom.close()
    print(f"[gpu-split-sort] {dims} {flow}: {len(out[0][1])} kept, {out[0][0]} removed", flush=True)
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][2], out[1][2])


def test_step_that_fails_has_pushed():
    """A step whose produced particles do not fit ends after its push, as the phases would."""
    cfg = host.Config(nx=6, ny=5, nz=4, flow=(True, False, False), gmin=(-30.0, -25.0, -20.0),
                      gmax=(30.0, 25.0, 20.0), ppc=(0, 3, 0, 0, 0, 0, 0, 0))
    d = host.derive(cfg)
    out = []
    for fused in (True, False):
        dom = host.Domain(cfg, max_particles=6 * 5 * 4 * 6 + 5, d=d, precision=_lib.PICARD_FP32_SPLIT)
        dom.calc_distance()
        dom.generate_initial(9)
        if fused:
            with pytest.raises(_lib.PicardError):
                dom.step((np.zeros((50, 8)), np.ones(50, np.int32)))
        else:
            dom.advance_position()
        out.append(_rows(dom))
        dom.close()
    assert np.array_equal(out[0], out[1])
