"""Large field reads through pinned chunks and several threads: sizes under, at and over
the chunk and the direct copy's bound give what was written, the split form's field E what the device
widens (read into pinned memory, which the GPU fills itself), and overlapping
reads of one domain do not mix."""
import ctypes as ct
import threading

import numpy as np
import pytest
import torch

from picard_amd import _lib, host

pytestmark = pytest.mark.gpu


def _dom(n, precision):
    cfg = host.Config(nx=n, ny=n + 1, nz=n - 1, flow=(True, False, False), gmin=(-5.0 * n,) * 3,
                      gmax=(5.0 * n,) * 3, ppc=(0, 1, 0, 0, 0, 0, 0, 0))
    return host.Domain(cfg, max_particles=64, precision=precision)


@pytest.mark.parametrize("precision", [_lib.PICARD_FP64, _lib.PICARD_FP32_SPLIT])
@pytest.mark.parametrize("n", [4, 18, 48, 79, 101, 127])
def test_fields_come_back(n, precision):
    dom = _dom(n, precision)
    rng = np.random.default_rng(n)
    want = {w: rng.normal(size=dom.shape) for w in (_lib.FIELD_U, _lib.FIELD_C)}
    for w, a in want.items():
        dom.set_field(w, a)
    dom.calc_efield()
    got = {}

    def read(w):
        got[w] = dom.field(w)

    threads = [threading.Thread(target=read, args=(w,)) for w in (*want, _lib.FIELD_E)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for w, a in want.items():
        assert np.array_equal(got[w], a)
    pin = torch.empty(dom.shape + (3,), dtype=torch.float64, pin_memory=True)
    p = ct.cast(pin.data_ptr(), ct.POINTER(ct.c_double))
    _lib.check("picard_field_read", _lib.lib().picard_field_read(dom.h, _lib.FIELD_E, p, pin.numel()))
    print(f"[gpu-readback] {n} {precision}: {got[_lib.FIELD_E].nbytes} bytes of E", flush=True)
    assert np.array_equal(got[_lib.FIELD_E], pin.numpy())
    assert np.abs(got[_lib.FIELD_E]).max() > 0
    dom.close()
