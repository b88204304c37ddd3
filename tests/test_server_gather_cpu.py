"""When an idle lane of the server starts its jobs (no device work: a stand-in ensemble whose step takes
2 ms, and a gathering time of 0.2 s, far above what a loaded machine adds): at once unless another job is
due within that time and fits beside it."""
import time
from types import SimpleNamespace

import pytest

from picard_amd import ensemble, server


class _Ensemble:
    def __init__(self, **kw):
        self.tuned, self.left, self.slots = 0, {}, 0

    def add(self, spec):
        self.slots += 1
        self.left[self.slots] = 0
        return self.slots

    def step(self):
        time.sleep(0.002)
        for s in self.left:
            self.left[s] += 1
        return SimpleNamespace(pushed=1)

    def status(self, slot):
        return SimpleNamespace(steps=self.left[slot], pushed=1)

    def remove(self, slot):
        del self.left[slot]

    def tune(self, sweeps):
        self.tuned += 1

    def close(self):
        pass


def _jobs(*arrivals, steps=2):
    spec = ensemble.SimSpec(nx=16, ny=16, nz=16, ppc=4, dx=10.0, density=5e6, kelvin=1e5, drift=4e5,
                            B=(0.0, 0.0, 5e-9), seed=1)
    return [server.Job(jid=i, arrival=a, spec=spec, steps=steps) for i, a in enumerate(arrivals)]


def _run(monkeypatch, jobs, time_limit=None, **kw):
    monkeypatch.setattr(ensemble, "Ensemble", _Ensemble)
    monkeypatch.setattr(server, "GATHER_S", 0.2)
    srv = server.Server(**kw)
    rep = srv.run(jobs, time_limit=time_limit)
    srv.close()
    return rep


def test_lone_jobs_start_at_once(monkeypatch):
    rep = _run(monkeypatch, _jobs(0.02, 0.42))
    assert rep["jobs_done"] == 2 and rep["peak_jobs"] == 1
    assert rep["p99_wait_s"] < 0.1


def test_jobs_due_together_start_together(monkeypatch):
    rep = _run(monkeypatch, _jobs(0.02, 0.16, 0.80))
    assert rep["peak_jobs"] == 2
    first, second, third = sorted(rep["done"], key=lambda j: j.arrival)
    assert first.admitted - first.arrival > 0.13
    assert second.admitted - second.arrival < 0.1 and third.admitted - third.arrival < 0.1


def test_a_full_lane_does_not_wait(monkeypatch):
    rep = _run(monkeypatch, _jobs(0.02, 0.20), max_sims=1)
    first = min(rep["done"], key=lambda j: j.arrival)
    assert rep["peak_jobs"] == 1 and first.admitted - first.arrival < 0.1


def test_the_time_limit_ends_the_wait(monkeypatch):
    rep = _run(monkeypatch, _jobs(0.02, 0.21), time_limit=0.05)
    assert rep["jobs_done"] == 0 and rep["wall_s"] < 0.15


@pytest.mark.parametrize("arrivals,now,want", [
    ((), 1.0, 1.0), ((2.0,), 1.0, 1.0), ((1.0,), 1.0, 1.0), ((1.0, 1.005), 1.001, 1.005),
    ((1.0, 1.001, 1.009), 1.002, 1.009), ((1.0, 1.02), 1.001, 1.001)])
def test_gather_until(arrivals, now, want):
    assert server.gather_until(_jobs(*arrivals), now, lambda jobs: True) == want
    assert server.gather_until(_jobs(*arrivals), now, lambda jobs: False) == now


@pytest.mark.parametrize("edge,tuned", [(16, 0), (1024, 0), (1025, 1)])
def test_only_jobs_that_are_swept_are_tuned_for(monkeypatch, edge, tuned):
    monkeypatch.setattr(ensemble, "Ensemble", _Ensemble)
    jobs = _jobs(0.0, 0.05)
    jobs[1].spec.nx, jobs[1].spec.ny, jobs[1].spec.nz = edge, 8, 8
    srv = server.Server(tune_sweeps=32)
    srv.run(jobs)
    assert srv.lanes[0].ens.tuned == tuned
    srv.close()
