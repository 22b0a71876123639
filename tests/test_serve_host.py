"""Host logic of the batched / served workloads (no GPU): request streams
and scene generation."""
import numpy as np
import pytest

from eulersf_amd import serve
from eulersf_amd.serve import BatchedServer, Server, poisson_requests, random_scene, summarize


def test_poisson_stream_statistics():
    rng = np.random.default_rng(1)
    reqs = poisson_requests(rng, rate=20.0, seconds=200.0, n_range=(32, 160), k_range=(10, 100))
    t = np.array([r["t"] for r in reqs])
    assert np.all(np.diff(t) > 0) and t[-1] <= 200.0
    assert abs(len(reqs) / 200.0 - 20.0) < 2.0          # rate
    gaps = np.diff(t)
    assert abs(gaps.std() / gaps.mean() - 1.0) < 0.15   # exponential gaps
    ns = np.array([r["n"] for r in reqs])
    ks = np.array([r["k"] for r in reqs])
    assert ns.min() >= 32 and ns.max() <= 160 and ks.min() >= 10 and ks.max() <= 100


def test_random_scene_has_one_to_three_spheres():
    rng = np.random.default_rng(2)
    for _ in range(20):
        text = random_scene(rng, 48)
        k = text.count("solid sphere radius")
        assert 1 <= k <= 3
        assert "number of solids = %d" % k in text


def test_summary_of_records():
    recs = [{"id": 0, "n": 32, "k": 2, "arrival": 0.0, "start": 0.1, "end": 0.5,
             "lat": [0.1, 0.2], "error": None},
            {"id": 1, "n": 64, "k": 1, "arrival": 0.2, "start": 0.5, "end": 0.9,
             "lat": [0.3], "error": None}]
    s = summarize(recs, 1.0)
    assert s["steps"] == 3 and s["steps_per_s"] == 3.0
    assert s["cells_steps_per_s"] == 2 * 32 ** 3 + 64 ** 3
    assert s["completion_latency_ms"]["p50"] == 600.0


class GrowingScene:
    """a context that holds 1300 bytes per node once made and 1500 once it
    has stepped (the sweeps' scratch comes with a FLIP scene's first step)"""

    def __init__(self, n):
        self.nodes, self.stepped = (n + 1) ** 3, False

    @classmethod
    def from_cfg_text(cls, text, precision):
        return cls(int(text))

    def device_bytes(self):
        return (1500 if self.stepped else 1300) * self.nodes

    def stepImplicit(self, alpha):
        self.stepped = True
        return {"status": 0}

    def close(self):
        pass


@pytest.mark.parametrize("kind", [Server, BatchedServer])
def test_admission_sees_what_contexts_hold_once_they_step(monkeypatch, kind):
    monkeypatch.setattr(serve, "CoupledIntegrator3D", GrowingScene)
    monkeypatch.setattr(serve, "step_batch", lambda gs: [g.stepImplicit(-1.0) for g in gs])
    reqs = [{"id": i, "t": 0.0, "n": 40 + i, "k": 1 + 2 * i, "text": str(40 + i)} for i in range(3)]
    s = kind(1 << 40, 4)
    recs, makespan, info = s.run(reqs)
    assert sorted(r["id"] for r in recs) == [0, 1, 2] and all(r["error"] is None for r in recs)
    for r in recs:
        assert len(r["lat"]) == r["k"] and r["bytes"] == 1500 * (r["n"] + 1) ** 3
    assert s.bytes_per_node == pytest.approx(1500.0)
