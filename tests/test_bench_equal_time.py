"""The bench's equal-time comparison: which pipeline its renders ask for."""
import sys
from pathlib import Path
from types import SimpleNamespace

import numpy as np

sys.path.insert(0, str(Path(__file__).resolve().parents[1]))
import bench  # noqa: E402


def test_equal_time_renders_take_the_default_pipeline(monkeypatch):
    """Plain and frozen-guide renders name no pool and no mode (an explicit pool
    takes the staged pipeline, the batched forms the default one: the comparison
    would be between pipelines); only the training has a pool of its own."""
    import time

    import narvalengine_amd
    calls = []
    clock = [0.0]
    monkeypatch.setattr(time, "perf_counter", lambda: clock[0])

    class Ctx:
        def synchronize(self):
            pass

        def render(self, g, cam, f, *, spp, **kw):
            calls.append(kw)
            clock[0] += 1e-4 * spp

    class Guide:
        def __init__(self, *a, **kw):
            pass

        def stats(self):
            return {"steps": 1}

        def close(self):
            pass

    monkeypatch.setattr(narvalengine_amd, "Guide", Guide)
    rng = np.random.default_rng(1)
    ref = np.full((4, 6, 3), 0.5)
    film = SimpleNamespace(clear=lambda: None, read=lambda: rng.uniform(10.0, 20.0, (4, 6, 3)))
    wl = SimpleNamespace(width=6, height=4, spp=64, max_bounces=8, camera=None)
    args = SimpleNamespace(batched=False, guide_probs=[0.5], guided_vertices=1, guide_cache=8, guide_cache_dirs=4,
                           train_spp=8, train_pool=1 << 17)
    bench.equal_time_budget(Ctx(), None, wl, args, ref, np.full_like(ref, 1e-6), film, 2)
    training = [kw for kw in calls if kw.get("train")]
    assert len(training) == 1 and training[0]["pool_size"] == args.train_pool
    others = [kw for kw in calls if not kw.get("train")]
    assert len(others) >= 3 and sum("guide" in kw for kw in others) >= 2
    for kw in others:
        assert not kw.get("pool_size") and not kw.get("mode"), kw
