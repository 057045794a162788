"""GPU seconds of reconstruct and advect: each call adds to its own sum, time
between the calls to neither, and the two stay within the host's clock; for every
last kernel a step can have (bounding by one workgroup, by separate launches,
none, snap and clip; split faces)."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,kw", [(8, {}), (40, {}), (8, {"nAlphaBounds": 0, "clip": False}),
                                  (8, {"nAlphaBounds": 0, "clip": True}), (8, {"splitWarpedFace": True}),
                                  (40, {"small": "0"}), (8, {"orientationMethod": "RDF"})])
def test_stage_times(monkeypatch, N, kw):
    import geometricvofext_amd as g
    print("timers", N, kw, flush=True)
    kw = dict(kw)
    if kw.pop("small", None):
        monkeypatch.setenv("SVP_BND_SMALL", "0")
    mesh = g.hex_box(N, perturb=0.2, seed=N)
    s = g.SolveVofEqu(mesh, dict(orientationMethod="LS") | kw)
    rng = np.random.default_rng(N)
    s.set_alpha(rng.uniform(0.0, 1.0, mesh.n_cells))
    s.set_flow(np.zeros(mesh.n_faces), np.zeros((mesh.n_cells, 3)))
    s.synchronize()
    assert s.timers()[:2] == (0.0, 0.0)
    s.reconstruct()          # (first use of the kernels is not timed by the host below)
    s.advect(1e-3)
    rec, adv, _ = s.timers()
    assert rec > 0.0 and adv > 0.0 and s.timers()[:2] == (rec, adv)
    for _ in range(3):
        t0 = time.perf_counter()
        s.reconstruct()
        s.synchronize()
        rec1, adv1, _ = s.timers()
        t1 = time.perf_counter()
        assert 0.0 < rec1 - rec < t1 - t0 and adv1 == adv
        time.sleep(0.05)
        t2 = time.perf_counter()
        s.advect(1e-3)
        s.synchronize()
        rec, adv, _ = s.timers()
        t3 = time.perf_counter()
        assert rec == rec1 and 0.0 < adv - adv1 < t3 - t2
    print("reconstruct", rec, "advect", adv, flush=True)
