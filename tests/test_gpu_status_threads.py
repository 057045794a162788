"""State words read by two threads on one handle: while one asks for the number of
mixed cells, the other's polygon export keeps its sizes."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_counts_while_exporting():
    import geometricvofext_amd as g
    print("status threads", flush=True)
    mesh = g.hex_box(16, perturb=0.1, seed=3)
    s = g.SolveVofEqu(mesh, dict(orientationMethod="LS"))
    s.init_alpha([((0.5, 0.5, 0.5), 0.3)])
    s.reconstruct()
    n, first = s.n_mixed(), s.plic_surface()
    assert n > 0 and len(first["cells"]) > 0
    stop, seen = threading.Event(), []

    def count():
        while not stop.is_set() and len(seen) < 20000:
            seen.append(s.n_mixed())

    t = threading.Thread(target=count)
    t.start()
    try:
        for _ in range(300):
            p = s.plic_surface()
            assert np.array_equal(p["cells"], first["cells"]) and np.array_equal(p["offsets"], first["offsets"])
    finally:
        stop.set()
        t.join()
    assert seen and set(seen) == {n}
