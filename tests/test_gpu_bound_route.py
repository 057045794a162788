"""The routes of a step's bounding passes, chosen by the candidates of an earlier
step: handles and batches whose candidates grow past the line and fall below it
again, against the oracle; batches with few and many candidates side by side and
with flat and warped meshes in one."""
import numpy as np
import pytest

from tests.helpers import bits_equal

pytestmark = pytest.mark.gpu

OPTS = dict(nAlphaBounds=3, clip=False)


def case(oracle_lib, kind, N, noise, seed):
    """mesh, oracle mesh, alpha (a ball and noise in a share of the cells), U, phi, cell size"""
    import geometricvofext_amd as g
    mesh = g.hex_box(N, perturb=0.2 if kind == "hexp" else 0.0, seed=N)
    om = oracle_lib.OracleMesh(mesh)
    rng = np.random.default_rng(seed)
    r = np.linalg.norm(om.C - 0.5, axis=1) * N
    alpha = np.clip(3.5 - r, 0.0, 1.0) + (rng.random(mesh.n_cells) < noise) * rng.normal(0.0, 0.5, mesh.n_cells)
    V = np.array([0.5, -0.4, 0.7])
    return (mesh, om, np.clip(alpha, 0.0, 1.0), np.tile(V, (mesh.n_cells, 1)), om.Sf @ V,
            float(np.min(om.V)) ** (1.0 / 3.0))


# 30^3 (one workgroup or separate launches at once) and 38^3 (one workgroup that
# looks itself where the flow has grown); a flow of 1e-16 moves no cell out of
# bounds
@pytest.mark.parametrize("N", [30, 38])
def test_candidates_grow_and_fall(oracle_lib, N):
    import geometricvofext_amd as g
    print("bound route", N, flush=True)
    mesh, om, alpha, U, phi, h = case(oracle_lib, "hexp", N, 0.3, N)
    gpu = g.SolveVofEqu(mesh, dict(orientationMethod="LS", **OPTS))
    ors = oracle_lib.OracleSolver(om, threads=8, **OPTS)
    seen = []
    gpu.upload_base_flow(U, phi)
    for s in (gpu, ors):
        s.set_alpha(alpha)
    for k, (factor, dt) in enumerate([(1e-16, 0.9), (1e-16, 0.9), (1.0, 0.9), (1.0, 0.9), (1e-16, 0.9), (1e-16, 0.9),
                                      (1e-16, 0.9), (-1.0, 0.9), (1e-16, 0.9), (0.9, 1e-16), (0.9, 0.9)]):
        gpu.scale_flow(factor)
        ors.set_flow(factor * phi, factor * U)
        for s in (gpu, ors):
            s.reconstruct()
            s.advect(dt * h)
        assert bits_equal(gpu.alpha(), ors.alpha()), k
        assert bits_equal(gpu.alpha_phi(), ors.alpha_phi()), k
        seen.append(int(gpu.bound_stats()[:1, 0].sum()))
    print("candidates", seen, flush=True)
    assert min(seen) <= 512 < max(seen)
    gpu.synchronize()


@pytest.mark.parametrize("kinds", [("hexp", "hex", "hex"), ("hexp", "hexp", "hex")])
@pytest.mark.parametrize("graph", ["1", "0"])
def test_batch_few_and_many(oracle_lib, monkeypatch, kinds, graph):
    import geometricvofext_amd as g
    print("batch route", kinds, graph, flush=True)
    monkeypatch.setenv("SVP_BATCH_GRAPH", graph)
    cases = [case(oracle_lib, kind, N, noise, N) for kind, N, noise in zip(kinds, (30, 13, 9), (0.3, 0.05, 0.0))]
    gpu = [g.SolveVofEqu(c[0], dict(orientationMethod="LS", **OPTS)) for c in cases]
    ors = [oracle_lib.OracleSolver(c[1], threads=8, **OPTS) for c in cases]
    for (_, _, alpha, U, phi, _), s, o in zip(cases, gpu, ors):
        for x in (s, o):
            x.set_alpha(alpha)
            x.set_flow(phi, U)
    b = g.CaseBatch(gpu)
    seen = []
    # the first case alone grows and falls; an idle case between
    for k, f in enumerate([(1e-16, 0.5, 0.5), (0.9, 0.5, 0.5), (0.9, 0.5, 0.0), (1e-16, 0.5, 0.5), (1e-16, 0.9, 0.5),
                           (0.9, 0.5, 0.5), (0.0, 0.5, 0.5), (0.0, 0.5, 0.5)]):
        dts = [x * c[5] for x, c in zip(f, cases)]
        b.step(dts)
        for j, (o, dt) in enumerate(zip(ors, dts)):
            if dt > 0.0:
                o.reconstruct()
                o.advect(dt)
            assert bits_equal(gpu[j].alpha(), o.alpha()), (k, j)
            if dt > 0.0:
                assert bits_equal(gpu[j].alpha_phi(), o.alpha_phi()), (k, j)
        seen.append(int(gpu[0].bound_stats()[:1, 0].sum()))
    print("candidates", seen, flush=True)
    assert min(seen) <= 512 < max(seen)
    b.close()
    # each handle alone goes on from there
    for (_, _, _, _, _, h), s, o in zip(cases, gpu, ors):
        for x in (s, o):
            x.reconstruct()
            x.advect(0.5 * h)
        assert bits_equal(s.alpha(), o.alpha())
        s.synchronize()


def test_batch_tune_keeps_the_route(oracle_lib):
    """Launch shapes tuned on a batch whose passes one workgroup takes: the steps after are the oracle's."""
    import geometricvofext_amd as g
    print("batch tune", flush=True)
    cases = [case(oracle_lib, "hexp", N, 0.05, N) for N in (9, 12)]
    gpu = [g.SolveVofEqu(c[0], dict(orientationMethod="LS", **OPTS)) for c in cases]
    ors = [oracle_lib.OracleSolver(c[1], threads=8, **OPTS) for c in cases]
    for (_, _, alpha, U, phi, _), s, o in zip(cases, gpu, ors):
        for x in (s, o):
            x.set_alpha(alpha)
            x.set_flow(phi, U)
    b = g.CaseBatch(gpu)
    dts = [0.5 * c[5] for c in cases]
    b.tune(dts)
    for _ in range(3):
        b.step(dts)
        for s, o, dt in zip(gpu, ors, dts):
            o.reconstruct()
            o.advect(dt)
            assert bits_equal(s.alpha(), o.alpha())


def test_flow_written_in_place(oracle_lib):
    """phi written through the device view, with no call that tells of it: few candidates, many, few, many."""
    import ctypes as C
    import geometricvofext_amd as g
    print("flow in place", flush=True)
    mesh, om, alpha, U, phi, h = case(oracle_lib, "hexp", 38, 0.3, 38)
    gpu = g.SolveVofEqu(mesh, dict(orientationMethod="LS", **OPTS))
    ors = oracle_lib.OracleSolver(om, threads=8, **OPTS)
    for s in (gpu, ors):
        s.set_alpha(alpha)
        s.set_flow(1e-16 * phi, U)
    hip = C.CDLL("libamdhip64.so.7")    # the runtime the library runs on
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    at = gpu.device_view().phi
    seen = []
    for k, f in enumerate([1e-16, 1e-16, 1.0, 1.0, 1e-16, 1e-16, 0.5]):
        gpu.synchronize()
        now = np.ascontiguousarray(f * phi)
        assert hip.hipMemcpy(at, now.ctypes.data, now.nbytes, 1) == 0
        ors.set_flow(f * phi, U)
        for s in (gpu, ors):
            s.reconstruct()
            s.advect(0.9 * h)
        assert bits_equal(gpu.alpha(), ors.alpha()), k
        seen.append(int(gpu.bound_stats()[:1, 0].sum()))
    print("candidates", seen, flush=True)
    assert min(seen) <= 512 < max(seen)
    gpu.synchronize()
