"""Meshes with empty patches under every bounding schedule (one workgroup, separate
launches with the dataflow pass or with rounds), as a handle and as cases of a
batch, against the oracle: every kernel that reads a face's empty flag meets set
and unset ones."""
import numpy as np
import pytest

from tests.helpers import bits_equal, empty_z_box

pytestmark = pytest.mark.gpu


def schedule_env(monkeypatch, schedule):
    if schedule != "one":
        monkeypatch.setenv("SVP_BND_SMALL", "0")
    if schedule == "rounds":
        monkeypatch.setenv("SVP_BND_FLOW", "0")


def fields(om, N):
    rng = np.random.default_rng(N)
    n = om.C.shape[0]
    alpha = np.clip(rng.normal(0.5, 0.6, n), 0.0, 1.0)
    V = np.array([0.5, -0.4, 0.7])      # its flux through the empty patches is not zero
    return alpha, np.tile(V, (n, 1)), om.Sf @ V, 0.6 * float(np.min(om.V)) ** (1.0 / 3.0)


@pytest.mark.parametrize("schedule", ["one", "flow", "rounds"])
@pytest.mark.parametrize("N", [5, 14])
def test_bound_with_empty_patches(oracle_lib, monkeypatch, schedule, N):
    import geometricvofext_amd as g
    print("empty patches", schedule, N, flush=True)
    schedule_env(monkeypatch, schedule)
    mesh = empty_z_box(N, 0.15, N)
    om = oracle_lib.OracleMesh(mesh)
    alpha, U, phi, dt = fields(om, N)
    gpu = g.SolveVofEqu(mesh, dict(orientationMethod="LS", nAlphaBounds=3, clip=False))
    ors = oracle_lib.OracleSolver(om, nAlphaBounds=3, clip=False, threads=8)
    for s in (gpu, ors):
        s.set_alpha(alpha)
        s.set_flow(phi, U)
    for step in range(3):
        for s in (gpu, ors):
            s.reconstruct()
            s.advect(dt)
        assert bits_equal(gpu.alpha(), ors.alpha()), step
        assert bits_equal(gpu.alpha_phi(), ors.alpha_phi()), step
    assert gpu.bound_totals()[3] > 0
    gpu.synchronize()


@pytest.mark.parametrize("schedule", ["one", "flow"])
def test_batch_with_empty_patches(oracle_lib, monkeypatch, schedule):
    import geometricvofext_amd as g
    print("batch of empty patches", schedule, flush=True)
    schedule_env(monkeypatch, schedule)
    cases = []
    for mesh in (empty_z_box(7, 0.15, 7), g.hex_box(6, perturb=0.2, seed=6), empty_z_box(12, 0.15, 12)):
        om = oracle_lib.OracleMesh(mesh)
        gpu = g.SolveVofEqu(mesh, dict(orientationMethod="LS", nAlphaBounds=3, clip=False))
        ors = oracle_lib.OracleSolver(om, nAlphaBounds=3, clip=False, threads=8)
        alpha, U, phi, dt = fields(om, mesh.n_cells)
        for s in (gpu, ors):
            s.set_alpha(alpha)
            s.set_flow(phi, U)
        cases.append((gpu, ors, dt))
    b = g.CaseBatch([c[0] for c in cases])
    for step in range(3):
        b.step([c[2] for c in cases])
        for k, (gpu, ors, dt) in enumerate(cases):
            ors.reconstruct()
            ors.advect(dt)
            assert bits_equal(gpu.alpha(), ors.alpha()), (step, k)
            assert bits_equal(gpu.alpha_phi(), ors.alpha_phi()), (step, k)
