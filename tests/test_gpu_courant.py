"""Courant maxima against the oracle: cells of up to six faces and of more, fewer
cells than a workgroup has lanes, and more than the grid takes in one pass; one
handle and a batch of all of them, whose cases fill different numbers of blocks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [("hex", 1), ("tet", 4), ("refined", 8), ("hex", 7), ("hex", 65)]


def case(oracle_lib, kind, N):
    import geometricvofext_amd as g
    mesh = {"hex": g.hex_box, "tet": g.tet_box, "refined": g.refined_hex_box}[kind](N)
    om = oracle_lib.OracleMesh(mesh)
    rng = np.random.default_rng(mesh.n_cells)
    return mesh, om, rng.uniform(0.0, 1.0, mesh.n_cells), rng.normal(size=om.Sf.shape[0])


@pytest.mark.parametrize("kind,N", SIZES)
def test_courant_every_form(oracle_lib, kind, N):
    import geometricvofext_amd as g
    print("courant", kind, N, flush=True)
    mesh, om, alpha, phi = case(oracle_lib, kind, N)
    s = g.SolveVofEqu(mesh, dict(orientationMethod="LS"))
    s.set_alpha(alpha)
    for _ in range(2):
        s.set_flow(phi, np.zeros((mesh.n_cells, 3)))
        assert tuple(s.courant()) == tuple(om.courant(phi, alpha))
        phi = 0.5 * phi


def test_courant_batch(oracle_lib):
    import geometricvofext_amd as g
    cases = [case(oracle_lib, *k) for k in SIZES if k[0] == "hex"]
    handles = [g.SolveVofEqu(mesh, dict(orientationMethod="LS")) for mesh, _, _, _ in cases]
    for s, (mesh, om, alpha, phi) in zip(handles, cases):
        s.set_alpha(alpha)
        s.set_flow(phi, np.zeros((mesh.n_cells, 3)))
    co, aco = g.CaseBatch(handles).courant()
    for k, (mesh, om, alpha, phi) in enumerate(cases):
        assert (co[k], aco[k]) == tuple(om.courant(phi, alpha))
