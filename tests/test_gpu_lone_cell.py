"""A cell without faces (first or last label, mixed alpha): the other cells'
interface, polygons, fluxes and alpha are those of the mesh without it; it has no
plane, and its Courant number is 0 / 0."""
import numpy as np
import pytest

from tests.helpers import bits_equal

pytestmark = pytest.mark.gpu


def with_lone_cell(mesh, first):
    from geometricvofext_amd.mesh import PolyMesh
    d = 1 if first else 0
    return PolyMesh(points=mesh.points, face_offsets=mesh.face_offsets, face_points=mesh.face_points,
                    owner=mesh.owner + np.int32(d), neighbour=mesh.neighbour + np.int32(d), n_cells=mesh.n_cells + 1,
                    patch_names=mesh.patch_names, patch_start=mesh.patch_start, patch_size=mesh.patch_size,
                    patch_type=mesh.patch_type, name=f"{mesh.name} and a cell without faces")


@pytest.mark.parametrize("kind,N", [("hex", 6), ("tet", 4), ("refined", 8)])
@pytest.mark.parametrize("first", [True, False])
def test_cell_without_faces(oracle_lib, kind, N, first):
    import geometricvofext_amd as g
    print("lone cell", kind, N, first, flush=True)
    mesh = {"hex": g.hex_box, "tet": g.tet_box, "refined": g.refined_hex_box}[kind](N)
    om = oracle_lib.OracleMesh(mesh)
    rng = np.random.default_rng(N)
    alpha = rng.uniform(0.1, 0.9, mesh.n_cells)
    V = np.array([0.3, -0.2, 0.1])
    U, phi = np.tile(V, (mesh.n_cells, 1)), om.Sf @ V
    at, d = (0, 1) if first else (mesh.n_cells, 0)
    opts = dict(orientationMethod="LS", nAlphaBounds=3, clip=False)
    a, b = g.SolveVofEqu(mesh, opts), g.SolveVofEqu(with_lone_cell(mesh, first), opts)
    a.set_alpha(alpha)
    a.set_flow(phi, U)
    b.set_alpha(np.insert(alpha, at, 0.5))
    b.set_flow(phi, np.insert(U, at, 0.0, axis=0))
    assert np.isnan(b.courant()[0])
    for s in (a, b):
        s.reconstruct()
    ia, ib = a.interface(), b.interface()
    keep = ib["cells"] != at
    assert keep.sum() == len(ia["cells"]) and len(keep) == keep.sum() + 1
    assert np.array_equal(ib["cells"][keep] - d, ia["cells"]) and ib["status"][~keep][0] != 0
    for k in ("d", "C", "S", "n"):
        assert bits_equal(ib[k][keep], ia[k]), k
    pa, pb = a.plic_surface(), b.plic_surface()
    assert np.array_equal(pb["cells"] - d, pa["cells"])
    assert np.array_equal(pb["offsets"], pa["offsets"]) and bits_equal(pb["points"], pa["points"])
    for s in (a, b):
        s.advect(0.02 / N)
    assert bits_equal(np.delete(b.alpha(), at), a.alpha())
    assert bits_equal(b.alpha_phi(), a.alpha_phi())
    b.synchronize()
