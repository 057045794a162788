"""Interface face volumes of every launch form, against the oracle: lanes per
face by mesh (triangles, flat quadrilaterals, warped ones, larger polygons),
below and above the pair counts at which a lane takes a whole polygon, and a
plane at rest (no sweep)."""
import numpy as np
import pytest

from tests.helpers import bits_equal

pytestmark = pytest.mark.gpu


def case_mesh(kind, N):
    import geometricvofext_amd as g
    if kind == "tet":
        return g.tet_box(N, perturb=0.1, seed=N)
    if kind == "refined":
        return g.refined_hex_box(N)
    if kind == "bricks":
        return g.brick_box(N, seed=N, perturb=0.1)
    return g.hex_box(N, perturb=0.2 if kind == "hexp" else 0.0, seed=N)


# pairs per cell are about 3 (hexahedra) and 4 (tetrahedra, upwind ones
# included); one lane per cut up to 36864 pairs of flat quadrilaterals, 12288 of
# warped ones, 49152 of triangles and 16384 of larger polygons
@pytest.mark.parametrize("kind,N,speed", [("hex", 3, 1.0), ("hex", 9, 1.0), ("hex", 28, 1.0), ("hexp", 5, 1.0),
                                          ("hexp", 20, 1.0), ("hexp", 20, 0.0), ("tet", 3, 1.0), ("tet", 14, 1.0),
                                          ("tet", 6, 0.0), ("refined", 8, 1.0), ("refined", 16, 1.0),
                                          ("bricks", 5, 1.0), ("bricks", 12, 1.0), ("hex", 7, 0.0)])
def test_flux_every_form(oracle_lib, kind, N, speed):
    import geometricvofext_amd as g
    print("flux", kind, N, speed, flush=True)
    mesh = case_mesh(kind, N)
    om = oracle_lib.OracleMesh(mesh)
    rng = np.random.default_rng(100 + N)
    alpha = rng.uniform(0.02, 0.98, mesh.n_cells)
    if kind == "bricks":
        # warped faces of up to 8 points: one direction oblique to all of them
        # (a plane along one crosses it more often than the library takes)
        x = om.C @ np.array([0.3, 0.5, 0.8])
        alpha = 0.02 + 0.96 * (x - x.min()) / (x.max() - x.min())
    V = np.array([0.6, -0.45, 0.3])
    U = speed * (V + 0.2 * rng.normal(size=(mesh.n_cells, 3)))
    phi = om.Sf @ V
    dt = 0.35 * float(np.min(om.V)) ** (1.0 / 3.0)
    gpu = g.SolveVofEqu(mesh, dict(orientationMethod="LS", nAlphaBounds=0, clip=False))
    ors = oracle_lib.OracleSolver(om, nAlphaBounds=0, clip=False, threads=8)
    for s in (gpu, ors):
        s.set_alpha(alpha)
        s.set_flow(phi, U)
        s.reconstruct()
        s.advect(dt)
    assert gpu.n_mixed() == mesh.n_cells
    assert bits_equal(gpu.alpha_phi(), ors.alpha_phi())
    assert bits_equal(gpu.alpha(), ors.alpha())
    gpu.synchronize()
