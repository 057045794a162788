"""PLIC polygons of every cell type against the oracle: lanes per cell by mesh,
fewer cells than a wave takes and more than the grid takes in one pass, planes
that cross a face four times (warped faces of up to 8 points), and cells
reconstructed through split faces.  Cells and polygon sizes are exact; a point
is held to 1e-12, since the copy of a crossing that an edge's two faces leave
is chosen by angles, where two atan2 can differ in the last place."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (63 cells a workgroup at most: 4096 workgroups of 10 hexahedra hold 40960)
CASES = [("hex", 1, {}), ("hex", 3, {}), ("hexp", 9, {}), ("hexp", 35, {}), ("tet", 2, {}), ("tet", 7, {}),
         ("refined", 8, {}), ("refined", 12, {}), ("bricks", 5, {}), ("bricks", 9, {}),
         ("hexp", 6, {"splitWarpedFace": True})]


@pytest.mark.parametrize("kind,N,kw", CASES)
def test_plic_every_cell_type(oracle_lib, kind, N, kw):
    import geometricvofext_amd as g
    print("plic", kind, N, kw, flush=True)
    mesh = {"hex": lambda: g.hex_box(N), "hexp": lambda: g.hex_box(N, perturb=0.2, seed=N),
            "tet": lambda: g.tet_box(N, perturb=0.1, seed=N), "refined": lambda: g.refined_hex_box(N),
            "bricks": lambda: g.brick_box(N, seed=N, perturb=0.1)}[kind]()
    om = oracle_lib.OracleMesh(mesh)
    rng = np.random.default_rng(N)
    alpha = rng.uniform(0.02, 0.98, mesh.n_cells)
    if kind == "bricks":
        x = om.C @ np.array([0.3, 0.5, 0.8])
        alpha = 0.02 + 0.96 * (x - x.min()) / (x.max() - x.min())
    opts = dict(nAlphaBounds=0, clip=False, **kw)
    gpu = g.SolveVofEqu(mesh, dict(orientationMethod="LS", **opts))
    ors = oracle_lib.OracleSolver(om, threads=8, **opts)
    for s in (gpu, ors):
        s.set_alpha(alpha)
        s.reconstruct()
    a, b = gpu.plic_surface(), ors.plic_surface()
    assert np.array_equal(a["cells"], b["cells"])
    assert np.array_equal(a["offsets"], b["offsets"])
    assert a["points"].size == 0 or np.max(np.abs(a["points"] - b["points"])) <= 1e-12
    print(len(a["cells"]), "polygons", len(a["points"]), "points", flush=True)
