"""Refusal of non-finite inputs: every value is looked at (first, last, and past
the first round of the grid), the count is exact, and phi is named before U."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,where", [(2, [0]), (2, [7]), (9, [0, 1, 728]), (65, [262143, 262144, 274624])])
def test_non_finite_alpha_and_flow(N, where):
    import geometricvofext_amd as g
    print("non-finite", N, where, flush=True)
    mesh = g.hex_box(N)
    s = g.SolveVofEqu(mesh, dict(orientationMethod="LS"))
    ok = np.full(mesh.n_cells, 0.25)
    bad = ok.copy()
    bad[where] = [(np.nan, np.inf, -np.inf)[k] for k in range(len(where))]
    with pytest.raises(Exception, match=f"alpha: {len(where)} non-finite"):
        s.set_alpha(bad)
    s.set_alpha(ok)
    phi, U = np.zeros(mesh.n_faces), np.zeros((mesh.n_cells, 3))
    badU, badPhi = U.copy(), phi.copy()
    badU[where, 2] = np.nan
    badPhi[-1] = np.inf
    with pytest.raises(Exception, match=f"U: {len(where)} non-finite"):
        s.set_flow(phi, badU)
    with pytest.raises(Exception, match="phi: 1 non-finite"):
        s.set_flow(badPhi, badU)
    s.set_flow(phi, U)
    assert np.array_equal(s.alpha(), ok)
