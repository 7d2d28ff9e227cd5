"""Least squares by the FP64 LU: the bordered matrix takes over the factors of its transpose.

Panel counts below, at and above one and two of the 512-row blocks whose inverses change sides, and counts
that are no multiple of 4 or 64.  Against the pivoted factorisations of both matrices: two solutions to rounding
of one problem, 1e-9 of the largest strength (the bound of the other least-squares tests).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nm,na", [(10, 16), (16, 32), (17, 31), (33, 32), (23, 55)])
@pytest.mark.parametrize("pres", [None, [(0, 0.3), (57, -0.1)]])
def test_transposed_factors_solve_the_bordered_system(fp, geo, nm, na, pres, monkeypatch):
    body = fp.RigidWakeBody(geo.sphere(n_meridional=nm, n_azimuthal=na), None, formulation=2)
    U = np.tile([[1.0], [0.2], [0.0]], (1, body.ncells))
    ctx = body.ctx
    ctx.profile(True)
    fp.solve(body, U, solver=fp.solve_ludiv, elprescribe=pres)
    count = {k: ctx.profile_get(k)[0] for k in ("lu_nopiv_diag", "lu_nopiv_blockinv", "panel_tslu")}
    ctx.profile(False)
    assert count["lu_nopiv_diag"] == 1 and count["lu_nopiv_blockinv"] == 1 and count["panel_tslu"] == 0
    x = body.strength.copy()
    monkeypatch.setenv("FLOWPANEL_LU64_PIVOTED", "1")
    fp.solve(body, U, solver=fp.solve_ludiv, elprescribe=pres)
    assert np.abs(x - body.strength).max() < 1e-9 * np.abs(body.strength).max()
