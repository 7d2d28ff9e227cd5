"""Coarse spaces from 512 vectors up: inverted through the randomized no-pivot LU, Gauss-Jordan behind it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _coupled(n, coarse, shift):
    rng = np.random.default_rng(8100 + n)
    A = rng.standard_normal((n, n)) / np.sqrt(n) + shift * np.eye(n)
    A += np.kron(rng.uniform(0.0, 0.4, (n // coarse + 1, n // coarse + 1)), np.ones((coarse, coarse)))[:n, :n] / coarse
    return A, rng.standard_normal(n)


def _refused(fp, call):
    """What `call` returns and the inverses by LU that it gave up: the set-up's first one, by whichever method, runs on a
    side stream that is not profiled; a Gauss-Jordan on the context's own stream is a repetition."""
    ctx = fp._native.context()
    ctx.profile(True)
    out = call()
    count = ctx.profile_get("coarse_inverse_gj")[0]
    ctx.profile(False)
    return out, count


@pytest.mark.parametrize("n,coarse,shift", [(1022, 2, 8.0), (1023, 2, 8.0), (1537, 3, 8.0), (2601, 1, 8.0), (2600, 2, 2.0)])
def test_default_inverse_preconditions_like_gauss_jordan(fp, n, coarse, shift, monkeypatch):
    # 511 vectors (below the rule), 512, 513 and 2,601; with a shift of 2 the coarse matrix is close to singular
    # and what FP32 makes of it may be refused: never worse than Gauss-Jordan by more than an iteration or two
    A, b = _coupled(n, coarse, shift)
    opts = dict(precond_block=100, coarse_block=coarse, tol=1e-12)
    y, refused = _refused(fp, lambda: fp.solve_gmres_ir(None, A, b, **opts))
    it = fp.solvers.last_stats["iterations"]
    assert shift < 4 or refused == 0
    monkeypatch.setenv("FLOWPANEL_COARSE_INV", "gj")
    y_gj = fp.solve_gmres_ir(None, A, b, **opts)
    it_gj = fp.solvers.last_stats["iterations"]
    x = np.linalg.solve(A, b)
    scale = np.abs(x).max()
    assert np.abs(y - x).max() < 1e-10 * scale * (1 if shift > 4 else 100)
    assert it <= it_gj + (1 if shift > 4 else 2), (it, it_gj)
    if (n + coarse - 1) // coarse < 512:
        assert np.array_equal(y, y_gj)


def test_singular_coarse_matrix_is_refused_by_both(fp, monkeypatch):
    # every 2 x 2 block of chunk sums is zero: E = 0, although A is not singular
    n = 1200
    A = np.kron(np.eye(n // 2), np.array([[2.0, 1.0], [-1.0, -2.0]]))
    b = np.ones(n)
    text = []
    for inv in ("", "gj"):
        monkeypatch.setenv("FLOWPANEL_COARSE_INV", inv)
        with pytest.raises(fp.FPError, match="Galerkin") as e:
            fp.solve_gmres_ir(None, A, b, precond_block=100, coarse_block=2, tol=1e-12)
        text.append(str(e.value))
    assert text[0] == text[1]
    # each time the LU's verdict was repeated by the Gauss-Jordan first
    monkeypatch.setenv("FLOWPANEL_COARSE_INV", "")

    def solve():
        with pytest.raises(fp.FPError):
            fp.solve_gmres_ir(None, A, b, precond_block=100, coarse_block=2, tol=1e-12)
    assert _refused(fp, solve)[1] == 1


@pytest.mark.parametrize("nc,ns,coarse", [(40, 40, 3), (60, 40, 3), (50, 60, 1), (46, 33, 2)])
@pytest.mark.parametrize("tri", [False, True])
def test_bodies_iterate_as_with_gauss_jordan(fp, geo, nc, ns, coarse, tri, monkeypatch):
    # 534 to 3,000 coarse vectors of a swept wing's own matrix, quads and triangles
    grid, sh = geo.loft_wing(n_chord=nc, n_span=ns, span=10.0, taper=0.5, sweep_deg=30.0)
    if tri:
        grid, sh = geo.triangulate(grid, sh)
        coarse *= 2
    b = fp.RigidWakeBody(grid, sh)
    V = fp.direction(4.0, 1.0)
    U, D = np.tile(V[:, None], (1, b.ncells)), np.tile(V[:, None], (1, b.nsheddings))
    strip = nc * (2 if tri else 1)
    iters, gamma = [], []
    for inv in ("", "gj"):
        monkeypatch.setenv("FLOWPANEL_COARSE_INV", inv)
        _, refused = _refused(fp, lambda: fp.solve(b, U, D, D, solver=fp.solve_gmres_ir, solver_optargs={
            "precond_block": 4 * strip, "coarse_block": coarse, "tol": 1e-10}))
        assert refused == 0
        iters.append(fp.solvers.last_stats["iterations"])
        gamma.append(b.strength.copy())
    assert abs(iters[0] - iters[1]) <= 1, iters
    assert np.abs(gamma[0] - gamma[1]).max() < 1e-7 * np.abs(gamma[1]).max()
