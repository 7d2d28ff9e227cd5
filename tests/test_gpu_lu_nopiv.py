"""The FP64 LU path: randomized no-pivot factors with refinement, and what falls back to pivoting.

Sizes straddle the 16-column sub-panels, the 64-row blocks, the 256-column outer blocks, the 32-column
groups of the U rows and the pad to a multiple of 4.  The reference is LAPACK on the same matrix; the
bound 64 n eps kappa is the usual forward bound of a backward stable solve with room for the constant.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def _matrix(n, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((n, n)) + 0.5 * np.sqrt(n) * np.eye(n), rng


def _counted(fp, A, B):
    ctx = fp._native.context()
    ctx.profile(True)
    X = fp.solve_ludiv(None, A, B)
    counts = {name: ctx.profile_get(name)[0] for name in ("getrs", "panel_tslu")}
    ctx.profile(False)
    return X, counts


@pytest.mark.parametrize("n", [1, 2, 5, 15, 17, 63, 64, 65, 129, 255, 256, 257, 288, 290, 321, 513, 771])
@pytest.mark.parametrize("k", [1, 3])
@pytest.mark.parametrize("pivoted", ["0", "1"])
def test_fp64_lu_matches_lapack(fp, n, k, pivoted, monkeypatch):
    monkeypatch.setenv("FLOWPANEL_LU64_PIVOTED", pivoted)
    A, rng = _matrix(n, 100 + n)
    X = rng.standard_normal((n, k))
    B = A @ X
    got, counts = _counted(fp, A, B if k > 1 else B[:, 0])
    assert (counts["panel_tslu"] > 0) == (pivoted == "1"), counts   # the path asked for, and no other
    got = got.reshape(n, k)
    ref = np.linalg.solve(A, B)
    bound = 64 * n * EPS * np.linalg.cond(A)
    assert np.abs(got - ref).max() <= bound * np.abs(ref).max()
    # and backward stable: the residual is at rounding whatever the condition
    r = np.linalg.norm(A @ got - B) / (np.linalg.norm(A) * np.linalg.norm(got))
    assert r < 16 * EPS * np.sqrt(n) + 4 * EPS, r


@pytest.mark.parametrize("n", [576, 577, 640, 835, 1029, 3303])
def test_updates_carried_by_the_next_block(fp, n):
    # from 513 unknowns on, part of each trailing update runs inside the launches that factor the next 256
    # columns; at 3,303 a part does not fit and is a product of its own.  The factors have to be good enough
    # by themselves: no pivoted panel runs.
    A, rng = _matrix(n, 200 + n)
    b = A @ rng.standard_normal(n)
    ctx = fp._native.context()
    ctx.profile(True)
    x = fp.solve_ludiv(None, A, b)
    counts = {name: ctx.profile_get(name)[0] for name in ("lu_nopiv_update", "panel_tslu", "gemm_f64")}
    ctx.profile(False)
    assert counts["lu_nopiv_update"] == (n + 3) // 4 * 4 // 256 - ((n + 3) // 4 * 4 % 256 == 0)
    assert counts["panel_tslu"] == 0
    assert (counts["gemm_f64"] > 0) == (n == 3303)
    r = np.linalg.norm(A @ x - b) / (np.linalg.norm(A) * np.linalg.norm(x))
    assert r < 16 * EPS * np.sqrt(n) + 4 * EPS, r


@pytest.mark.parametrize("n", [64, 300])
def test_permutation_needs_no_pivots(fp, n):
    # a zero diagonal: plain elimination without pivoting stops at the first column
    rng = np.random.default_rng(n)
    A = np.eye(n)[rng.permutation(n)] * rng.uniform(1, 2, n)
    b = rng.standard_normal(n)
    x = fp.solve_ludiv(None, A, b)
    assert np.abs(A @ x - b).max() < 1e-13


def test_singular_matrix_is_refused_as_before(fp):
    # exactly singular (a zero column), consistent right-hand side: the pivoted LU meets a zero pivot
    A, rng = _matrix(200, 3)
    A[:, 77] = 0.0
    with pytest.raises(fp.FPError) as e:
        fp.solve_ludiv(None, A, A @ rng.standard_normal(200))
    assert e.value.code == 6


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_not_finite_is_an_error(fp, bad):
    A, rng = _matrix(130, 4)
    b = rng.standard_normal(130)
    b[5] = bad
    with pytest.raises(fp.FPError):
        fp.solve_ludiv(None, A, b)


def test_nearly_singular_matrix_matches_pivoted(fp, monkeypatch):
    # condition 1e14: both paths give a backward stable solution of their own
    rng = np.random.default_rng(9)
    n = 150
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    P, _ = np.linalg.qr(rng.standard_normal((n, n)))
    A = Q @ np.diag(np.logspace(0, -14, n)) @ P
    b = A @ rng.standard_normal(n)
    for pv in ("0", "1"):
        monkeypatch.setenv("FLOWPANEL_LU64_PIVOTED", pv)
        x = fp.solve_ludiv(None, A, b)
        assert np.linalg.norm(A @ x - b) < 64 * n * EPS * (np.linalg.norm(x) + np.linalg.norm(b))


@pytest.mark.parametrize("n,k", [(37, 1), (300, 1), (300, 5), (1031, 2)])
def test_refined_solution_is_accurate_to_the_data(fp, n, k):
    # integer data, so that b = A x is exact: the residuals of twice FP64 take the solution to its own
    # rounding (condition up to 1e6 here; a plain FP64 solve is left with about condition x eps)
    rng = np.random.default_rng(n + k)
    A = rng.integers(-50, 51, (n, n)).astype(float)
    A[:, 0] = A[:, 1:].sum(axis=1) + rng.integers(-1, 2, n)
    X = rng.integers(-9, 10, (n, k)).astype(float)
    got = fp.solve_ludiv(None, A, A @ X).reshape(n, k)
    assert np.abs(got - X).max() < 1e-14 * np.abs(X).max()


def _butterfly(m, seed):
    """One side of the randomization of order 4 m that the library draws from `seed` (splitmix64)."""
    def draw(i):
        mask = (1 << 64) - 1
        z = (seed + (i + 1) * 0x9E3779B97F4A7C15) & mask
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        return np.exp((((z ^ (z >> 31)) >> 11) * 2.0 ** -53 - 0.5) / 10.0)
    F, h = np.zeros((4 * m, 4 * m)), np.sqrt(0.5)
    for q in range(m):
        r = [draw(8 * q + j) for j in range(8)]
        Z = h * np.array([[r[0], 0, r[1], 0], [0, r[2], 0, r[3]], [r[0], 0, -r[1], 0], [0, r[2], 0, -r[3]]])
        Y = h * np.array([[r[4], r[5], 0, 0], [r[4], -r[5], 0, 0], [0, 0, r[6], r[7]], [0, 0, r[6], -r[7]]])
        at = q + m * np.arange(4)
        F[np.ix_(at, at)] = Y @ Z
    return F


SEED = 0x46504C5533324952


def _passes_the_pivots_only(n=64):
    """Condition ~200, but the randomized matrix starts with two pivots of 1e-10 of its norm one behind the other:
    above the pivot test's 1e-11, with an element growth of 1e16 that leaves the factors no correct digit."""
    rng = np.random.default_rng(1)
    M = rng.standard_normal((n, n))
    M[0, 0] = M[1, 1] = 1e-10 * np.linalg.norm(M)
    M[1, 0] = 0.0
    U, V = _butterfly(n // 4, SEED), _butterfly(n // 4, SEED ^ 0x5DEECE66D)
    return np.linalg.solve(U.T, M) @ np.linalg.inv(V)


@pytest.mark.parametrize("k", [1, 3])
def test_factors_without_a_correct_digit_fall_back_to_pivoting(fp, k):
    A = _passes_the_pivots_only()
    n = A.shape[0]
    X = np.random.default_rng(2).standard_normal((n, k))
    B = A @ X
    got, counts = _counted(fp, A, B if k > 1 else B[:, 0])
    assert counts["getrs"] >= 3 and counts["panel_tslu"] > 0, counts   # refined, found wanting, then pivoted
    bound = 64 * n * EPS * np.linalg.cond(A)
    assert np.abs(got.reshape(n, k) - X).max() <= bound * np.abs(X).max()


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("at", [0, 1, 2])
def test_a_column_that_is_not_finite_leaves_the_others(fp, bad, at):
    # the pivoted LU treats columns independently; so does the refined one, also where only pivoting serves
    for A in (_matrix(200, 11)[0], _passes_the_pivots_only()):
        n = A.shape[0]
        X = np.random.default_rng(12).standard_normal((n, 3))
        B = A @ X
        B[5, at] = bad
        got = fp.solve_ludiv(None, A, B)
        assert not np.isfinite(got[:, at]).all()
        rest = [c for c in range(3) if c != at]
        bound = 64 * n * EPS * np.linalg.cond(A)
        assert np.abs(got[:, rest] - X[:, rest]).max() <= bound * np.abs(X[:, rest]).max()


@pytest.mark.parametrize("scale", [1e-200, 1e200])
def test_columns_beyond_the_range_of_their_squares(fp, scale):
    # |b|^2 over- or underflows: the acceptance test cannot see such a column, and a right-hand side of zeros is one
    # with nothing to see
    A = _passes_the_pivots_only()
    n = A.shape[0]
    X = np.random.default_rng(13).standard_normal((n, 3))
    X[:, 1] = 0.0
    B = A @ X
    B[:, 0] *= scale
    got = fp.solve_ludiv(None, A, B)
    got[:, 0] /= scale
    bound = 64 * n * EPS * np.linalg.cond(A)
    assert np.abs(got - X).max() <= bound * np.abs(X).max()
    assert not got[:, 1].any()
    # zeros alone are no reason to pivot
    A, rng = _matrix(130, 14)
    X = rng.standard_normal((130, 3))
    X[:, 1] = 0.0
    got, counts = _counted(fp, A, A @ X)
    assert counts["panel_tslu"] == 0 and not got[:, 1].any()


@pytest.mark.parametrize("n", [257, 258, 259, 260, 5])
@pytest.mark.parametrize("scale", [1e-12, 1.0, 1e12])
@pytest.mark.parametrize("solver", ["solve_ludiv", "solve_lu32_ir"])
def test_units_do_not_decide_the_path(fp, n, scale, solver):
    # the randomized matrix is padded to a multiple of 4: its pad has the matrix's own scale, and is no part of its norm
    A, rng = _matrix(n, 300 + n)
    A += 1.5 * np.sqrt(n) * np.eye(n)   # no eigenvalue near zero: FP32 factors refine it
    X = rng.standard_normal(n)
    ctx = fp._native.context()
    ctx.profile(True)
    x = getattr(fp, solver)(None, scale * A, scale * (A @ X))
    pivoted = ctx.profile_get("panel_tslu")[0]
    ctx.profile(False)
    assert pivoted == 0
    assert np.abs(x - X).max() <= max(64 * n * EPS, 1e-12) * np.linalg.cond(A) * np.abs(X).max()


@pytest.mark.parametrize("solver", ["solve_ludiv", "solve_lu32_ir"])
def test_more_columns_than_a_launch_takes_are_refused_as_by_the_pivoted_lu(fp, solver, monkeypatch):
    A, _ = _matrix(4, 15)
    text = []
    for pivoted in ("1", "0"):
        monkeypatch.setenv("FLOWPANEL_LU64_PIVOTED", pivoted)
        monkeypatch.setenv("FLOWPANEL_LU32_PIVOTED", pivoted)
        with pytest.raises(fp.FPError) as e:
            getattr(fp, solver)(None, A, np.ones((4, 65536)))
        assert e.value.code == 10
        text.append(str(e.value))
    assert text[0] == text[1]
    X = getattr(fp, solver)(None, A, A @ np.ones((4, 65535)))
    assert np.abs(X - 1).max() < 1e-10
