"""Solves where the device memory is nearly used up: what the randomized factors need beyond the matrix may be
missing, never the answer.

The context is given a byte limit (a request beyond it fails as hipMalloc does on a full device), in steps from less
than the pivoted LU in place needs to more than every path needs.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
NOMEM = 9


@pytest.fixture
def limit(fp):
    ctx = fp._native.context()
    f = fp._native.lib().fp_test_limit_bytes
    f.argtypes, f.restype = [ctypes.c_void_p, ctypes.c_int64], None

    def set_limit(nbytes, trim=True):
        if trim:
            ctx.trim()
        f(ctx.handle, int(nbytes))
    yield set_limit
    f(ctx.handle, -1)


def _attempt(fp, call):
    try:
        return call()
    except fp.FPError as e:
        assert e.code == NOMEM, e
        return None


def _solve_mat(fp, solver, A, B, nbytes, limit):
    """The solver functions' path, with the limit on the solve alone (the matrix is in place)."""
    nat = fp._native
    L, ctx, n, k = nat.lib(), nat.context(), A.shape[0], B.shape[1]
    h, Af, Bf, X = ctypes.c_void_p(), nat.f64(A), nat.f64(B), np.zeros(B.shape, order="F")
    limit(-1)
    ctx.check(L.fp_mat_upload(ctx.handle, n, nat.dptr(Af), ctypes.byref(h)))
    try:
        limit(nbytes)
        o = nat.opts(fp.solvers._CODES[solver])
        ctx.check(L.fp_solve_mat(ctx.handle, h, nat.dptr(Bf), k, nat.dptr(X), ctypes.byref(o), None))
    finally:
        L.fp_mat_destroy(h)
    return X


def _matrix(n):
    rng = np.random.default_rng(n)
    return rng.standard_normal((n, n)) + 2 * np.sqrt(n) * np.eye(n), rng


@pytest.mark.parametrize("k", [1, 3, 40])
def test_fp64_lu_serves_wherever_the_pivoted_one_does(fp, limit, monkeypatch, k):
    n = 700   # the copy takes 3.9 MB, its block inverses 10.5 MB
    A, rng = _matrix(n)
    X = rng.standard_normal((n, k))
    B = A @ X
    ctx, paths = fp._native.context(), set()
    for mb in np.arange(3.5, 40.0, 0.7):
        got = []
        for pivoted in ("1", "0"):
            monkeypatch.setenv("FLOWPANEL_LU64_PIVOTED", pivoted)
            ctx.profile(True)
            got.append(_attempt(fp, lambda: _solve_mat(fp, fp.solve_ludiv, A, B, mb * 1e6, limit)))
            tslu = ctx.profile_get("panel_tslu")[0]
            ctx.profile(False)
        if got[0] is not None:
            assert got[1] is not None, mb
        if got[1] is not None:
            assert np.abs(got[1] - X).max() < 1e-11 * np.abs(X).max(), mb
            paths.add(tslu > 0)
    assert paths == {True, False}


@pytest.mark.parametrize("k", [1, 2, 3, 40])
def test_fp32_lu_serves_wherever_its_matrix_and_a_copy_fit(fp, limit, k):
    # the explicit inverses (from four columns on) take three more FP32 matrices, the block inverses 5.2 MB
    n, ld = 700, 704
    A, rng = _matrix(n)
    X = rng.standard_normal((n, k))
    B = A @ X
    need = 2 * 4 * n * ld + 9 * 8 * n * max(k, 4) + 2 * 8 * 128 * 128 * 6
    for nbytes in [need] + [need + x * 1e6 for x in np.arange(0.4, 18.0, 1.1)]:
        got = _solve_mat(fp, fp.solve_lu32_ir, A, B, nbytes, limit)
        assert np.abs(got - X).max() < 1e-9 * np.abs(X).max(), nbytes


def test_a_released_limit_gives_the_randomized_path_back(fp, limit):
    A, rng = _matrix(300)
    limit(1000)
    assert _attempt(fp, lambda: fp.solve_ludiv(None, A, A[:, 0])) is None
    limit(-1)
    x = fp.solve_ludiv(None, A, A[:, 0])
    assert abs(x[0] - 1) < 1e-12 and np.abs(x[1:]).max() < 1e-12


def test_buffers_kept_for_reuse_give_way_to_a_matrix(fp, limit):
    # 18 MB stay in the pool after the solve; the next matrix (3.9 MB and as much to bring it up) is not the pool's own
    A, rng = _matrix(700)
    limit(-1)
    fp.solve_ludiv(None, A, A[:, 0])
    limit(9e6, trim=False)
    body = fp.RigidWakeBody(*fp.geometry.loft_wing(n_chord=20, n_span=10))
    assert body.ncells == 200
    x = fp.solve_ludiv(None, A, A[:, 0])
    assert abs(x[0] - 1) < 1e-12 and np.abs(x[1:]).max() < 1e-12


def test_least_squares_serves_wherever_the_pivoted_one_does(fp, geo, limit, monkeypatch):
    # the factors of the first matrix stay for the second, unless its copy needs their room
    body = fp.RigidWakeBody(geo.sphere(n_meridional=23, n_azimuthal=24), None, formulation=2)
    U = np.tile([[1.0], [0.2], [0.0]], (1, body.ncells))
    ctx, factored = fp._native.context(), set()
    ref = None
    for mb in list(np.arange(45.0, 6.0, -0.5)):
        got = []
        for pivoted in ("1", "0"):
            monkeypatch.setenv("FLOWPANEL_LU64_PIVOTED", pivoted)
            limit(mb * 1e6)
            ctx.profile(True)
            ok = _attempt(fp, lambda: fp.solve(body, U, solver=fp.solve_ludiv) or True)
            counts = tuple(ctx.profile_get(c)[0] > 0 for c in ("lu_nopiv_diag", "panel_tslu"))
            ctx.profile(False)
            got.append(body.strength.copy() if ok else None)
        if got[0] is not None:
            ref = got[0] if ref is None else ref
            assert got[1] is not None, mb
        if got[1] is not None:
            assert np.abs(got[1] - ref).max() < 1e-9 * np.abs(ref).max(), mb
            factored.add(counts)
    assert {(True, False), (False, True)} <= factored


def test_batch_bodies_without_room_for_a_randomized_copy_are_pivoted(fp, geo, limit):
    # 800, 1,008 and 384 panels, whose block inverses take 5.2, 5.2 and 2.6 MB
    V = fp.direction(4.0, 0.0)
    bodies, ref = [], []
    for nc, ns in ((40, 20), (42, 24), (16, 24)):
        b = fp.RigidWakeBody(*geo.loft_wing(n_chord=nc, n_span=ns, span=8.0, taper=0.5, sweep_deg=20.0))
        U, D = np.tile(V[:, None], (1, b.ncells)), np.tile(V[:, None], (1, b.nsheddings))
        fp.solve(b, U, D, D, solver=fp.solve_ludiv)
        ref.append(b.strength.copy())
        bodies.append(b)

    def solve():
        batch = fp.BodyBatch(bodies, solver=fp.solve_lu32_ir)
        for _ in range(3):   # replays of one graph
            batch.solve()
        return [b.strength.copy() for b in bodies]

    # FP64 and FP32 matrices, their copies, and the workspaces of two substitutions and a pivoted panel
    sizes = [(b.ncells, (b.ncells + 63) // 64 * 64) for b in bodies]
    need = sum(16 * n * ld + 2 * 8 * (2 * n + 2 * 16384 * ((n + 127) // 128)) + 1200000 + 200 * n for n, ld in sizes)
    served = 0
    for nbytes in [need] + [need + x * 1e6 for x in np.arange(-22.0, 14.0, 1.5)]:
        limit(nbytes)
        got = _attempt(fp, solve)
        assert got is not None or nbytes < need
        if got is not None:
            served += 1
            for g, r in zip(got, ref):
                assert np.abs(g - r).max() < 1e-8 * np.abs(r).max(), nbytes
    assert served >= 10


@pytest.mark.parametrize("what", ["Uind", "phi"])
def test_field_without_room_for_partial_sums(fp, geo, limit, what):
    # 530,000 targets and what is returned there fit, the partial sums of the splits do not
    b = fp.RigidWakeBody(*geo.loft_wing(n_chord=24, n_span=40, span=8.0, sweep_deg=20.0))
    V = fp.direction(4.0, 0.0)
    U, D = np.tile(V[:, None], (1, b.ncells)), np.tile(V[:, None], (1, b.nsheddings))
    fp.solve(b, U, D, D)
    nt = 530000
    T = np.asfortranarray(np.random.default_rng(7).uniform([[-1.0], [-4.0], [-1.0]], [[3.0], [4.0], [1.0]], (3, nt)))
    out = [np.zeros((3, nt) if what == "Uind" else nt, order="F") for _ in range(2)]
    getattr(fp, what)(b, T, out[0])
    limit(24 * nt + out[0].nbytes + 4096)
    getattr(fp, what)(b, T, out[1])
    # the same terms in one sum instead of several
    assert np.abs(out[0] - out[1]).max() < 2000 * np.finfo(float).eps * np.abs(out[0]).max()
