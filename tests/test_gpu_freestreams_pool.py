"""Many freestreams in one call, and the context's pool of small buffers."""
import ctypes
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 3, 65])
@pytest.mark.parametrize("nc,ns", [(4, 1), (8, 33)])
def test_freestreams_match_single_solves(fp, geo, k, nc, ns):
    # 4 and 264 panels: less than a workgroup of points, and one with a remainder
    grid, sh = geo.loft_wing(n_chord=nc, n_span=ns, span=5.0, sweep_deg=10.0)
    b = fp.RigidWakeBody(grid, sh)
    rng = np.random.Generator(np.random.PCG64(k))
    U = rng.uniform(0.5, 1.5, (3, b.ncells, k))
    D = np.tile(fp.direction(2.0, 0.0)[:, None], (1, b.nsheddings))
    many = fp.solve_freestreams(b, U, D, D, solver=fp.solve_ludiv)[0]
    for c in {0, k // 2, k - 1}:
        fp.solve(b, np.asfortranarray(U[:, :, c]), D, D, solver=fp.solve_ludiv)
        # both are solutions to rounding; a wing with a sharp trailing edge: 1e-11 of the largest strength
        assert np.abs(np.asarray(many)[:, c] - b.strength).max() < 1e-10 * np.abs(b.strength).max()
    for bad in (np.nan, np.inf):
        V = U.copy()
        V[2, b.ncells - 1, k - 1] = bad
        with pytest.raises(fp.FPError, match="finite"):
            fp.solve_freestreams(b, V, D, D, solver=fp.solve_ludiv)


def test_small_buffers_survive_many_sizes_and_a_closed_context(fp):
    # more sizes than the pool keeps, then a trim, then another context closed with buffers in its pool
    rng = np.random.Generator(np.random.PCG64(5))
    for n in list(range(3, 90)) + [40, 40]:
        A = rng.standard_normal((n, n)) + n * np.eye(n)
        x = rng.standard_normal(n)
        got = fp.solve_ludiv(None, A, A @ x)
        assert np.abs(got - x).max() < 64 * n * np.finfo(float).eps * np.linalg.cond(A) * np.abs(x).max()
    fp.context().trim()
    A = rng.standard_normal((50, 50)) + 50 * np.eye(50)
    assert np.allclose(fp.solve_ludiv(None, A, A @ np.ones(50)), 1.0)
    nat = fp._native
    L, other = nat.lib(), nat.Context(0)
    h, Af, x = ctypes.c_void_p(), nat.f64(A), np.zeros((50, 1), order="F")
    other.check(L.fp_mat_upload(other.handle, 50, nat.dptr(Af), ctypes.byref(h)))
    o = nat.opts(nat.FP_SOLVER_LU)
    other.check(L.fp_solve_mat(other.handle, h, nat.dptr(nat.f64((A @ np.ones(50)).reshape(50, 1))), 1, nat.dptr(x),
                               ctypes.byref(o), None))
    L.fp_mat_destroy(h)
    assert np.allclose(x, 1.0)
    del other   # with the solve's buffers in its pool
    gc.collect()
    assert np.allclose(fp.solve_ludiv(None, A, A @ np.ones(50)), 1.0)


def test_a_failed_call_leaves_nothing_behind_in_the_pool(fp, geo):
    # the call is refused by the preconditioner's set-up while its assembly is still queued; the matrix uploaded next
    # has the assembly's size (n = 4,800 is a multiple of 64, so that n x n and n x ld are the same)
    grid, sh = geo.loft_wing(n_chord=60, n_span=80, span=10.0, taper=0.5, sweep_deg=30.0)
    b = fp.RigidWakeBody(grid, sh)
    V = fp.direction(4.0, 0.0)
    U, D = np.tile(V[:, None], (1, b.ncells)), np.tile(V[:, None], (1, b.nsheddings))
    rng = np.random.Generator(np.random.PCG64(6))
    n = b.ncells
    A = rng.standard_normal((n, n)) + n * np.eye(n)
    for _ in range(3):
        with pytest.raises(fp.FPError, match="4096"):
            fp.solve(b, U, D, D, solver=fp.solve_gmres, solver_optargs={"precond_block": 60, "coarse_block": 1})
        got = fp.solve_ludiv(None, A, A @ np.ones(n))
        assert np.abs(got - 1.0).max() < 1e-12


@pytest.mark.parametrize("k", [8, 9, 16, 17, 32, 33, 64, 65])
@pytest.mark.parametrize("nc,ns", [(6, 7), (10, 5), (8, 33)])
def test_many_refined_freestreams_match_single_solves(fp, geo, k, nc, ns):
    # the refinement's products with many columns: column groups of 8 (vector form), 16, 32 and 64 and one more;
    # 42, 50 and 264 rows (tiles of 16, rows no multiple of 4 or 16).  Uniform freestreams: the
    # ring matrix of a closed body is nearly singular for one with a net flux through it
    grid, sh = geo.loft_wing(n_chord=nc, n_span=ns, span=5.0, sweep_deg=10.0)
    b = fp.RigidWakeBody(grid, sh)
    rng = np.random.Generator(np.random.PCG64(100 + k))
    V = np.stack([fp.direction(a, s) for a, s in rng.uniform(-5, 5, (k, 2))], axis=1)
    U = np.repeat(V[:, None, :], b.ncells, axis=1)
    D = np.tile(fp.direction(2.0, 0.0)[:, None], (1, b.nsheddings))
    many = np.asarray(fp.solve_freestreams(b, U, D, D, solver=fp.solve_lu32_ir)[0])
    for c in sorted({0, 7, k // 2, k - 1}):
        fp.solve(b, np.asfortranarray(U[:, :, c]), D, D, solver=fp.solve_ludiv)
        # refined to a residual of 1e-12; the wing's amplification of it stays below 1e-8 of the largest strength
        assert np.abs(many[:, c] - b.strength).max() < 1e-8 * np.abs(b.strength).max(), c
