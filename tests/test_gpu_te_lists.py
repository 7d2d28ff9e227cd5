"""Trailing-edge lists: Kutta averaging and the trailing-edge terms of -1/2 grad(mu), an entry per lane.

List lengths around the 64 lanes of a wave, with disjoint panels (every edge at once), panels that belong
to several edges (list order matters) and edges without a second panel.  The averages are the ones in list
order: equal to the plain loop to the rounding of a quarter of a sum of four, 4 eps of the largest value
per edge that a panel belongs to (at most 40 here).
"""
import types

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [1, 63, 64, 65, 200])
@pytest.mark.parametrize("kind", ["disjoint", "shared", "mixed"])
@pytest.mark.parametrize("mode", [1, 2])
def test_kutta_lists_match_the_loop(fp, ns, kind, mode):
    nat = fp._native
    assert {nat.FP_KUTTA_REFERENCE, nat.FP_KUTTA_PAIR} == {1, 2}
    rng = np.random.Generator(np.random.PCG64(ns))
    n = 4 * ns + 4
    if kind == "disjoint":
        q = rng.permutation(ns)
        pi, pj = 4 * q, 4 * q + 3
    else:
        pi, pj = rng.integers(1, 12, ns), rng.integers(1, n - 1, ns)
        if kind == "mixed":
            pi = np.where(np.arange(ns) < ns // 2, 4 * np.arange(ns), pi)
            pj = np.where(rng.random(ns) < 0.3, -1, pj)
    pi, pj = np.minimum(pi, n - 2), np.where(pj < 0, -1, np.maximum(pj, 1))
    sh = np.zeros((ns, 6), dtype=np.int64)
    sh[:, 0], sh[:, 3] = pi, pj
    U = np.asfortranarray(rng.uniform(-1, 1, (3, n)))
    out = np.zeros(n)
    ctx = nat.context()
    ctx.check(nat.lib().fp_calcfield_cp(ctx.handle, nat.dptr(U), n, 1.5, nat.iptr(sh), ns, 0, mode, nat.dptr(out)))
    ref = 1 - (np.sqrt((U * U).sum(axis=0)) / 1.5) ** 2
    for i, j in zip(pi, pj):
        if mode == nat.FP_KUTTA_REFERENCE:
            at = [i, i + 1] + ([j, j - 1] if j != -1 else [])
            ref[at] = sum(ref[k] for k in at) / len(at)
        elif j != -1:
            ref[[i, j]] = (ref[i] + ref[j]) / 2
    assert np.abs(out - ref).max() < 40 * 4 * np.finfo(float).eps * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("ns", [1, 31, 32, 33, 100])
@pytest.mark.parametrize("repeats", [False, True])
def test_te_terms_match_oracle(fp, geo, orc, ns, repeats):
    grid, sh = geo.loft_wing(n_chord=4, n_span=ns, span=5.0, sweep_deg=10.0)
    sh = np.array(sh)
    if repeats:   # edges that name the panels of another edge once more
        sh[:, -1] = sh[:, 0]
        sh[:, ns // 2] = sh[:, 0]
    b = fp.RigidWakeBody(grid, sh)
    g = np.random.Generator(np.random.PCG64(ns)).uniform(-1, 1, b.ncells)
    V = fp.direction(3.0, 1.0)
    D = np.tile(V[:, None], (1, b.nsheddings))
    fp.solvers.set_freestream(b, np.tile(V[:, None], (1, b.ncells)), D, D)
    b.ctx.check(fp._native.lib().fp_body_set_strength(b.ctx.handle, b.handle, fp._native.dptr(g)))
    b.solved = True
    ob = types.SimpleNamespace(nodes=grid.nodes, cell_ptr=grid.cell_ptr, cell_idx=grid.cell_idx, ncells=b.ncells,
                               element="vortexring", shedding=b.shedding, nsheddings=b.nsheddings,
                               kerneloffset=b.kerneloffset, kernelcutoff=b.kernelcutoff, CPoffset=b.CPoffset,
                               charlen_kind=0)
    out = fp.calcfield_Ugradmu_cell(b)
    ref = orc.ugradmu_cell(ob, g, b.shedding, te=True)
    assert np.abs(out - ref).max() < 1e-11 * max(1.0, np.abs(ref).max())
