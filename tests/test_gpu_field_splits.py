"""Split field launches: the panel stream and the wake horseshoes are both cut over the splits.

Target counts on either side of where the number of splits changes (one workgroup of targets, 512
workgroups = 131,072 targets, and the first count above it), a body with more horseshoes than splits and
one with fewer.  Against the oracle's plain sums at a sample of the targets: 1e-10 of the largest
velocity (the field tests' bound), 1e-9 for the potential.
"""
import types

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,ns", [(8, 3), (6, 40)])
@pytest.mark.parametrize("nt", [1, 257, 131072, 131073])
def test_field_splits_match_oracle(fp, geo, orc, nc, ns, nt):
    grid, sh = geo.loft_wing(n_chord=nc, n_span=ns, span=5.0, sweep_deg=15.0)
    b = fp.RigidWakeBody(grid, sh)
    V = fp.direction(3.0, 1.0)
    D = np.tile(V[:, None], (1, b.nsheddings))
    fp.solvers.set_freestream(b, np.tile(V[:, None], (1, b.ncells)), D, D)
    rng = np.random.Generator(np.random.PCG64(nt))
    g = rng.uniform(-1, 1, b.ncells)
    b.ctx.check(fp._native.lib().fp_body_set_strength(b.ctx.handle, b.handle, fp._native.dptr(g)))
    X = np.asfortranarray(rng.uniform([[-1.0], [-3.0], [-1.0]], [[4.0], [3.0], [1.0]], (3, nt)))
    at = np.unique(np.concatenate([[0, nt - 1], rng.integers(0, nt, 200)]))
    ob = types.SimpleNamespace(nodes=grid.nodes, cell_ptr=grid.cell_ptr, cell_idx=grid.cell_idx, ncells=b.ncells,
                               element="vortexring", shedding=b.shedding, nsheddings=b.nsheddings,
                               kerneloffset=b.kerneloffset, kernelcutoff=b.kernelcutoff, CPoffset=b.CPoffset,
                               charlen_kind=0)
    U = fp.Uind(b, X, np.zeros_like(X))[:, at]
    Uo = orc.uind(ob, g, X[:, at], D, D)
    assert np.abs(U - Uo).max() < 1e-10 * np.abs(Uo).max()
    p = fp.phi(b, X, np.zeros(nt))[at]
    po = orc.phi(ob, g, X[:, at], D, D)
    assert np.abs(p - po).max() < 1e-9 * np.abs(po).max()
