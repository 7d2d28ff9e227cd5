"""Wake columns of the AIC: horseshoes grouped by column, one lane per group.

The edges of that split: more than 64 groups (two waves of columns), target counts that are no
multiple of a workgroup's targets, panels that shed from two edges (a group of several horseshoes,
added in shedding order) and one-sided edges.  Against the oracle's AIC, whose wake is a plain loop
over the shedding list: 1e-12 of the largest entry, the bound of the FP64 assembly tests.
"""
import types

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _shedding(sh, case):
    if case == "plain":
        return sh
    if case == "one-sided":
        out = sh.copy()
        out[3, ::2] = -1
        return out
    # every third upper panel sheds from its next edge too (local vertices 3, 2 beside 2, 1)
    more = sh[:, ::3].copy()
    more[1], more[2], more[3] = 3, 2, -1
    return np.hstack([sh, more, sh[:, 1:3]])


@pytest.mark.parametrize("nc,ns", [(4, 2), (6, 33), (10, 71)])
@pytest.mark.parametrize("case", ["plain", "one-sided", "shared"])
def test_wake_groups_match_oracle(fp, geo, orc, nc, ns, case):
    grid, sh = geo.loft_wing(n_chord=nc, n_span=ns, span=6.0, sweep_deg=20.0)
    b = fp.RigidWakeBody(grid, _shedding(sh, case))
    V = fp.direction(4.0, 1.0)
    D = np.tile(V[:, None], (1, b.nsheddings))
    fp.solvers.set_freestream(b, np.tile(V[:, None], (1, b.ncells)), D, D)
    ob = types.SimpleNamespace(nodes=grid.nodes, cell_ptr=grid.cell_ptr, cell_idx=grid.cell_idx, ncells=b.ncells,
                               element="vortexring", shedding=b.shedding, nsheddings=b.nsheddings,
                               kerneloffset=b.kerneloffset, kernelcutoff=b.kernelcutoff, CPoffset=b.CPoffset,
                               charlen_kind=0)
    Go, _, _ = orc.assemble([ob], [D], [D])
    G = fp.assemble(b, "f64")
    assert np.abs(G - Go).max() < 1e-12 * np.abs(Go).max()
    G32 = fp.assemble(b, "f32")
    assert np.abs(G32 - Go).max() < 2e-7 * np.abs(Go).max()   # two roundings to FP32
