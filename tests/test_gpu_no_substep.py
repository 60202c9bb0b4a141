"""An instance whose CFL bound admits no substep count (an infinite depth: NT overflows)
takes none: its averages and maxima stay those of the step before, in block launches as
in the phase kernels, and its neighbours are not touched."""
import numpy as np
import pytest

import block_forms

pytestmark = pytest.mark.gpu
NAMES = ["rivout_avg", "fldout_avg", "outflw_avg", "rivvel_avg", "pthout_avg", "runoff_avg", "outflw_max", "rivdph_max",
         "storge_max", "rivout", "fldout", "outflw", "rivvel"]


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("form", ["ens_whole", "ens_2"])           # closed, open partition
def test_instance_without_substeps(form, prec):
    got = []
    for graph in (0, 1):
        g, st, ro = block_forms.model(form, prec)
        g.set_tune(graph=graph)
        g.set_state(st)
        g.set_runoff(ro)
        g.ensemble_advance(86400.0, nt_cap=7)
        assert (g.block_info()["launches"] > 0) == (graph == 0)
        before = g.get_state(NAMES)
        first = g.get_state(["rivsto"])["rivsto"]
        first[1, 5] = np.inf                                       # second member of the first domain
        g.set_state(dict(rivsto=first))
        nt, _ = g.ensemble_advance(86400.0, nt_cap=7)
        assert nt.tolist().count(nt[1]) == 1 and nt[1] < 1 and (np.delete(nt, 1) > 0).all()
        after = g.get_state(NAMES)
        cells = int(g.dom_cells[0])
        for k in NAMES:
            assert np.array_equal(after[k][1, :cells], before[k][1, :cells]), k
        got.append(after)
        g.close()
    for k in NAMES:
        assert np.array_equal(got[0][k], got[1][k]), k
