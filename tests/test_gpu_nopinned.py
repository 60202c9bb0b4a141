"""Results without pinned memory equal those with it: states, output-period values,
budget rows beyond the first sixteen, and inference over several chunks of rows."""
import pytest

import hip_stub

pytestmark = pytest.mark.gpu

CODE = """
import numpy as np
import block_forms
from cmf.surrogate import MLP, N_IN
rng = np.random.default_rng(3)
x = rng.normal(size=(40001, N_IN)).astype(np.float32)
runs = []
for none in (False, True):
    for form in ("cut_lev_dam", "one_round"):
        g, st, ro = block_forms.model(form, "fp64")      # cmf_hip_create needs some
        m = MLP(max_batch=20000, seed=1)
        stub.stub_fail(0, 0, int(none), 0)
        g.set_state(st)
        g.set_runoff(ro)
        nt, glb = g.physics_advance(86400.0, nt_cap=40, budget=True)
        assert len(glb) == 40
        g.diag_avemax_output(3600.0)
        runs.append(dict(g.get_state(), glb=glb, one=g.get_state(["rivsto"])["rivsto"], y=m.forward(x), y1=m.forward(x[:7]),
                         **{"out_" + k: v for k, v in g.get_output().items()}))
        g.close()
        m.close()
        assert (stub.stub_refused() > 0) == none
        stub.stub_fail(0, 0, 0, 0)
for a, b in zip(runs[:2], runs[2:]):
    assert a.keys() == b.keys()
    for k in a:
        assert np.array_equal(a[k], b[k]), k
result(len(runs[0]))
"""


def test_same_results(tmp_path):
    assert hip_stub.run(tmp_path, CODE, "hip_nopin.c", timeout=100) > 30
