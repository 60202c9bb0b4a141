"""Paths with an end outside the network carry nothing: their flows, averages and sums
are zero after a step, whatever was uploaded, also where no path has both ends inside.
Then the partition follows the rivers alone."""
import numpy as np
import pytest

import block_forms
import hip_stub
from test_gpu_blocks import PATH_KEYS, STATE_KEYS

CODE = """
import block_forms
dead = block_forms.regional(9000, 0.3, 60, "fp64", 12, 5, 1)[0]
none = block_forms.regional(9000, 0.3, 60, "fp64")[0]
result([dead.block_info(), none.block_info()])
"""


def test_partition_without_live_paths(tmp_path):
    dead, none = hip_stub.run(tmp_path, CODE)
    assert none["cells"] > 0 and dead == none


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("cells, dead", [(9000, 1), (9000, 3), (600, 1)])
def test_dead_paths(cells, dead, prec):
    got = []
    for graph in (0, 1):                                   # block launches, phase kernels
        g, st, ro = block_forms.regional(cells, 0.3, 60, prec, 12, 5, dead)
        rng = np.random.default_rng(5)
        st.update({k: rng.uniform(0.5, 3.0, st[k].shape) for k in ("pthflw", "pthflw_pre", "pthflwsum") if k in st})
        gone = (g.map.pth_upst < 0) | (g.map.pth_down < 0)
        assert gone.all() if dead == 1 else 0 < gone.sum() < g.map.npth
        g.set_tune(graph=graph)
        g.set_state(st)
        g.set_runoff(ro)
        out = []
        for cap in (4, 1, 11):
            g.physics_advance(86400.0, nt_cap=cap)
            assert graph == 1 or cap == 1 or g.block_info()["launches"] > 0
            out.append(g.get_state(STATE_KEYS + PATH_KEYS + ["levsto", "damsto"]))
            for k in ("pthflw", "pthflw_avg", "pthflwsum", "pthflwsum_avg"):
                if k in out[-1]:
                    assert not out[-1][k][..., gone].any(), (k, cap)
        got.append(out)
        g.close()
    for a, b in zip(*got):
        for k in a:
            assert np.array_equal(a[k], b[k]), k
