"""The autotuner against block launches: a form that switches them off is kept only
where it beats them by wall clock. On the CPU the stand-in of the HIP runtime makes the
persistent kernel win by kernel events (one interval per substep instead of three) and
lose by wall clock (its launches, and graphs, take 2 ms)."""
import numpy as np
import pytest

import block_forms
import hip_stub

CODE = """
import numpy as np
from cmf import maps, synth
from cmf.model import CMFModel
stub.stub_slow(2)
out = []
for order in ("dfs", "nseq"):                  # with and without a partition
    import os
    os.environ["CMF_HIP_ORDER"] = order
    net = synth.make_network(48, 24, seed=21)
    g = CMFModel(maps.build_map(net, maps.Options(ladpstp=False)))
    best, rep = g.autotune(3600.0, nsub=4)
    g.physics_advance(3600.0)
    out.append([best["fused"], [int(r[0]) for r in rep if r[0] > 1], g.block_info()["launches"]])
result(out)
"""


def test_persistent_kernel_has_to_beat_blocks(tmp_path):
    blocks, none = hip_stub.run(tmp_path, CODE)
    assert blocks[0] == 0 and blocks[1] == [2, 3, 4] and blocks[2] == 1
    assert none == [1, [], 0]                  # nothing to compare with: kernel events decide, as ever


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["all", "cut_lev_dam", "one_round", "ens_2", "ens_32"])
def test_keeps_the_fastest_whole_step(form):
    g, st, ro = block_forms.model(form, "fp64")
    g.set_state(st)
    g.set_runoff(ro)
    before = g.get_state()
    best, rep = g.autotune(86400.0, nsub=4)
    walls = {int(r[0]): r[7] for r in rep if r[0] > 1}
    assert {2, 3} <= set(walls)
    kept = 4 if best["fused"] else (3 if best["graph"] else 2)
    assert walls[kept] == min(walls.values())
    after = g.get_state()
    for k in before:
        assert np.array_equal(before[k], after[k]), k
    step = g.ensemble_advance if g.ensemble else g.physics_advance
    step(86400.0, nt_cap=9)
    assert (g.block_info()["launches"] > 0) == (kept == 2 and form != "ens_32")
    g.close()
