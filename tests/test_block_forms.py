"""Which models step in block launches, and that they do: the comparisons of
test_gpu_blocks.py hold of themselves where both handles run the phase kernels, so
the partition of each of their models is stated here, and the launches are counted."""
import numpy as np
import pytest

import block_forms
import hip_stub

CODE = """
import block_forms
out = {}
for form in block_forms.FORMS:
    for prec in ("fp64", "mixed"):
        g = block_forms.model(form, prec)[0]
        out[form + "/" + prec] = block_forms.partition(g)
        g.close()
result(out)
"""


def test_partitions(tmp_path):
    got = hip_stub.run(tmp_path, CODE)
    for form in block_forms.FORMS:
        for prec in ("fp64", "mixed"):
            want = block_forms.wanted(form, prec)
            assert got[f"{form}/{prec}"] == (None if want is None else list(want)), (form, prec)


# a launch moves the whole state once: least substeps of a step in block launches, where
# it is not one (closed partitions) or two
LEAST = {"ens_rounds": 3, "ens_dam_16": 3}


def launches(form, part, nt):
    if part is None or nt < LEAST.get(form, 1 if part[2] else 2):
        return 0
    return 1 if part[2] else 2 * -(-nt // (2 * part[1]))


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("form", list(block_forms.FORMS))
def test_steps_in_block_launches(form, prec):
    g, st, ro = block_forms.model(form, prec)
    part = block_forms.wanted(form, prec)
    assert block_forms.partition(g) == part
    g.set_state(st)
    g.set_runoff(ro)
    step = g.ensemble_advance if g.ensemble else g.physics_advance
    assert g.block_info()["launches"] == 0
    for cap in (1, 2, 3, 13):
        nt = step(86400.0, nt_cap=cap)
        nt = min(int(np.max(nt[0] if g.ensemble else nt)), cap)
        assert g.block_info()["launches"] == launches(form, part, nt), cap
    g.close()


@pytest.mark.gpu
def test_steps_left_to_the_phase_kernels():
    g, st, ro = block_forms.model("cut_lev_dam", "fp64")
    g.set_state(st)
    g.set_runoff(ro)

    def used(adv=lambda: g.physics_advance(86400.0, nt_cap=6)):
        adv()
        return g.block_info()["launches"]
    assert used() == 2
    assert used(lambda: g.physics_advance_noalloc(3600.0)) == 0
    g.set_tune(graph=1)
    assert used() == 0
    g.set_tune(graph=0, fused=1)
    assert used() == 0
    g.set_tune(fused=0)
    g.kernel_times(True)
    assert used() == 0
    g.kernel_times(False)
    g.set_state(dict(daminf=np.ones(g.map.n)))
    assert used() == 0
    g.set_state(dict(daminf=np.zeros(g.map.n)))
    for switch in (g.set_kinematic, g.set_slopemix):
        switch(True)
        assert used() == 0
        switch(False)
    assert used() == 2
    g.close()


# the lines of the rule: (cells or domains, members, substeps a launch needs in FP64 and
# in the mixed form); steps of nt substeps of an open partition take two launches per
# 2*kmax of them
@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("sizes, members, least", [
    (600000, 1, (1, 1)), (900000, 1, (1.5, 1.5)), ([60000] * 2, 2, (1, 1)), ([60000] * 2, 4, (1.5, 1.5)),
    ([9000], 8, (1.5, 1.5)), ([60000], 8, (2, 2)), ([9000], 16, (2.5, 2.5)), ([30000], 16, (3.5, 3.9)),
    ([900] * 10, 8, (2, 2)), ([900] * 10, 16, (3, 3))])
def test_short_steps_stay_on_the_phase_kernels(sizes, members, least, prec):
    build = block_forms.regional if members == 1 else block_forms.ensemble
    g, st, ro = build(sizes, 0.0, 0, prec) if members == 1 else build(sizes, members, 0.0, 0, prec)
    _, kmax, closed, _ = block_forms.partition(g)
    g.set_state(st)
    g.set_runoff(ro)
    step = g.ensemble_advance if g.ensemble else g.physics_advance
    for cap in (1, 2, 3, 4, 5, 6, 8, 9, 16):
        nt = step(86400.0, nt_cap=cap)
        nt = min(int(np.max(nt[0] if g.ensemble else nt)), cap)
        nl = 1 if closed else 2 * -(-nt // (2 * kmax))
        want = nl if nt >= (1 if closed else 2) and nt / nl >= least[prec == "mixed"] else 0
        assert g.block_info()["launches"] == want, cap
    g.close()
