"""Models for which some memory cannot be had (on the CPU, over the stand-in of the HIP
runtime): the partition is optional, pinned memory beyond that of cmf_hip_create is
too, and nothing is left behind. The slots of a state's transfer come with the map."""
import pytest

import hip_stub

CODE = """
import block_forms
from cmf.model import CMFError
out = dict(made=[], left=[], pinned=None)
make = lambda: block_forms.model(%r, "fp64")
g, st, ro = make()                                       # (builders use the stand-in once)
stub.stub_fail(0, 0, 0, 0)
g.get_state()
out["first get"] = [stub.stub_device_allocs(), stub.stub_pinned_allocs()]
g.close()
stub.stub_fail(0, 0, 0, 0)
make()[0].close()
for k in range(1, stub.stub_device_allocs() + 1):
    stub.stub_fail(k, k, 0, 0)
    try:
        g = make()[0]
        out["made"].append(g.block_info()["cells"] > 0)
        g.close()
    except CMFError:
        out["made"].append(None)
    out["left"].append(stub.stub_live())
stub.stub_fail(0, 0, 4, 10**9)                           # only the three of cmf_hip_create
g = make()[0]
g.set_state(st)
g.set_runoff(ro)
g.get_state()
g.diag_avemax_output(3600.0)
g.get_output()
g.close()
out["pinned"] = [stub.stub_pinned_allocs() > 4, stub.stub_live()]
result(out)
"""


@pytest.mark.parametrize("form", ["plain", "cut_lev_dam", "paths_all"])
def test_partition_is_optional(tmp_path, form):
    got = hip_stub.run(tmp_path, CODE % form)
    made = got["made"]
    first = made.index(False)                            # the first allocation of the partition
    assert made == [None] * first + [False] * (len(made) - first)
    assert first > 60 and len(made) - first >= (6 if form == "plain" else 7)
    assert not any(got["left"])
    assert got["first get"] == [0, 0]
    assert got["pinned"] == [True, 0]
