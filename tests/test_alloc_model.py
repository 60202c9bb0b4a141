"""Models for which some memory cannot be had (on the CPU, over the stand-in of the HIP
runtime): the partition is optional, and nothing is left behind."""
import pytest

import hip_stub

CODE = """
import block_forms
from cmf.model import CMFError
out = dict(made=[], left=[])
make = lambda: block_forms.model(%r, "fp64")
g, st, ro = make()                                       # (builders use the stand-in once)
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
