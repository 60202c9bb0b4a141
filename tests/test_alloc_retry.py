"""A call that allocates on first use and fails half way leaves nothing half made: the
same call makes the rest later, and others refuse until then (on the CPU, over the
stand-in of the HIP runtime)."""
import hip_stub

CODE = """
import numpy as np
import block_forms
from cmf.model import CMFError
from cmf.surrogate import MLP, SurrogateError
errors = (CMFError, SurrogateError)

def first_use(make, call, blocked=None):
    h = make()
    base = stub.stub_live()
    stub.stub_fail(0, 0, 0, 0)
    call(h)
    n, kept = stub.stub_device_allocs(), stub.stub_live() - base
    h.close()
    out = [n, kept, []]
    for k in range(1, n + 1):
        h = make()
        base = stub.stub_live()
        stub.stub_fail(k, k, 0, 0)
        try:
            call(h)
            out[2].append("no error")
            continue
        except errors:
            pass
        if blocked:
            launches = stub.stub_launches()
            try:
                blocked(h)
                out[2].append("not refused")
                continue
            except errors:
                assert stub.stub_launches() == launches
        call(h)
        out[2].append(stub.stub_live() - base)
        h.close()
    return out

x, t = np.zeros((80, 24), np.float32), np.zeros((80, 2), np.float32)
model = lambda: block_forms.model("paths_all", "fp64")[0]
ens = lambda: block_forms.model("ens_2", "fp64")[0]
result([first_use(model, lambda g: g.diag_avemax_output(60.0), lambda g: g.get_output()),
        first_use(model, lambda g: g.diag_reset_output(), lambda g: g.diag_getave_output()),
        first_use(ens, lambda g: g.set_runoff_scaled(np.ones(g.map.n), np.ones(g.ninst))),
        first_use(ens, lambda g: g.instance_storage()),
        first_use(lambda: MLP(max_batch=64),
                  lambda g: g._check(g.lib.cmf_mlp_set_data(g.h, x.ctypes.data, t.ctypes.data, 80)),
                  lambda g: g._check(g.lib.cmf_mlp_train(g.h, np.arange(64).ctypes.data, 64, 32, 1e-3, 0.9, 0.999, 1e-8, 0, None)))])
"""


def test_calls_after_a_failed_allocation(tmp_path):
    for n, kept, after in hip_stub.run(tmp_path, CODE):
        assert n >= 2 and after == [kept] * n
