"""Allocations of the surrogate network (on the CPU, over the stand-in of the HIP
runtime): cmf_mlp_create makes them all or fails whole, so no later call meets a handle
with some of its buffers, or pays for buffers in its first pass. Inference can do
without its pinned slot and the device's side of it."""
import pytest

import hip_stub

CODE = """
import numpy as np
from cmf.surrogate import MLP, SurrogateError
kw = dict(n_in=%d, hidden=%d, n_out=%d, max_batch=9000)
x, t = np.zeros((64, kw["n_in"]), np.float32), np.zeros((64, kw["n_out"]), np.float32)
out = dict(create=[], refused=[], left=[])
g = MLP(**kw)
ndev, npin = stub.stub_device_allocs(), stub.stub_pinned_allocs()
stub.stub_fail(0, 0, 0, 0)
g.grad(x, t)
g.grad(np.repeat(x, 140, 0), np.repeat(t, 140, 0))           # split weight gradients
g.forward(x)
out["first calls"] = [stub.stub_device_allocs(), stub.stub_pinned_allocs()]
g.close()
for k in range(1, ndev + npin + 1):
    if k <= ndev:
        stub.stub_fail(k, k, 0, 0)
    else:
        stub.stub_fail(0, 0, k - ndev, k - ndev)
    try:
        g = MLP(**kw)
        g.grad(x, t)
        g.forward(np.repeat(x, 300, 0))
        g.close()
        out["refused"].append(False)
    except SurrogateError:
        out["refused"].append(True)
    out["left"].append(stub.stub_live())
result(out)
"""


@pytest.mark.parametrize("n_in, hidden, n_out", [(24, 256, 2), (24, 64, 2)])
def test_create_allocates_all(tmp_path, n_in, hidden, n_out):
    got = hip_stub.run(tmp_path, CODE % (n_in, hidden, n_out))
    assert got["first calls"] == [0, 0]
    assert len(got["refused"]) > 15
    assert got["refused"].count(False) == (2 if hidden == 256 else 0)
    assert not any(got["left"])
