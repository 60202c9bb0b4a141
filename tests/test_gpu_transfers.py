"""Arrays through the pinned chunks: what was set is read back in place, with arrays
below, across and above one chunk (262,144 values), members, both precisions and cell
orders; inference over several chunks of rows (16,384) equals that over each alone."""
import numpy as np
import pytest

from cmf import maps, synth
from cmf.model import CMFModel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["dfs", "nseq"])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("cells, members", [(300, 1), (300, 4), (9000, 1), (20000, 2), (140000, 1), (140000, 2)])
def test_state_round_trip(cells, members, prec, order, monkeypatch):
    monkeypatch.setenv("CMF_HIP_ORDER", order)
    net = synth.regional_networks([cells], 3, land_frac=0.9)[0]
    synth.add_bifurcations(net, max(10, net.ncells // 20), 5, 3)
    synth.add_levees(net, 0.2, 3)
    m = maps.build_map(net, maps.Options(lpthout=True, llevee=True))
    kw = dict(members=members, dom_cells=[m.n]) if members > 1 else {}
    g = CMFModel(m, prec, **kw)
    rng = np.random.default_rng(cells + members)
    lead = (members,) if members > 1 else ()
    st = {k: rng.uniform(0.0, 9.0, lead + (m.n,)) for k in ("rivsto", "fldsto", "levsto", "rivout_pre", "fldout_pre",
                                                            "rivdph_pre", "fldsto_pre")}
    st["pthflw_pre"] = rng.uniform(-1.0, 1.0, lead + (m.npthlev, m.npth))
    st["rivout"], st["fldout"], st["pthflw"] = st["rivout_pre"], st["fldout_pre"], st["pthflw_pre"]
    g.set_state(st)
    for names in (list(st), ["levsto"], ["pthflw_pre", "rivsto"]):
        got = g.get_state(names)
        for k in names:
            want = st[k] if prec == "fp64" or k.endswith("sto") else st[k].astype(np.float32)
            assert np.array_equal(got[k], want.astype(np.float64)), k
    g.close()


@pytest.mark.parametrize("rows", [16384, 16385, 32769, 300001])
def test_inference_chunks(rows):
    from cmf.surrogate import MLP, N_IN, init_params
    rng = np.random.default_rng(rows)
    x = rng.normal(size=(rows, N_IN)).astype(np.float32)
    g = MLP(max_batch=1024)
    g.set_params(init_params(7))
    y = g.forward(x)
    for r0 in {0, 16384, rows // 16384 * 16384, rows - 5}:
        part = g.forward(x[r0:r0 + 16384])
        # tiles of other heights sum a row in the same order
        assert np.array_equal(part, y[r0:r0 + 16384]), r0
    g.close()
