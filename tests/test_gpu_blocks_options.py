"""Block launches against the phase kernels, to the bit, over the options and inputs that
test_gpu_blocks.py leaves at their defaults: no floodplain flow, no floodplains, one to
sixteen floodplain layers (some of them in LDS), other parameters, a fixed step, a dry
model, negative and undefined runoff; two models stepped by two threads at once."""
import threading

import numpy as np
import pytest

from cases import STATE_KEYS
from cmf import maps, synth
from cmf.model import CMFModel

pytestmark = pytest.mark.gpu
NAMES = STATE_KEYS + ["levsto", "levdph", "damsto", "daminf", "daminf_avg", "pthflw", "pthflwsum", "pthflw_avg",
                      "pthflwsum_avg"]


def layers(net, n):
    h = net.fldhgt
    if n <= h.shape[0]:
        net.fldhgt = np.ascontiguousarray(h[:n])
    else:
        more = [h[-1] + np.float32(k) * (h[-1] - h[-2] + np.float32(1.0)) for k in range(1, n - h.shape[0] + 1)]
        net.fldhgt = np.concatenate([h, np.stack(more)]).astype(h.dtype)


def model(cells, lev, dam, per, nlfp=10, wet=1.6, **opts):
    net = synth.regional_networks([cells], 3, land_frac=0.9)[0]
    if nlfp != 10:
        layers(net, nlfp)
    if per:
        synth.add_bifurcations(net, net.ncells // per, 5, 3)
    if lev:
        synth.add_levees(net, lev, 3, hmin=0.5, hmax=3.0, fmin=0.05, fmax=0.5)
    if dam:
        synth.add_dams(net, max(3, net.ncells // dam), 3)
    m = maps.build_map(net, maps.Options(lpthout=per > 0, llevee=lev > 0, ldamout=dam > 0, **opts))
    assert m.nlfp == nlfp
    st = maps.cold_start(m)
    st["rivsto"] = m.rivstomax.clip(max=1e9) * np.random.default_rng(3).uniform(0.0, wet, m.n)
    if dam:
        maps.init_dams(m, net, st)
    return m, st, m.vec(synth.make_runoff(net, 1, 3, mean_mm_day=20.0)[0])


def run(m, st, ro, prec, graph, caps, dt=86400.0):
    g = CMFModel(m, prec)
    g.set_tune(graph=graph)
    g.set_state(st)
    g.set_runoff(ro)
    out = []
    for cap in caps:
        nt, glb = g.physics_advance(dt, nt_cap=cap, budget=True)
        out.append((nt, g.block_info()["launches"], g.get_state([k for k in NAMES if g._available(k)])))
    g.close()
    return out


def compare(m, st, ro, prec, caps=(5, 14), dt=86400.0):
    a, b = run(m, st, ro, prec, 0, caps, dt), run(m, st, ro, prec, 1, caps, dt)
    for (nt, launches, x), (nt1, none, y) in zip(a, b):
        assert nt == nt1 and launches > 0 and none == 0
        for k in x:
            assert np.array_equal(x[k], y[k], equal_nan=True), k
    return a


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("lev, dam, per", [(0.0, 0, 0), (0.3, 60, 0), (0.3, 60, 10)])
@pytest.mark.parametrize("opts", [
    dict(lfldout=False), dict(lfplain=False), dict(pmanfld=0.03, pgrv=3.7, pcadp=0.4, pdstmth=500.0), dict(nlfp=1),
    dict(nlfp=4), dict(nlfp=8), dict(nlfp=16)], ids=lambda o: "-".join(f"{k}{v}" for k, v in o.items()))
def test_options(opts, lev, dam, per, prec):
    compare(*model(9000, lev, dam, per, **opts), prec)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("lev, dam, per", [(0.0, 0, 0), (0.3, 60, 0), (0.2, 0, 12)])
def test_fixed_step(lev, dam, per, prec):
    """One substep of DT: whole basins take it in a launch."""
    compare(*model(500, lev, dam, per, ladpstp=False), prec, caps=(0, 0, 0), dt=600.0)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("inputs", ["dry", "negative", "undefined"])
def test_inputs(inputs, prec):
    m, st, ro = model(9000, 0.3, 60, 10, wet=0.0 if inputs == "dry" else 1.6)
    if inputs == "dry":
        ro = 0.0 * ro
    elif inputs == "negative":
        ro = -ro
    else:
        ro = ro.copy()
        ro[[7, 2500]] = np.nan, np.inf
    # an infinite depth leaves no CFL bound for another step
    x = compare(m, st, ro, prec, (14,) if inputs == "undefined" else (5, 14))[-1][2]
    if inputs == "undefined":
        assert not np.isfinite(x["rivsto"]).all() and np.isfinite(x["rivsto"]).any()


def test_two_threads():
    models = [model(9000, 0.3, 60, 10), model(9000, 0.0, 0, 0)]
    want = [run(*m, "fp64", 1, (5, 14, 20)) for m in models]
    got = [None, None]

    def step(k):
        got[k] = [run(*models[k], "fp64", 0, (5, 14, 20)) for _ in range(3)]
    th = [threading.Thread(target=step, args=(k,)) for k in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for k in range(2):
        for r in got[k]:
            for (_, launches, x), (_, _, y) in zip(r, want[k]):
                assert launches > 0
                for name in x:
                    assert np.array_equal(x[name], y[name]), name
