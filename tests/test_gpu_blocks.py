"""Substeps in block launches (k_block) against the three-phase kernels (graph
replay selects them): the same statements on the same inputs, so the state must be
the same bits; the budget sums, compensated in another order, agree to a few ulps."""
import numpy as np
import pytest

from cases import STATE_KEYS, prepare, rel_err, upload_keys
from cmf import maps, synth
from cmf.model import CMFModel

pytestmark = pytest.mark.gpu


def big_basins(cells, lev, dam, seed=3):
    """One regional domain with basins larger than a block."""
    net = synth.regional_networks([cells], seed, land_frac=0.9)[0]
    if lev:
        synth.add_levees(net, lev, seed, hmin=0.5, hmax=3.0, fmin=0.05, fmax=0.5)
    if dam:
        synth.add_dams(net, max(3, net.ncells // dam), seed)
    m = maps.build_map(net, maps.Options(llevee=lev > 0, ldamout=dam > 0))
    st = maps.cold_start(m)
    st["rivsto"] = m.rivstomax * np.random.default_rng(seed).uniform(0.3, 1.6, m.n)
    if dam:
        maps.init_dams(m, net, st)
    ro = m.vec(synth.make_runoff(net, 1, seed, mean_mm_day=20.0)[0])
    return m, st, ro


def compare(m, st, runoff, prec, caps, dt=86400.0, prep=None):
    g = {k: CMFModel(m, prec) for k in ("blocks", "phases")}
    g["phases"].set_tune(graph=1)
    for x in g.values():
        x.set_state(st)
        if prep:
            prep(x)
        x.set_runoff(runoff)
    names = [k for k in STATE_KEYS + ["levsto", "levdph", "damsto", "daminf", "daminf_avg"] if g["blocks"]._available(k)]
    for cap in caps:
        out = {k: x.physics_advance(dt, nt_cap=cap, budget=True) for k, x in g.items()}
        assert out["blocks"][0] == out["phases"][0]
        for k in range(11):
            assert rel_err(out["blocks"][1][:, k], out["phases"][1][:, k]) < 1e-14, k
        a, b = (x.get_state(names) for x in g.values())
        for k in names:
            assert np.array_equal(a[k], b[k]), (k, cap, rel_err(a[k], b[k]))
    for x in g.values():
        x.close()


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("case", ["plain", "lev", "dam", "levwet", "damh22"])
def test_whole_basins(case, prec):
    m, net, st, rvec = prepare(case, 1)
    compare(m, upload_keys(st), rvec[0], prec, [0, 1, 97])


# launches of a cut network come in pairs of at most kmax substeps each: 1 substep
# (the three-phase kernels), below, at and above one pair, many, and all of them
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("lev, dam", [(0.0, 0), (0.2, 60), (0.6, 0), (0.0, 25)])
def test_cut_basins(lev, dam, prec):
    m, st, ro = big_basins(9000, lev, dam)
    assert np.bincount(maps.basin_of(m)).max() > 1024
    compare(m, st, ro, prec, [1, 2, 3, 11, 12, 13, 0])


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("cells", [140000, 300000])
def test_larger_blocks(cells, prec):
    m, st, ro = big_basins(cells, 0.03, 400)
    compare(m, st, ro, prec, [9, 21])


def test_restart_and_host_daminf():
    """The first substep's RIVVEL from a restart's D2RIVOUT; DAMINF set outside the
    dam cells takes the three-phase path; both on one handle."""
    m, st, ro = big_basins(9000, 0.2, 60)

    def restart(x):
        x.physics_fldstg()
        x.calc_outpre()
    compare(m, st, ro, "fp64", [5, 14], prep=restart)
    st2 = dict(st, daminf=np.random.default_rng(1).uniform(0.0, 50.0, m.n))
    compare(m, st2, ro, "fp64", [5], prep=restart)
    compare(m, st2, ro, "fp64", [5], prep=lambda x: x.set_state(dict(daminf=np.zeros(m.n))))


def test_upstream_inflow():
    m, st, ro = big_basins(9000, 0.0, 0)
    u = np.random.default_rng(2).uniform(0.0, 5.0, m.n)
    compare(m, st, ro, "fp64", [14], prep=lambda x: x.set_upsinf(u))


# every instance its own number of substeps, some of them one; domains of blocks cut
# from basins and of whole ones (1200 cells), a small and a large chip share
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("sizes, members, lev, dam", [
    ([9000, 1200, 5000], 1, 0.2, 60), ([9000, 1200, 5000], 2, 0.0, 0), ([9000, 1200], 4, 0.3, 0),
    ([1200, 700], 16, 0.0, 40), ([1500, 900], 2, 0.0, 0), ([60000, 40000], 4, 0.0, 0), ([6000], 32, 0.0, 0)])
def test_ensemble(sizes, members, lev, dam, prec):
    doms = []
    for d, net in enumerate(synth.regional_networks(sizes, 11, land_frac=0.9)):
        if lev:
            synth.add_levees(net, lev, d, hmin=0.5, hmax=3.0, fmin=0.05, fmax=0.5)
        if dam:
            synth.add_dams(net, max(3, net.ncells // dam), d)
        m = maps.build_map(net, maps.Options(llevee=lev > 0, ldamout=dam > 0, pdstmth=4.0e5))
        st = maps.cold_start(m)
        st["rivsto"] = m.rivstomax * np.random.default_rng(d).uniform(0.0, 0.4 + d, m.n)
        if dam:
            maps.init_dams(m, net, st)
        doms.append((m, upload_keys(st), m.vec(synth.make_runoff(net, 1, d, mean_mm_day=20.0)[0])))
    cm, dom_cells = maps.concat_maps([d[0] for d in doms])
    init = {k: np.stack([np.concatenate([d[1][k] for d in doms])] * members) for k in doms[0][1]}
    level = np.random.default_rng(4).uniform(0.02, 1.0, size=(members, 1))
    init["rivsto"] = init["rivsto"] * level
    ro = np.concatenate([d[2] for d in doms])
    g = {k: CMFModel(cm, prec, members=members, dom_cells=dom_cells) for k in ("blocks", "phases")}
    g["phases"].set_tune(graph=1)
    fac = np.exp(np.random.default_rng(5).normal(0.0, 1.5, size=len(sizes) * members))
    for x in g.values():
        x.set_state(init)
        x.set_runoff_scaled(ro, fac)
    names = [k for k in STATE_KEYS + ["levsto", "levdph", "damsto", "daminf", "daminf_avg"] if g["blocks"]._available(k)]
    spread = set()
    for dt, cap in ((900.0, 0), (3600.0, 0), (86400.0, 9), (86400.0, 26)):
        nt = {k: x.ensemble_advance(dt, nt_cap=cap)[0] for k, x in g.items()}
        assert np.array_equal(nt["blocks"], nt["phases"])
        spread |= set(np.minimum(nt["blocks"], cap or 10**6).tolist())
        a, b = (x.get_state(names) for x in g.values())
        for k in names:
            assert np.array_equal(a[k], b[k]), (k, dt, cap, rel_err(a[k], b[k]))
    print("substeps", sorted(spread), flush=True)
    for x in g.values():
        x.close()


PATH_KEYS = ["pthflw", "pthflwsum", "pthflw_avg", "pthflwsum_avg", "pthout_avg", "pthout"]


def compare_paths(m, st, runoff, prec, caps, dt=86400.0):
    g = {k: CMFModel(m, prec) for k in ("blocks", "phases")}
    g["phases"].set_tune(graph=1)
    for x in g.values():
        x.set_state(st)
        x.set_runoff(runoff)
    names = STATE_KEYS + PATH_KEYS + ["levsto", "levdph", "damsto", "daminf", "daminf_avg"]
    names = [k for k in dict.fromkeys(names) if g["blocks"]._available(k)]
    flows = 0.0
    for cap in caps:
        out = {k: x.physics_advance(dt, nt_cap=cap, budget=True) for k, x in g.items()}
        assert out["blocks"][0] == out["phases"][0]
        for k in range(11):
            assert rel_err(out["blocks"][1][:, k], out["phases"][1][:, k]) < 1e-14, k
        a, b = (x.get_state(names) for x in g.values())
        for k in names:
            assert np.array_equal(a[k], b[k]), (k, cap, rel_err(a[k], b[k]))
        flows = max(flows, np.abs(a["pthflwsum"]).max())
    for x in g.values():
        x.close()
    assert flows > 0.0                                     # the paths carry water


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("case", ["pth", "levpth", "all", "allwet"])
def test_paths_small(case, prec):
    m, net, st, rvec = prepare(case, 1)
    compare_paths(m, upload_keys(st), rvec[0], prec, [0, 1, 2, 31])


# blocks grown along the paths, with paths that leave them, cells with several paths,
# masked cells (dams) and paths with an end outside the network; one level to ten
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("cells, per, levels, lev, dam, dead", [
    (9000, 12, 5, 0.0, 0, 0), (9000, 8, 5, 0.3, 60, 40), (9000, 20, 1, 0.2, 0, 0), (5000, 15, 10, 0.0, 25, 7),
    (140000, 12, 5, 0.0, 0, 0)])
def test_paths_cut(cells, per, levels, lev, dam, dead, prec):
    net = synth.regional_networks([cells], 3, land_frac=0.9)[0]
    synth.add_bifurcations(net, net.ncells // per, levels, 3)
    if lev:
        synth.add_levees(net, lev, 3, hmin=0.5, hmax=3.0, fmin=0.05, fmax=0.5)
    if dam:
        synth.add_dams(net, max(3, net.ncells // dam), 3)
    m = maps.build_map(net, maps.Options(lpthout=True, llevee=lev > 0, ldamout=dam > 0))
    st = maps.cold_start(m)
    st["rivsto"] = m.rivstomax * np.random.default_rng(3).uniform(0.3, 1.9, m.n)
    if dam:
        maps.init_dams(m, net, st)
    if dead:
        m.pth_upst[::dead] = -1
        m.pth_down[1::dead] = -1
        st["pthflw"][:, ::dead] = 3.0
    ro = m.vec(synth.make_runoff(net, 1, 3, mean_mm_day=20.0)[0])
    compare_paths(m, upload_keys(st), ro, prec, [1, 2, 3, 11, 12, 13] if cells < 100000 else [9])
