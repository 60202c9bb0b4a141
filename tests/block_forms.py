"""The models of test_gpu_blocks.py with the partition that each of them has to get:
(cells per block, substeps per launch, closed, along paths), None for none."""
import numpy as np

from cases import prepare, upload_keys
from cmf import maps, synth
from cmf.model import CMFModel


def whole(case, prec):
    m, net, st, rvec = prepare(case, 1)
    return CMFModel(m, prec), upload_keys(st), rvec[0]


def regional(cells, lev, dam, prec, per=0, levels=5, dead=0):
    net = synth.regional_networks([cells], 3, land_frac=0.9)[0]
    if per:
        synth.add_bifurcations(net, net.ncells // per, levels, 3)
    if lev:
        synth.add_levees(net, lev, 3, hmin=0.5, hmax=3.0, fmin=0.05, fmax=0.5)
    if dam:
        synth.add_dams(net, max(3, net.ncells // dam), 3)
    m = maps.build_map(net, maps.Options(lpthout=per > 0, llevee=lev > 0, ldamout=dam > 0))
    st = maps.cold_start(m)
    st["rivsto"] = m.rivstomax * np.random.default_rng(3).uniform(0.3, 1.6, m.n)
    if dam:
        maps.init_dams(m, net, st)
    if dead:
        m.pth_upst[::dead] = -1
        m.pth_down[1::dead] = -1
    return CMFModel(m, prec), upload_keys(st), m.vec(synth.make_runoff(net, 1, 3, mean_mm_day=20.0)[0])


def ensemble(sizes, members, lev, dam, prec):
    doms = []
    for d, net in enumerate(synth.regional_networks(sizes, 11, land_frac=0.9)):
        if lev:
            synth.add_levees(net, lev, d, hmin=0.5, hmax=3.0, fmin=0.05, fmax=0.5)
        if dam:
            synth.add_dams(net, max(3, net.ncells // dam), d)
        m = maps.build_map(net, maps.Options(llevee=lev > 0, ldamout=dam > 0, pdstmth=4.0e5))
        st = maps.cold_start(m)
        if dam:
            maps.init_dams(m, net, st)
        doms.append((m, upload_keys(st), m.vec(synth.make_runoff(net, 1, d, mean_mm_day=20.0)[0])))
    cm, dom_cells = maps.concat_maps([d[0] for d in doms])
    init = {k: np.stack([np.concatenate([d[1][k] for d in doms])] * members) for k in doms[0][1]}
    return (CMFModel(cm, prec, members=members, dom_cells=dom_cells), init,
            np.stack([np.concatenate([d[2] for d in doms])] * members))


# name: builder, its arguments, the partition in FP64, and in the mixed form where it
# is another one (blocks of 512 over many rounds)
FORMS = {k: (whole, (k,), p) for k, p in dict(
    plain=(256, 2, 1, 0), lev=(256, 2, 1, 0), dam=(256, 2, 1, 0), levwet=(256, 2, 1, 0), damh22=(512, 6, 1, 0),
    pth=(512, 6, 1, 1), levpth=(512, 6, 0, 1), all=(256, 1, 1, 1), allwet=(512, 6, 1, 1)).items()}
FORMS.update({
    "cut": (regional, (9000, 0.0, 0), (512, 6, 0, 0)),
    "cut_lev_dam": (regional, (9000, 0.2, 60), (512, 6, 0, 0)),
    "cut_many_lev": (regional, (9000, 0.6, 0), (512, 4, 0, 0)),
    "cut_many_dam": (regional, (9000, 0.0, 25), (1024, 4, 0, 0)),
    "one_round": (regional, (140000, 0.03, 400), (1024, 4, 0, 0)),
    "rounds": (regional, (300000, 0.03, 400), (1024, 5, 0, 0), (512, 3, 0, 0)),
    "ens_lev_dam": (ensemble, ([9000, 1200, 5000], 1, 0.2, 60), (512, 4, 0, 0)),
    "ens_2": (ensemble, ([9000, 1200, 5000], 2, 0.0, 0), (512, 6, 0, 0)),
    "ens_lev_4": (ensemble, ([9000, 1200], 4, 0.3, 0), (512, 6, 0, 0)),
    "ens_dam_16": (ensemble, ([1200, 700], 16, 0.0, 40), (512, 6, 1, 0)),
    "ens_whole": (ensemble, ([1500, 900], 2, 0.0, 0), (256, 2, 1, 0)),
    "ens_rounds": (ensemble, ([60000, 40000], 4, 0.0, 0), (512, 4, 0, 0)),
    "ens_32": (ensemble, ([6000], 32, 0.0, 0), None),
    "paths": (regional, (9000, 0.0, 0, 12), (512, 4, 0, 1)),
    "paths_all": (regional, (9000, 0.3, 60, 8, 5, 40), (512, 4, 0, 1)),
    "paths_one_level": (regional, (9000, 0.2, 0, 20, 1), (512, 4, 0, 1)),
    "paths_ten_levels": (regional, (5000, 0.0, 25, 15, 10, 7), (512, 2, 0, 1)),
    "paths_rounds": (regional, (140000, 0.0, 0, 12), (512, 3, 0, 1)),
})


def model(form, prec):
    """(handle, state, runoff) of a form."""
    build, args = FORMS[form][:2]
    if build is regional:
        args = args[:3] + (prec,) + args[3:]
        return build(*args)
    return build(*args, prec)


def wanted(form, prec):
    f = FORMS[form]
    return f[3] if prec == "mixed" and len(f) > 3 else f[2]


def partition(g):
    i = g.block_info()
    return (i["cells"], i["substeps"], i["closed"], i["paths"]) if i["cells"] else None
