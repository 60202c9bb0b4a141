"""build_block_plan refuses a shape as soon as it is known not to do (on the CPU, over
the stand-in of the HIP runtime): the partitions are those that building every shape in
full gave, and a closed one holds whole groups of basins joined by paths."""
import hip_stub

CODE = """
import numpy as np
from cmf import maps, synth
from cmf.model import CMFModel

def partition(cells, per=0, lev=0.0):
    net = synth.regional_networks([cells], 3, land_frac=0.9)[0]
    if per:
        synth.add_bifurcations(net, net.ncells // per, 5, 3)
    if lev:
        synth.add_levees(net, lev, 3, hmin=0.5, hmax=3.0, fmin=0.05, fmax=0.5)
    m = maps.build_map(net, maps.Options(lpthout=per > 0, llevee=lev > 0))
    group = maps.basin_of(m)
    if per:                                              # basins joined by paths
        to = np.arange(group.max() + 1)
        for u, d in zip(m.pth_upst, m.pth_down):
            if u >= 0 and d >= 0:
                a, b = to[group[u]], to[group[d]]
                to[to == b] = a
        group = to[group]
    g = CMFModel(m)
    i = g.block_info()
    g.close()
    return [int(np.bincount(group).max()), i["cells"], i["substeps"], i["blocks"], i["closed"]]
result([partition(*a) for a in %r])
"""
# cells, cells per path, levees: the largest group, cells and substeps of a block, blocks, closed
WANT = {(300,): (63, 256, 2, 1, 1), (700,): (155, 256, 2, 3, 1), (1400,): (314, 512, 6, 3, 1),
        (3000,): (359, 512, 6, 6, 1), (15000,): (1547, 512, 6, 47, 0), (200, 40): (49, 256, 1, 1, 1),
        (300, 12): (112, 256, 1, 1, 1), (600, 12): (367, 512, 6, 2, 1), (900, 12, 0.2): (267, 512, 6, 2, 1),
        (3000, 100): (360, 512, 6, 7, 0), (15000, 15): (6186, 512, 4, 51, 0)}


def test_partitions_and_groups(tmp_path):
    got = hip_stub.run(tmp_path, CODE % (list(WANT),))
    for (key, want), have in zip(WANT.items(), got):
        assert tuple(have) == want, key
        assert not (have[4] and have[0] > have[1])
