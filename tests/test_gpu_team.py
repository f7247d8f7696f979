"""Searches whose chains run on a team of four waves each (launches of few chains) against the same search inside a
launch of many chains, one wave per chain: the same poses and energies, bit for bit. Ligand 0 is searched
alone and as the first of a set of copies large enough to leave the team's range; its random stream is keyed by
its index, so its chains are the same. One to two atoms per lane, rigid and flexible, both inter terms,
0 and more MC steps, constraint docking."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PROBES = [2, 3, 4, 5, 6, 10, 11, 15]


def _search(gpu, scene, ls, nchain, mode, mc_steps, opt_steps):
    import torch
    pb = gpu.PoseBuffers(ls, nchain)
    pb.init()
    stats = torch.zeros(4, dtype=torch.int64, device="cuda")
    prm = gpu.McParams(mc_steps=mc_steps, opt_steps=opt_steps, randomize=1, seed=77, mode=mode, lig_index_base=0,
                       stats_d=stats.data_ptr())
    gpu.check(gpu.lib().ud2_mc(scene.h, ls.h, pb.ref, C.byref(prm), gpu.stream_ptr()), "ud2_mc")
    torch.cuda.synchronize()
    lig = ls.ligands[0]
    n = nchain * lig.natom * 3
    return (pb.x[:n].cpu().numpy(), pb.c[:3 * nchain].cpu().numpy(), pb.rv[:3 * nchain].cpu().numpy(),
            pb.dihe[:nchain * lig.ntors].cpu().numpy(), pb.e[:nchain].cpu().numpy()), int(stats[0])


@pytest.mark.parametrize("mode", ["grid", "direct"])
@pytest.mark.parametrize("n,t,mc,opt,constraint", [(9, 0, 3, 9, False), (24, 5, 4, 20, False), (32, 14, 2, 12, False),
                                                   (47, 9, 3, 16, False), (64, 15, 2, 14, True), (65, 6, 2, 10, False),
                                                   (96, 12, 1, 8, False), (30, 4, 0, 8, False), (30, 4, 3, 0, False)])
def test_team_is_the_one_wave_search(gpu, receptor, box, mode, n, t, mc, opt, constraint):
    from unidock_engine import synthetic as S
    print(f"team search: {n} atoms, {t} torsions, {mc} x {opt}, {mode}", flush=True)
    scene = gpu.Scene(receptor, box)
    scene.build_grids(S.GRID_SPACING, PROBES)
    lig = S.make_ligand(8800 + n, n, t).ligand
    nchain, m = 8, gpu.MODE_GRID if mode == "grid" else gpu.MODE_DIRECT
    alone, ev1 = _search(gpu, scene, gpu.LigSet([lig], constraint=constraint), nchain, m, mc, opt)
    copies = 400 if mode == "grid" else 200  # 3,200 and 1,600 chains
    many, evn = _search(gpu, scene, gpu.LigSet([lig] * copies, constraint=constraint), nchain, m, mc, opt)
    for a, b in zip(alone, many):
        assert np.array_equal(a, b)
    assert ev1 > 0 or mc == 0
    # the evaluations counted do not depend on how a chain is run: a set of 8 copies, each a team's
    few, ev8 = _search(gpu, scene, gpu.LigSet([lig] * 8, constraint=constraint), nchain, m, mc, opt)
    for a, b in zip(alone, few):
        assert np.array_equal(a, b)
    assert abs(ev8 / 8 - evn / copies) <= 0.25 * evn / copies
