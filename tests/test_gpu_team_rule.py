"""Searches on either side of the line between team and one-wave launches: ligands of one size, where it lies at 8 chains
per CU, and sets of a large ligand among small ones, where it lies at the work of as many chains of the large one. The
first ligand's chains have the same bits in all of them (its random stream is keyed by its index)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PROBES = [2, 3, 4, 5, 6, 10, 11, 15]


def _first(gpu, scene, ligs, nchain):
    import torch
    ls = gpu.LigSet(ligs)
    pb = gpu.PoseBuffers(ls, nchain)
    pb.init()
    prm = gpu.McParams(mc_steps=2, opt_steps=6, randomize=1, seed=31, mode=gpu.MODE_GRID, lig_index_base=0, stats_d=None)
    gpu.check(gpu.lib().ud2_mc(scene.h, ls.h, pb.ref, C.byref(prm), gpu.stream_ptr()), "ud2_mc")
    torch.cuda.synchronize()
    lig = ligs[0]
    return (pb.x[:nchain * lig.natom * 3].cpu().numpy(), pb.c[:3 * nchain].cpu().numpy(),
            pb.dihe[:nchain * lig.ntors].cpu().numpy(), pb.e[:nchain].cpu().numpy())


@pytest.mark.parametrize("others", ["same", "small"])
def test_either_side_of_the_line(gpu, receptor, box, others):
    import torch
    from unidock_engine import synthetic as S
    print(f"team rule: {others}", flush=True)
    scene = gpu.Scene(receptor, box)
    scene.build_grids(S.GRID_SPACING, PROBES)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    lig = S.make_ligand(8900, 41, 6).ligand
    other = lig if others == "same" else S.make_ligand(8901, 12, 2).ligand
    nchain = 16
    ref = _first(gpu, scene, [lig], nchain)
    for n in (8 * cus // nchain - 1, 8 * cus // nchain, 12 * cus // nchain, 12 * cus // nchain + 1):
        got = _first(gpu, scene, [lig] + [other] * (n - 1), nchain)
        for a, b in zip(ref, got):
            assert np.array_equal(a, b), n
