"""A refused request for grid maps (doubled or unknown probe types, a spacing or a grid of fewer than two points) leaves the
scene's maps as they were: the same grid, maps and energies as before, for every ligand atom type that they hold."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PROBES = [2, 3, 4, 5, 6, 10, 11, 15]


def test_refused_maps_change_nothing(gpu, receptor, box):
    import torch
    from unidock_engine import synthetic as S
    lig = S.make_ligand(9300, 30, 4).ligand
    ls = gpu.LigSet([lig])
    scene = gpu.Scene(receptor, box)
    scene.build_grids(0.75, PROBES)
    pv = torch.from_numpy(S.random_pose_vectors(64, lig.ntors, box, seed=4)).cuda()

    def state():
        e, g = torch.zeros(64, device="cuda"), torch.zeros((64, 6 + lig.ntors), device="cuda")
        gpu.check(gpu.lib().ud2_score_posevecs(scene.h, ls.h, 0, 64, C.c_void_p(pv.data_ptr()), C.c_void_p(e.data_ptr()),
                                               C.c_void_p(g.data_ptr()), gpu.MODE_GRID, 10.0, 1e6, gpu.stream_ptr()))
        torch.cuda.synchronize()
        n, org, sp, nt = scene.grid_info()
        return e.cpu().numpy(), g.cpu().numpy(), scene.download_maps(), n, org, np.float32(sp), np.int32(nt)

    before = state()
    n, org, _, _ = scene.grid_info()
    maps = np.zeros((1, 4, 4, 4), np.float32)
    refused = [lambda: scene.build_grids(0.75, [2, 3, 2]), lambda: scene.build_grids(0.75, [2, 0]),
               lambda: scene.build_grids(0.75, [2, 99]), lambda: scene.build_grids(0.75, []),
               lambda: scene.build_grids(0.0, PROBES), lambda: scene.build_grids(500.0, PROBES),
               lambda: scene.set_grids([4, 4, 1], org, 1.0, [2], maps), lambda: scene.set_grids([4, 4, 4], org, 1.0, [3, 3], maps),
               lambda: scene.set_grids([4, 4, 4], org, -1.0, [3], maps)]
    for k, call in enumerate(refused):
        print(f"refused maps {k}", flush=True)
        with pytest.raises(gpu.Ud2Error):
            call()
        n2, org2, _, nt2 = scene.grid_info()
        assert np.array_equal(n2, n) and np.array_equal(org2, org) and nt2 == len(PROBES), k
        for a, b in zip(before, state()):
            assert np.array_equal(a, b), k
