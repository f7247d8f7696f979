"""Selections of every length of the pose operations, over ligands of one to three atom slots in mixed order: short
ones travel with the kernel's arguments (up to 64 poses), longer ones are copied. Each pose's energy and gradient
have the bits of a long selection's, and a pose id out of range is refused at any length."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129])
def test_selection_lengths(gpu, receptor, box, n):
    import torch
    from unidock_engine import synthetic as S
    print(f"selection of {n} poses", flush=True)
    ligs = [S.make_ligand(8600 + k, k, 5).ligand for k in (20, 130, 45, 70)]
    scene, ls, nchain = gpu.Scene(receptor, box), gpu.LigSet(ligs), 40
    pb = gpu.PoseBuffers(ls, nchain)
    pb.init()

    def energies(sel):
        sel_d = torch.as_tensor(np.asarray(sel, np.int32), device="cuda")
        e, g = torch.zeros(len(sel), device="cuda"), torch.zeros((len(sel), 64), device="cuda")
        rc = gpu.lib().ud2_energy_grad(scene.h, ls.h, pb.ref, C.c_void_p(sel_d.data_ptr()), len(sel), gpu.MODE_DIRECT,
                                       10.0, 1e6, C.c_void_p(e.data_ptr()), C.c_void_p(g.data_ptr()),
                                       gpu.stream_ptr())
        torch.cuda.synchronize()
        return rc, e.cpu().numpy(), g.cpu().numpy()

    prm = gpu.McParams(mc_steps=0, opt_steps=0, randomize=1, seed=5, mode=gpu.MODE_DIRECT, lig_index_base=0)
    gpu.check(gpu.lib().ud2_mc(scene.h, ls.h, pb.ref, C.byref(prm), gpu.stream_ptr()), "ud2_mc")
    rc, e_all, g_all = energies(range(4 * nchain))
    assert rc == 0 and len(np.unique(e_all)) > 100
    sel = np.random.default_rng(n).permutation(4 * nchain)[:n]
    rc, e, g = energies(sel)
    assert rc == 0
    assert np.array_equal(e, e_all[sel]) and np.array_equal(g, g_all[sel])
    for bad in (-1, 4 * nchain):
        rc, e, g = energies(np.concatenate([sel[:-1], [bad]]))
        assert rc != 0 and not e.any() and not g.any()
