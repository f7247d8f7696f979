"""Pose gradients by number of torsions against the oracle (FP64): the torques about the torsion axes are staged in
chunks (24 torsions with one atom per lane, 32 with two, 48 with three and four) and summed four at a time, two
and two. One to four torsions, and the edges of a chunk and one past it.

Tolerances as in test_gpu_parity: energies and gradients within 1e-4 relative (floor 1.0), no box penalty."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natom,ntors", [(9, 1), (10, 2), (14, 3), (20, 4), (60, 24), (60, 25), (64, 27), (70, 32),
                                         (110, 33), (128, 35), (190, 49), (250, 50)])
def test_gradient_by_torsion_count(gpu, receptor, box, natom, ntors):
    import torch
    from unidock_engine import synthetic as S
    lig = S.make_ligand(7700 + natom + ntors, natom, ntors).ligand
    assert lig.ntors == ntors
    print(f"torsion counts: {natom} atoms, {ntors} torsions", flush=True)
    scene, ls, n = gpu.Scene(receptor, box), gpu.LigSet([lig]), 12
    pv = S.random_pose_vectors(n, ntors, box, seed=natom)
    pv[:, 0:3] = np.asarray(S.POCKET_CENTER, np.float32) + np.random.default_rng(ntors).uniform(-6, 6, (n, 3))
    pv_d = torch.as_tensor(pv, device="cuda")
    e, g = torch.zeros(n, device="cuda"), torch.zeros((n, 6 + ntors), device="cuda")
    gpu.check(gpu.lib().ud2_score_posevecs(scene.h, ls.h, 0, n, C.c_void_p(pv_d.data_ptr()), C.c_void_p(e.data_ptr()),
                                           C.c_void_p(g.data_ptr()), gpu.MODE_DIRECT, 10.0, 0.0, gpu.stream_ptr()),
              "ud2_score_posevecs")
    torch.cuda.synchronize()
    er, gr, _ = O.score_posevecs(O.Topo(lig), O.Scene(receptor, box), pv, v_cap=10.0, slope=0.0)
    assert (np.abs(e.cpu().numpy() - er) / np.maximum(np.abs(er), 1.0)).max() < 1e-4
    assert (np.abs(g.cpu().numpy() - gr) / np.maximum(np.abs(gr).max(axis=1, keepdims=True), 1.0)).max() < 1e-4
