"""Energy and gradient of ligands of two atom slots (65-128 atoms) against the oracle (FP64): their second slot is
scored for four, two or one pair diagonals at once by how many atoms it holds. Both sides of each such edge,
odd and even atom counts.

Tolerances as in test_gpu_parity: energies and gradients within 1e-4 relative (floor 1.0), no box penalty."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natom", [65, 66, 79, 80, 81, 82, 95, 96, 97, 111, 127, 128])
def test_two_slot_ligands(gpu, receptor, box, natom):
    import torch
    from unidock_engine import synthetic as S
    lig = S.make_ligand(7400 + natom, natom, 7).ligand
    print(f"two slots: {natom} atoms", flush=True)
    scene, ls, n = gpu.Scene(receptor, box), gpu.LigSet([lig]), 12
    pv = S.random_pose_vectors(n, lig.ntors, box, seed=natom)
    pv[:, 0:3] = np.asarray(S.POCKET_CENTER, np.float32) + np.random.default_rng(natom).uniform(-6, 6, (n, 3))
    pv_d = torch.as_tensor(pv, device="cuda")
    e, g = torch.zeros(n, device="cuda"), torch.zeros((n, 6 + lig.ntors), device="cuda")
    gpu.check(gpu.lib().ud2_score_posevecs(scene.h, ls.h, 0, n, C.c_void_p(pv_d.data_ptr()), C.c_void_p(e.data_ptr()),
                                           C.c_void_p(g.data_ptr()), gpu.MODE_DIRECT, 10.0, 0.0, gpu.stream_ptr()),
              "ud2_score_posevecs")
    torch.cuda.synchronize()
    er, gr, _ = O.score_posevecs(O.Topo(lig), O.Scene(receptor, box), pv, v_cap=10.0, slope=0.0)
    assert (np.abs(e.cpu().numpy() - er) / np.maximum(np.abs(er), 1.0)).max() < 1e-4
    assert (np.abs(g.cpu().numpy() - gr) / np.maximum(np.abs(gr).max(axis=1, keepdims=True), 1.0)).max() < 1e-4
