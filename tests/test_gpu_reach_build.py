"""The reach lists' build where it changes shape: receptors around the chunks of 1,024 atoms that it takes at a time,
cells that are no whole bricks, and a receptor so dense that the cells get coarser. Direct energies and gradients
against the oracle's sum over the whole receptor (FP64); tolerance as in test_gpu_reach."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rec,size", [(1023, 30.0), (1024, 17.0), (1025, 5.0), (2049, 23.0), (24000, 30.0)])
def test_lists_at_chunk_and_brick_edges(gpu, receptor, n_rec, size):
    import torch
    from unidock_engine import synthetic as S
    from unidock_engine import topology as T
    print(f"reach build: {n_rec} receptor atoms, box {size}", flush=True)
    copies = -(-n_rec // len(receptor.types))
    rng = np.random.default_rng(n_rec)
    # copies of the shell shifted by a fraction of an angstrom each
    xyz = np.concatenate([receptor.xyz + rng.uniform(-0.8, 0.8, 3) for _ in range(copies)])[:n_rec].astype(np.float32)
    rec = dataclasses.replace(receptor, xyz=xyz, types=np.tile(receptor.types, copies)[:n_rec].copy())
    box = T.Box.from_center_size(S.POCKET_CENTER, (size, size, size))
    lig = S.make_ligand(8310, 21, 3).ligand
    ls = gpu.LigSet([lig])
    scene = gpu.Scene(rec, box)
    n = 64
    pv = S.random_pose_vectors(n, lig.ntors, T.Box.from_center_size(S.POCKET_CENTER, (24.0,) * 3), seed=6)
    pv_d = torch.as_tensor(pv, device="cuda")
    e = torch.zeros(n, device="cuda")
    g = torch.zeros((n, 6 + lig.ntors), device="cuda")
    gpu.check(gpu.lib().ud2_score_posevecs(scene.h, ls.h, 0, n, C.c_void_p(pv_d.data_ptr()), C.c_void_p(e.data_ptr()),
                                           C.c_void_p(g.data_ptr()), gpu.MODE_DIRECT, 1e30, 0.0, gpu.stream_ptr()))
    torch.cuda.synchronize()
    er, gr, _ = O.score_posevecs(O.Topo(lig), O.Scene(rec, box), pv, v_cap=1e30, slope=0.0)
    err = np.abs(e.cpu().numpy() - er) / np.maximum(np.abs(er), 1.0)
    assert err.max() < 1e-4, err.max()
    gs = np.maximum(np.abs(gr).max(axis=1, keepdims=True), 1.0)
    assert (np.abs(g.cpu().numpy() - gr) / gs).max() < 1e-4
