"""The direct receptor sum from the scene's reach lists against the oracle's sum over the whole receptor (FP64):
poses in the box, across the edge of the listed space and beyond it, receptors of none, one and around 64 atoms,
with an atom that is nowhere, in boxes that make fine and coarse cells.

Tolerance as in test_gpu_parity (1e-4 relative, floor 1.0): at slope 0 no box penalty enters."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rec,size,nowhere", [(0, 30.0, False), (1, 30.0, False), (63, 8.0, True), (65, 30.0, False),
                                                (2000, 30.0, True), (2000, 3.0, False), (2000, 400.0, False)])
def test_reach_lists_match_whole_receptor(gpu, receptor, n_rec, size, nowhere):
    import torch
    from unidock_engine import synthetic as S
    from unidock_engine import topology as T
    print(f"reach lists: {n_rec} receptor atoms, box {size}, an atom nowhere: {nowhere}", flush=True)
    rec = dataclasses.replace(receptor, xyz=receptor.xyz[:n_rec].copy(), types=receptor.types[:n_rec].copy())
    ref_rec = rec
    if nowhere:
        xyz = rec.xyz.copy()
        xyz[n_rec // 2] = np.nan
        keep = np.arange(n_rec) != n_rec // 2
        ref_rec = dataclasses.replace(rec, xyz=rec.xyz[keep], types=rec.types[keep])
        rec = dataclasses.replace(rec, xyz=xyz)
    box = T.Box.from_center_size(S.POCKET_CENTER, (size, size, size))
    lig = S.make_ligand(8300, 37, 4).ligand
    ls = gpu.LigSet([lig])
    scene = gpu.Scene(rec, box)
    rng = np.random.default_rng(3)
    n = 96
    pv = S.random_pose_vectors(n, lig.ntors, T.Box.from_center_size(S.POCKET_CENTER, (20.0,) * 3), seed=5)
    u = rng.normal(size=(n, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    far = np.repeat([0.0, 8.0, 20.0, 27.0, 34.0, 300.0], n // 6)[:, None] + rng.uniform(-3, 3, (n, 1))
    pv[:, :3] = np.asarray(S.POCKET_CENTER) + u * far
    pv_d = torch.as_tensor(pv, device="cuda")
    e = torch.zeros(n, device="cuda")
    g = torch.zeros((n, 6 + lig.ntors), device="cuda")
    gpu.check(gpu.lib().ud2_score_posevecs(scene.h, ls.h, 0, n, C.c_void_p(pv_d.data_ptr()), C.c_void_p(e.data_ptr()),
                                           C.c_void_p(g.data_ptr()), gpu.MODE_DIRECT, 1e30, 0.0, gpu.stream_ptr()))
    torch.cuda.synchronize()
    er, gr, _ = O.score_posevecs(O.Topo(lig), O.Scene(ref_rec, box), pv, v_cap=1e30, slope=0.0)
    err = np.abs(e.cpu().numpy() - er) / np.maximum(np.abs(er), 1.0)
    assert err.max() < 1e-4, err.max()
    gs = np.maximum(np.abs(gr).max(axis=1, keepdims=True), 1.0)
    gerr = (np.abs(g.cpu().numpy() - gr) / gs).max()
    assert gerr < 1e-4, gerr
