"""Pair tables of small ligands beside larger ones: sets that mix ligands of at most 32 atoms, whose tables are written
on the GPU, with ligands of 33-64 and more atoms and with ligands without any scored pair, in several orders. Energies and
gradients of every ligand have the bits that it gives in a set of its own, and agree with the oracle (FP64; tolerance as
in test_gpu_parity)."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _grad(gpu, scene, ls, nchain, pv_of):
    import torch
    out = []
    for l, lig in enumerate(ls.ligands):
        pv = pv_of(lig)
        pv_d = torch.as_tensor(pv, device="cuda")
        e = torch.zeros(nchain, device="cuda")
        g = torch.zeros((nchain, 6 + lig.ntors), device="cuda")
        gpu.check(gpu.lib().ud2_score_posevecs(scene.h, ls.h, l, nchain, C.c_void_p(pv_d.data_ptr()),
                                               C.c_void_p(e.data_ptr()), C.c_void_p(g.data_ptr()), gpu.MODE_DIRECT, 1e30,
                                               0.0, gpu.stream_ptr()))
        torch.cuda.synchronize()
        out.append((e.cpu().numpy(), g.cpu().numpy()))
    return out


@pytest.mark.parametrize("order", [0, 1, 2])
def test_mixed_sets(gpu, receptor, box, order):
    from unidock_engine import synthetic as S
    ligs = [S.make_ligand(8800 + n, n, t).ligand
            for n, t in ((4, 0), (7, 1), (16, 3), (31, 5), (32, 4), (33, 4), (50, 6), (64, 8), (65, 6), (130, 7))]
    bare = S.make_ligand(8850, 14, 1).ligand
    ligs += [dataclasses.replace(bare, pairs=bare.pairs[:0]),
             dataclasses.replace(ligs[6], pairs=ligs[6].pairs[:0])]
    ligs = [ligs[i] for i in np.random.default_rng(order).permutation(len(ligs))]
    print(f"pair tables: order {order}", flush=True)
    scene = gpu.Scene(receptor, box)
    n = 12
    pv_of = lambda lig: S.random_pose_vectors(n, lig.ntors, box, seed=lig.natom)  # noqa: E731
    mixed = _grad(gpu, scene, gpu.LigSet(ligs), n, pv_of)
    for lig, (e, g) in zip(ligs, mixed):
        e1, g1 = _grad(gpu, scene, gpu.LigSet([lig]), n, pv_of)[0]
        assert np.array_equal(e, e1) and np.array_equal(g, g1), lig.natom
        er, gr, _ = O.score_posevecs(O.Topo(lig), O.Scene(receptor, box), pv_of(lig), v_cap=1e30, slope=0.0)
        assert (np.abs(e - er) / np.maximum(np.abs(er), 1.0)).max() < 1e-4, lig.natom
        gs = np.maximum(np.abs(gr).max(axis=1, keepdims=True), 1.0)
        assert (np.abs(g - gr) / gs).max() < 1e-4, lig.natom
