"""The direct sum of poses inside the listed space, across its edge and beyond it: the same poses scored in scenes of
one receptor whose boxes, and so their listed spaces, lie elsewhere give the same bits (slope 0: no box penalty), and so do
their final scores and decompositions."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _score(gpu, scene, ls, lig, pv):
    import torch
    n = len(pv)
    pv_d = torch.as_tensor(pv, device="cuda")
    e = torch.zeros(n, device="cuda")
    g = torch.zeros((n, 6 + lig.ntors), device="cuda")
    gpu.check(gpu.lib().ud2_score_posevecs(scene.h, ls.h, 0, n, C.c_void_p(pv_d.data_ptr()), C.c_void_p(e.data_ptr()),
                                           C.c_void_p(g.data_ptr()), gpu.MODE_DIRECT, 10.0, 0.0, gpu.stream_ptr()))
    torch.cuda.synchronize()
    return e.cpu().numpy(), g.cpu().numpy()


def _final(gpu, scene, ls, pb, n, stride):
    import torch
    sel = torch.arange(n, dtype=torch.int32, device="cuda")
    o4 = torch.zeros((n, 4), device="cuda")
    dec = torch.zeros((n, stride, 5), device="cuda")
    gpu.check(gpu.lib().ud2_final_score(scene.h, ls.h, pb.ref, C.c_void_p(sel.data_ptr()), n,
                                        C.c_void_p(o4.data_ptr()), gpu.stream_ptr()))
    gpu.check(gpu.lib().ud2_score_decomp(scene.h, ls.h, pb.ref, C.c_void_p(sel.data_ptr()), n, stride,
                                         C.c_void_p(dec.data_ptr()), gpu.stream_ptr()))
    torch.cuda.synchronize()
    return o4[:, :2].cpu().numpy(), dec.cpu().numpy()


@pytest.mark.parametrize("natom,ntors", [(17, 2), (57, 9), (90, 7)])
def test_listed_and_whole_sums_have_the_same_bits(gpu, receptor, natom, ntors):
    import torch
    from unidock_engine import synthetic as S
    from unidock_engine import topology as T
    print(f"listed and whole sums: {natom} atoms", flush=True)
    lig = S.make_ligand(8400 + natom, natom, ntors).ligand
    ls = gpu.LigSet([lig])
    centre = np.asarray(S.POCKET_CENTER)
    n = 48
    pv = S.random_pose_vectors(n, lig.ntors, T.Box.from_center_size(S.POCKET_CENTER, (22.0,) * 3), seed=7)
    pb = gpu.PoseBuffers(ls, n)
    pb.init()
    x = lig.coords.astype(np.float64) - lig.coords.mean(axis=0)
    at = np.random.default_rng(8).uniform(-11, 11, (n, 1, 3)) + centre
    pb.x.copy_(torch.from_numpy((x[None] + at).astype(np.float32).reshape(-1)))
    got = []
    for shift, size in ((0.0, 30.0), (0.0, 2.0), (13.0, 4.0), (25.0, 3.0)):
        box = T.Box.from_center_size(tuple(centre + np.array([shift, 0.0, -shift])), (size,) * 3)
        scene = gpu.Scene(receptor, box)
        got.append(_score(gpu, scene, ls, lig, pv) + _final(gpu, scene, ls, pb, n, natom))
    assert np.isfinite(got[0][0]).all() and (got[0][2][:, 1] != 0).any()
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b), np.abs(a - b).max()
