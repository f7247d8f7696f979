"""ud2_cluster of few poses over many ligands, where a ligand's block shrinks with its pose count (a wave for every
four poses, up to 64 poses), against the oracle's greedy clustering. Membership and order are exact."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nchain", [1, 3, 4, 5, 8, 9, 16, 17, 32, 33, 64, 65])
def test_few_poses_of_many_ligands(gpu, nchain):
    import torch
    from oracle import oracle as O
    from unidock_engine import synthetic as S
    print(f"cluster: 300 ligands of {nchain} poses", flush=True)
    kinds = [S.make_ligand(8500 + n, n, t).ligand for n, t in ((7, 0), (33, 3), (66, 4))]
    ligs = [kinds[l % 3] for l in range(300)]
    rng = np.random.default_rng(nchain)
    xs, es = [], []
    for lig in ligs:
        at = rng.uniform(-3, 3, (4, 3))[rng.integers(0, 4, nchain)]
        x = lig.coords.astype(np.float64)[None] + at[:, None] + rng.normal(0, 0.3, (nchain, lig.natom, 3))
        xs.append(x.astype(np.float32))
        es.append(np.round(rng.normal(-5, 1, nchain), 1).astype(np.float32))  # ties
    ls = gpu.LigSet(ligs)
    pb = gpu.PoseBuffers(ls, nchain)
    pb.x.copy_(torch.from_numpy(np.concatenate([x.reshape(-1) for x in xs])))
    pb.e.copy_(torch.from_numpy(np.concatenate(es)))
    leaders = torch.full((len(ligs), nchain), -1, dtype=torch.int32, device="cuda")
    nlead = torch.zeros(len(ligs), dtype=torch.int32, device="cuda")
    gpu.check(gpu.lib().ud2_cluster(ls.h, pb.ref, 1.5, C.c_void_p(leaders.data_ptr()), C.c_void_p(nlead.data_ptr()),
                                    gpu.stream_ptr()))
    torch.cuda.synchronize()
    got, n = leaders.cpu().numpy(), nlead.cpu().numpy()
    for l, lig in enumerate(ligs):
        ref = O.cluster(es[l], xs[l].reshape(nchain, -1), lig.types, 1.5)
        assert np.array_equal(got[l, :n[l]], ref), (l, n[l], len(ref))
