"""ud2_cluster at the most poses per ligand that it takes, against the oracle, and one pose more, refused."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nchain", [8191, 8192])
def test_most_poses(gpu, nchain):
    import torch
    from oracle import oracle as O
    from unidock_engine import synthetic as S
    print(f"cluster: {nchain} poses", flush=True)
    lig = S.make_ligand(8600, 6, 0).ligand
    rng = np.random.default_rng(nchain)
    at = rng.uniform(-6, 6, (40, 3))[rng.integers(0, 40, nchain)]
    x = (lig.coords.astype(np.float64)[None] + at[:, None] + rng.normal(0, 0.2, (nchain, lig.natom, 3))).astype(np.float32)
    e = np.round(rng.normal(-5, 1, nchain), 2).astype(np.float32)  # ties
    ls = gpu.LigSet([lig])
    pb = gpu.PoseBuffers(ls, nchain)
    pb.x.copy_(torch.from_numpy(x.reshape(-1)))
    pb.e.copy_(torch.from_numpy(e))
    leaders = torch.full((nchain,), -1, dtype=torch.int32, device="cuda")
    nlead = torch.zeros(1, dtype=torch.int32, device="cuda")
    gpu.check(gpu.lib().ud2_cluster(ls.h, pb.ref, 2.0, C.c_void_p(leaders.data_ptr()), C.c_void_p(nlead.data_ptr()),
                                    gpu.stream_ptr()))
    torch.cuda.synchronize()
    ref = O.cluster(e, x.reshape(nchain, -1), lig.types, 2.0)
    assert 10 <= len(ref) < nchain // 4
    assert np.array_equal(leaders[:int(nlead[0])].cpu().numpy(), ref), (int(nlead[0]), len(ref))


def test_more_poses_are_refused(gpu):
    from unidock_engine import synthetic as S
    ls = gpu.LigSet([S.make_ligand(8600, 6, 0).ligand])
    pb = gpu.PoseBuffers(ls, 8193)
    assert gpu.lib().ud2_cluster(ls.h, pb.ref, 2.0, C.c_void_p(pb.e.data_ptr()), C.c_void_p(pb.e.data_ptr()),
                                 gpu.stream_ptr()) != 0
