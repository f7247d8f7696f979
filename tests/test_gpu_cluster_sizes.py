"""ud2_cluster against the oracle's greedy clustering at the sizes where its rounds change shape: pose counts
around a wave and a block, one pose, limits that merge nothing, a few or all, poses with NaN energies and
coordinates, hydrogens, and ligands of one to four atoms per lane. Membership and order are exact."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _set(ls_ligs, gpu, nchain, seed, spread):
    import torch
    rng = np.random.default_rng(seed)
    ls = gpu.LigSet(ls_ligs)
    pb = gpu.PoseBuffers(ls, nchain)
    xs, es = [], []
    for lig in ls_ligs:
        basin = rng.integers(0, 6, nchain)
        at = rng.uniform(-4, 4, (6, 3))
        x = lig.coords.astype(np.float64)[None] + at[basin][:, None] + rng.normal(0, spread, (nchain, lig.natom, 3))
        xs.append(x.astype(np.float32))
        es.append(np.round(rng.normal(-5, 1, nchain), 2).astype(np.float32))  # ties
    if nchain > 2:
        es[0][1] = np.nan
        xs[0][2, 0, 0] = np.nan
    pb.x.copy_(torch.from_numpy(np.concatenate([x.reshape(-1) for x in xs])))
    pb.e.copy_(torch.from_numpy(np.concatenate(es)))
    return ls, pb, xs, es


@pytest.mark.parametrize("nchain", [1, 2, 63, 64, 65, 130, 1024, 1100])
@pytest.mark.parametrize("limit", [0.0, 0.7, 3.0, 999.0])
def test_cluster_sizes(gpu, nchain, limit):
    import torch
    from oracle import oracle as O
    from unidock_engine import synthetic as S
    print(f"cluster: {nchain} poses, limit {limit}", flush=True)
    sizes = [(9, 0), (70, 4), (140, 5), (205, 3)] if nchain < 1000 else [(11, 1)]
    ligs = [S.make_ligand(8200 + n, n, t).ligand for n, t in sizes]
    ligs[0].types[3] = 0
    if len(ligs) > 1:
        ligs[1].types[::5] = 0
    ls, pb, xs, es = _set(ligs, gpu, nchain, 11 + nchain, 0.3)
    leaders = torch.full((len(ligs), nchain), -1, dtype=torch.int32, device="cuda")
    nlead = torch.zeros(len(ligs), dtype=torch.int32, device="cuda")
    gpu.check(gpu.lib().ud2_cluster(ls.h, pb.ref, limit, C.c_void_p(leaders.data_ptr()), C.c_void_p(nlead.data_ptr()),
                                    gpu.stream_ptr()))
    torch.cuda.synchronize()
    for l, lig in enumerate(ligs):
        e = np.where(np.isnan(es[l]), np.inf, es[l]).astype(np.float32)
        ref = O.cluster(e, xs[l].reshape(nchain, -1), lig.types, limit)
        got = leaders[l, :int(nlead[l])].cpu().numpy()
        assert np.array_equal(got, ref), (l, len(got), len(ref))
