"""Ligands of 129-256 atoms, whose pairs beyond the cutoff are computed and dropped instead of skipped: an atom that is
nowhere (NaN) and the same atom far from all others leave the same energy and the same force on the ligand's centre,
and so does half of a ligand beyond the other half's reach against each half's own pairs."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _energy(gpu, scene, lig, xs):
    import torch
    ls = gpu.LigSet([lig])
    n = len(xs)
    pb = gpu.PoseBuffers(ls, n)
    pb.init()
    pb.x.copy_(torch.from_numpy(np.stack(xs).astype(np.float32).reshape(-1)))
    sel = torch.arange(n, dtype=torch.int32, device="cuda")
    e, g = torch.zeros(n, device="cuda"), torch.zeros((n, 64), device="cuda")
    gpu.check(gpu.lib().ud2_energy_grad(scene.h, ls.h, pb.ref, C.c_void_p(sel.data_ptr()), n, gpu.MODE_DIRECT, 1e30, 0.0,
                                        C.c_void_p(e.data_ptr()), C.c_void_p(g.data_ptr()), gpu.stream_ptr()))
    torch.cuda.synchronize()
    return e.cpu().numpy(), g.cpu().numpy()


@pytest.mark.parametrize("natom", [129, 150, 192, 193, 256])
def test_pairs_beyond_the_cutoff(gpu, receptor, box, natom):
    from unidock_engine import synthetic as S
    print(f"wide ligands' pairs: {natom} atoms", flush=True)
    lig = S.make_ligand(9200 + natom, natom, 3).ligand
    scene = gpu.Scene(dataclasses.replace(receptor, xyz=receptor.xyz[:0], types=receptor.types[:0]), box)  # pairs only
    x0 = lig.coords.astype(np.float32)
    for atom in (0, natom // 2, natom - 1):
        nowhere, far = x0.copy(), x0.copy()
        nowhere[atom] = np.nan
        far[atom] += 1e4
        e, g = _energy(gpu, scene, lig, [nowhere, far])
        assert np.isfinite(e).all() and e[0] == e[1] and np.array_equal(g[0, :3], g[1, :3]), (atom, e)
    # the two halves of the atoms 1,000 A apart: the sum of what each half's pairs give (FP32 sums of a few hundred terms)
    half = np.arange(natom) < natom // 2
    apart = x0.copy()
    apart[half] += 1000.0
    p = np.asarray(lig.pairs).reshape(-1, 2)
    both = half[p[:, 0]] == half[p[:, 1]]
    e, _ = _energy(gpu, scene, lig, [apart])
    parts = [_energy(gpu, scene, dataclasses.replace(lig, pairs=p[both & (half[p[:, 0]] == h)]), [apart])[0][0]
             for h in (False, True)]
    assert abs(float(e[0]) - float(sum(parts))) <= 1e-5 * max(1.0, sum(abs(float(v)) for v in parts)), (e, parts)
