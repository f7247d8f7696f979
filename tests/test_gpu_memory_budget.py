"""The device memory that a run counts against its budget is what it holds: a scene's share with its reach lists, a batch's
topology with its pair-step tables; and a budget that has no room for the lists gives them up, native and Python-driven run
alike, instead of refusing the run or going over it."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIB = 1 << 20
PROBES = [2, 3, 4, 5, 6, 10, 11, 15]


def _free(gpu):
    import torch
    torch.cuda.synchronize()
    return gpu.device_memory()[0]


def test_scene_share_is_counted(gpu, receptor, box):
    from unidock_engine import synthetic as S
    from unidock_engine.api.python import pipeline
    print("scene memory", flush=True)
    first = gpu.Scene(receptor, box)  # what the process's first kernels allocate is no scene's
    first.build_grids(S.GRID_SPACING, PROBES)
    first.close()
    before = _free(gpu)
    scenes = [gpu.Scene(receptor, box) for _ in range(4)]
    for s in scenes:
        s.build_grids(S.GRID_SPACING, PROBES)
    held = before - _free(gpu)
    counted = sum(pipeline.scene_bytes(receptor, s) for s in scenes)
    assert all(s.reach_bytes() > 8 * MIB for s in scenes)
    # the driver gives memory out in pieces of 2 MB: four arrays a scene
    assert held <= counted + 4 * 8 * MIB, (held / MIB, counted / MIB)
    for s in scenes:
        s.close()


@pytest.mark.parametrize("lo,hi", [(17, 32), (33, 64), (65, 80)])
def test_batch_topology_is_counted(gpu, lo, hi):
    from unidock_engine import synthetic as S
    from unidock_engine.api.python import pipeline
    print(f"ligand set memory: {lo}-{hi} atoms", flush=True)
    kinds = [S.make_ligand(8700 + k, n, min(8, n // 6)).ligand for k, n in enumerate(range(lo, hi + 1))]
    ligs = (kinds * 200)[:3000]
    est = pipeline.BatchSize()
    for l in ligs:
        est = est.add(l)
    gpu.LigSet(ligs[:1]).close()
    before = _free(gpu)
    ls = gpu.LigSet(ligs)
    held = before - _free(gpu)
    # ten arrays in pieces of 2 MB, and a tenth for what is not counted
    assert held <= 1.1 * est.bytes(0) + 20 * MIB, (held / MIB, est.bytes(0) / MIB)
    ls.close()


def test_lists_are_given_up_and_change_nothing(gpu, receptor, box):
    import torch
    from unidock_engine import synthetic as S
    lig = S.make_ligand(8710, 40, 6).ligand
    ls = gpu.LigSet([lig])
    scene = gpu.Scene(receptor, box)
    n = 500
    pv = torch.from_numpy(S.random_pose_vectors(n, lig.ntors, box, seed=3)).cuda()
    got = []
    print("scores with and without the reach lists", flush=True)
    for keep in (True, False):
        assert (scene.reach_bytes(keep=keep) > 0) == keep
        e, g = torch.zeros(n, device="cuda"), torch.zeros((n, 6 + lig.ntors), device="cuda")
        gpu.check(gpu.lib().ud2_score_posevecs(scene.h, ls.h, 0, n, C.c_void_p(pv.data_ptr()), C.c_void_p(e.data_ptr()),
                                               C.c_void_p(g.data_ptr()), gpu.MODE_DIRECT, 10.0, 1e6, gpu.stream_ptr()))
        torch.cuda.synchronize()
        got.append((e.cpu().numpy(), g.cpu().numpy()))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("inter_mode", [0, 1])
def test_tight_budgets(gpu, tmp_path, inter_mode):
    """With room for the lists and with a megabyte less than that, the native run and its Python-driven twin write the
    same files."""
    from unidock_engine import synthetic as S
    from unidock_engine.api.python import pipeline
    from unidock_engine.topology import Box, receptor_from_json
    docs = {s.ligand.name: s.json_obj for s in S.config1_ligands(24) if s.ligand.natom <= 40 and s.ligand.ntors <= 8}
    docs = dict(list(docs.items())[:5])
    rec = S.receptor_json(S.make_receptor())
    c = S.POCKET_CENTER
    box = dict(center_x=c[0], center_y=c[1], center_z=c[2], size_x=S.BOX_SIZE, size_y=S.BOX_SIZE, size_z=S.BOX_SIZE)
    r = receptor_from_json(rec, Box.from_center_size(c, (S.BOX_SIZE,) * 3))
    scene = gpu.Scene(r, Box.from_center_size(c, (S.BOX_SIZE,) * 3))
    if inter_mode == 1:
        scene.build_grids(S.GRID_SPACING, PROBES)
    nchain = 512
    share = pipeline.scene_bytes(r, scene)
    lists = scene.reach_bytes()
    ligs = [s.ligand for s in S.config1_ligands(24) if s.ligand.name in docs]
    one = max(pipeline.BatchSize().add(l).bytes(nchain) for l in ligs) // MIB
    scene.close()
    for limit in (share // MIB + one + 1, share // MIB + one, (share - lists) // MIB + one + 1):
        outs = []
        for host in ("native", "python"):
            print(f"budget {limit} MB, mode {inter_mode}, {host}", flush=True)
            d = tmp_path / f"{host}{limit}"
            p = pipeline.DockingPipeline(output_dir=str(d), name_json="run", search_mode="free", exhaustiveness=nchain,
                                         mc_steps=2, refine_steps=1, seed=3, max_gpu_mem=limit, **box)
            p.inter_mode = inter_mode
            p.host = host
            p.set_receptor(rec)
            p.add_ligands(docs)
            p.run()
            outs.append({os.path.basename(f): open(f, "rb").read() for f in p.output_files})
        assert outs[0] and outs[0] == outs[1], limit
