"""The tuned table and searches of few chains: a table that puts every small ligand on a half-wave variant leaves such a
search on its teams (the same poses, in the time of an untuned process), and a cache file of another build's version is
measured anew instead of taken."""
import ctypes as C
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PROBES = [2, 3, 4, 5, 6, 10, 11, 15]


@pytest.fixture(autouse=True)
def restore_policy(gpu):
    yield
    gpu.set_tile_policy(gpu.TILE_AUTO)


def _search(gpu, scene, ls, nchain=128):
    import torch
    pb = gpu.PoseBuffers(ls, nchain)
    pb.init()
    prm = gpu.McParams(mc_steps=6, opt_steps=20, randomize=1, seed=9, mode=gpu.MODE_GRID, lig_index_base=0, stats_d=None)
    times = []
    for _ in range(6):
        torch.cuda.synchronize()
        t = time.perf_counter()
        gpu.check(gpu.lib().ud2_mc(scene.h, ls.h, pb.ref, C.byref(prm), gpu.stream_ptr()), "ud2_mc")
        torch.cuda.synchronize()
        times.append(time.perf_counter() - t)
    return min(times), pb.x.cpu().numpy(), pb.e.cpu().numpy()


def test_tuned_table_leaves_teams_and_old_caches(gpu, receptor, box, tmp_path):
    from unidock_engine import synthetic as S
    scene = gpu.Scene(receptor, box)
    scene.build_grids(S.GRID_SPACING, PROBES)
    ligs = [S.make_ligand(8950 + k, 20, 4).ligand for k in range(2)]
    ls = gpu.LigSet(ligs)
    path = tmp_path / "tune.txt"
    print("tuned table and teams: measure a table", flush=True)
    gpu.autotune(scene, ls, opt_steps=4, mc_steps=2, cache_path=str(path))
    key, line = path.read_text().splitlines()
    words = line.split()
    # a table with a half-wave variant, in a file of this build, is taken as it is
    path.write_text("\n".join([key, " ".join([words[0], str(gpu.MC_HALF4), "9.5", "1.5", "2.5", "3.5"])]) + "\n")
    info = gpu.autotune(scene, ls, opt_steps=4, mc_steps=2, cache_path=str(path))
    b = int(words[0])
    assert info["variant"][b] == gpu.MC_HALF4 and info["ms"][b][0] == 9.5
    tuned = _search(gpu, scene, ls)
    gpu.set_tile_policy(gpu.TILE_NEVER)
    whole = _search(gpu, scene, ls)
    gpu.set_tile_policy(gpu.TILE_ALWAYS, gpu.MC_HALF4)
    half = _search(gpu, scene, ls)
    print(f"2 x 128 chains: tuned {tuned[0] * 1e3:.2f} ms, never {whole[0] * 1e3:.2f}, always {half[0] * 1e3:.2f}", flush=True)
    for other in (whole, half):
        assert np.array_equal(tuned[1], other[1]) and np.array_equal(tuned[2], other[2])
    # two chains per wave take about twice a team's time
    assert tuned[0] < 1.4 * whole[0], (tuned[0], whole[0])
    # the same table in a file of the version before
    gpu.set_tile_policy(gpu.TILE_AUTO)
    assert key.startswith("ud2-mc-tune 3 ")
    path.write_text(path.read_text().replace("ud2-mc-tune 3 ", "ud2-mc-tune 2 "))
    info = gpu.autotune(scene, ls, opt_steps=4, mc_steps=2, cache_path=str(path))
    assert info["ms"][b][0] != 9.5 and path.read_text().startswith(key)
