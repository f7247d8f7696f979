"""The builds of the plain search that launches of different sizes run, against each other: a search of few chains (a team
of four waves per chain), of a chip a quarter or half full and of a full one (one wave per chain, builds of other register
budgets), in direct mode and on maps, with bias sites (which turn the trial screen off), with an axis of zero length
(whose search directions are not finite) and over a part of the uneven batch. A ligand's random streams are keyed by its
index, so the same chains come out of all of them, bit for bit; half-wave variants are not run in direct mode,
whatever the policy."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PROBES = [2, 3, 4, 5, 6, 10, 11, 15]


@pytest.fixture(autouse=True)
def restore_policy(gpu):
    yield
    gpu.set_tile_policy(gpu.TILE_AUTO)


@pytest.fixture(scope="module")
def scene(gpu, receptor, box):
    from unidock_engine import synthetic as S
    sc = gpu.Scene(receptor, box)
    sc.build_grids(S.GRID_SPACING, PROBES)
    return sc


def _search(gpu, scene, ligs, n_first, nchain, mode, mc, opt, **kw):
    """Pose buffers of the first n_first ligands."""
    import torch
    ls = gpu.LigSet(ligs, **kw)
    pb = gpu.PoseBuffers(ls, nchain)
    pb.init()
    prm = gpu.McParams(mc_steps=mc, opt_steps=opt, randomize=1, seed=19, mode=mode, lig_index_base=0, stats_d=None)
    gpu.check(gpu.lib().ud2_mc(scene.h, ls.h, pb.ref, C.byref(prm), gpu.stream_ptr()), "ud2_mc")
    torch.cuda.synchronize()
    na = sum(l.natom for l in ligs[:n_first]) * nchain
    nt = sum(l.ntors for l in ligs[:n_first]) * nchain
    n = n_first * nchain
    return [t.cpu().numpy() for t in (pb.x[:3 * na], pb.c[:3 * n], pb.rv[:3 * n], pb.dihe[:nt], pb.e[:n])]


def _same(a, b, what):
    for x, y in zip(a, b):
        assert np.array_equal(x, y, equal_nan=True), what


def _with_sites(lig):
    rng = np.random.default_rng(lig.natom)
    start = np.zeros(lig.natom + 1, np.int32)
    rows = []
    for a in range(lig.natom):
        if a % 3 == 0:
            rows.append([*(lig.coords[a] + rng.uniform(-1.5, 1.5, 3)), -3.0, 2.0])
        start[a + 1] = len(rows)
    return dataclasses.replace(lig, bias_start=start, bias=np.asarray(rows, np.float32))


def _without_axis(lig):
    x = lig.coords.copy()
    ax = np.asarray(lig.axis).reshape(-1, 2)[lig.ntors // 2]
    x[ax[1]] = x[ax[0]]
    return dataclasses.replace(lig, coords=x)


@pytest.mark.parametrize("natom,ntors", [(9, 1), (22, 4), (32, 14), (50, 7), (70, 8)])
@pytest.mark.parametrize("kind", ["plain", "pos", "align", "constraint", "no_axis"])
def test_direct_builds(gpu, scene, natom, ntors, kind):
    from unidock_engine import synthetic as S
    print(f"direct builds: {natom} atoms, {kind}", flush=True)
    lig = S.make_ligand(9000 + natom, natom, ntors).ligand
    kw = {}
    if kind in ("pos", "align"):
        lig, kw = _with_sites(lig), dict(bias=kind, bias_k=0.7)
    elif kind == "constraint":
        kw = dict(constraint=True)
    elif kind == "no_axis":
        lig = _without_axis(lig)
    # 80, 1,600 and 2,400 chains: teams, one wave per chain at up to two and up to four blocks per CU
    runs = [_search(gpu, scene, [lig] * copies, 1, 8, gpu.MODE_DIRECT, 2, 7, **kw) for copies in (10, 200, 300)]
    _same(runs[0], runs[1], "teams against the sparse build")
    _same(runs[0], runs[2], "teams against the dense build")
    gpu.set_tile_policy(gpu.TILE_ALWAYS, gpu.MC_HALF4)
    _same(runs[0], _search(gpu, scene, [lig] * 10, 1, 8, gpu.MODE_DIRECT, 2, 7, **kw), "half waves asked for")


@pytest.mark.parametrize("natom,ntors", [(22, 4), (50, 7), (70, 8)])
@pytest.mark.parametrize("kind", ["pos", "align", "no_axis"])
def test_grid_teams(gpu, scene, natom, ntors, kind):
    from unidock_engine import synthetic as S
    print(f"grid teams: {natom} atoms, {kind}", flush=True)
    lig = S.make_ligand(9000 + natom, natom, ntors).ligand
    kw = {}
    if kind == "no_axis":
        lig = _without_axis(lig)
    else:
        lig, kw = _with_sites(lig), dict(bias=kind, bias_k=0.7)
    runs = [_search(gpu, scene, [lig] * copies, 1, 8, gpu.MODE_GRID, 3, 10, **kw) for copies in (10, 400, 900)]
    _same(runs[0], runs[1], "teams against the four-wave build")
    _same(runs[0], runs[2], "teams against the six-wave build")


def test_part_of_the_uneven_batch(gpu, scene):
    from unidock_engine import synthetic as S
    print("48 ligands of the uneven batch, as teams and in a full launch", flush=True)
    ligs = [s.ligand for s in S.config1_ligands(256)]
    few = _search(gpu, scene, ligs[:48], 48, 24, gpu.MODE_GRID, 8, 28)
    full = _search(gpu, scene, ligs, 48, 24, gpu.MODE_GRID, 8, 28)
    _same(few, full, "teams against a full launch")


@pytest.mark.parametrize("natom,ntors", [(22, 4), (70, 8)])
@pytest.mark.parametrize("mode", ["grid", "direct"])
def test_evaluations_counted(gpu, scene, natom, ntors, mode):
    """The counters of a team's chains are those of one wave per chain: the 301st copy's chains alone (by its index in the
    stream key) count what they add to a launch of 300 copies."""
    import torch
    from unidock_engine import synthetic as S
    print(f"evaluations: {natom} atoms, {mode}", flush=True)
    lig = S.make_ligand(9100 + natom, natom, ntors).ligand
    m = gpu.MODE_GRID if mode == "grid" else gpu.MODE_DIRECT

    def counted(copies, base):
        ls = gpu.LigSet([lig] * copies)
        pb = gpu.PoseBuffers(ls, 8)
        pb.init()
        stats = torch.zeros(4, dtype=torch.int64, device="cuda")
        prm = gpu.McParams(mc_steps=3, opt_steps=10, randomize=1, seed=23, mode=m, lig_index_base=base,
                           stats_d=stats.data_ptr())
        gpu.check(gpu.lib().ud2_mc(scene.h, ls.h, pb.ref, C.byref(prm), gpu.stream_ptr()), "ud2_mc")
        torch.cuda.synchronize()
        return stats.cpu().numpy()

    alone = counted(1, 300)
    assert alone[0] > 0 and alone[3] == 8
    assert np.array_equal(alone, counted(301, 0) - counted(300, 0))
