"""The docking work this framework is used for, as cases that can be timed and compared.

Each case is one pass through a public entry point of ``unidock_engine`` over seeded synthetic inputs
of the repository's own workloads: the receptor shell of 2,000 heavy atoms, the 30 A box, ligands of
10-60 (screening batch) or 10-80 heavy atoms (large batch) with 0-20 rotatable bonds, grid maps at
0.375 A. ``exact`` restates scoring, grid maps and the network's training step in 64 bits. Searches
(Monte Carlo over BFGS-refined poses) have no such value.
"""
import ctypes as C
import dataclasses
import functools
import json
import math
import os
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "uni-dock2_amd"))

from unidock_engine import _native as N  # noqa: E402
from unidock_engine import proposal as LP  # noqa: E402
from unidock_engine import synthetic as S  # noqa: E402
from unidock_engine.engine import DEFAULT_PROBE_TYPES, heuristic_opt_steps  # noqa: E402
from unidock_engine.api.python.pipeline import DockingPipeline  # noqa: E402
from unidock_engine.topology import Box  # noqa: E402

SPACING = S.GRID_SPACING
MODES = {"grid": N.MODE_GRID, "direct": N.MODE_DIRECT}
MEAN_PAIRS = 0.33  # scored intra pairs of the synthetic ligands, as a share of natom ** 2


# ------------------------------------------------------------------ cases
def listed():
    return [
        # virtual screening with the learned search: the benchmark's 1,024-ligand batch, the largest case
        dict(name="dock_learned_1024", kind="dock", n_lig=1024, pool="screen", lo=10, hi=60, nchain=32, mc_steps=40,
             opt_steps=28, mode="grid", search="learned"),
        # the reference's search on ligands of every size, those past 64 atoms among them
        dict(name="dock_plain_256", kind="dock", n_lig=256, pool="large", lo=10, hi=80, nchain=128, mc_steps=40,
             opt_steps=-1, mode="grid", search="plain"),
        # one ligand at a time, as an interactive user or a service docks: 24 atoms, 128 chains, 20 steps
        dict(name="dock_single", kind="dock", n_lig=1, pool="screen", lo=24, hi=24, nchain=128, mc_steps=20,
             opt_steps=50, mode="grid", search="plain"),
        # the reference's search semantics (direct receptor sum) on a few leads
        dict(name="dock_direct_8", kind="dock", n_lig=8, pool="screen", lo=17, hi=53, nchain=128, mc_steps=10,
             opt_steps=28, mode="direct", search="plain"),
        # the drop-in: engine JSON in, result files out, the "fast" preset on a small library
        dict(name="pipeline_fast_16", kind="pipeline", n_lig=16, lo=10, hi=60, preset="fast"),
        # the scoring microbenchmark: energy and gradient of a million poses of a 40-atom ligand
        dict(name="score_grid_1m", kind="score", n_pose=1 << 20, natom=40, ntors=8, mode="grid"),
        # scoring by the direct receptor sum, ragged sizes
        dict(name="score_direct_20k", kind="score", n_pose=20011, natom=57, ntors=13, mode="direct"),
        # the smallest call: energy and gradient of a handful of poses for a caller's own optimiser
        dict(name="energy_grad_37", kind="energy_grad", n_lig=1, lo=31, hi=31, nchain=37, mode="grid"),
        # final re-score of a screen's kept poses with the per-atom decomposition
        dict(name="rescore_10k", kind="rescore", n_lig=1021, lo=10, hi=60, nchain=10),
        # RMSD clustering of a detailed search's poses
        dict(name="cluster_64x512", kind="cluster", n_lig=64, lo=10, hi=60, nchain=512),
        # a new receptor: the maps of a run, built and saved
        dict(name="build_grids", kind="grids", n_rec=2000, box=30.0, n_types=8),
        # one optimiser step of the proposal network at the trainer's minibatch
        dict(name="train_1024", kind="train", groups=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dock", "dock", "dock_direct", "pipeline", "score", "score", "energy_grad", "rescore",
                       "cluster", "grids", "train"])
    lo = rng.randint(10, 40)
    hi = rng.randint(lo + 4, 60)
    if kind == "dock":
        search = rng.choice(["plain", "learned"])
        pool = rng.choice(["screen", "large"])
        return dict(kind="dock", n_lig=_log(rng, 1, 120), pool=pool, lo=lo, hi=hi if pool == "screen" else 80,
                    nchain=_log(rng, 16, 128), mc_steps=rng.randint(10, 40), opt_steps=rng.choice([-1, 12, 28]),
                    mode="grid", search=search)
    if kind == "dock_direct":
        return dict(kind="dock", n_lig=_log(rng, 1, 8), pool="screen", lo=lo, hi=hi, nchain=_log(rng, 16, 128),
                    mc_steps=rng.randint(4, 10), opt_steps=rng.choice([-1, 12, 28]), mode="direct", search="plain")
    if kind == "pipeline":
        return dict(kind="pipeline", n_lig=_log(rng, 1, 40), lo=lo, hi=hi, preset="fast")
    if kind == "score":
        natom = rng.randint(10, 60)
        mode = rng.choice(["grid", "grid", "direct"])
        return dict(kind="score", n_pose=_log(rng, 1, 1 << 19 if mode == "grid" else 30000), natom=natom,
                    ntors=rng.randint(0, min(15, natom - 6)), mode=mode)
    if kind == "energy_grad":
        return dict(kind="energy_grad", n_lig=_log(rng, 1, 60), lo=lo, hi=hi, nchain=_log(rng, 1, 64),
                    mode=rng.choice(["grid", "direct"]))
    if kind == "rescore":
        return dict(kind="rescore", n_lig=_log(rng, 1, 1024), lo=lo, hi=hi, nchain=rng.randint(1, 10))
    if kind == "cluster":
        return dict(kind="cluster", n_lig=_log(rng, 1, 128), lo=lo, hi=hi, nchain=_log(rng, 24, 512))
    if kind == "grids":
        return dict(kind="grids", n_rec=rng.randint(600, 2000), box=float(rng.randint(36, 60)) / 2.0,
                    n_types=rng.randint(4, 12))
    return dict(kind="train", groups=16 * _log(rng, 4, 64))


# ----------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=None)
def _base_receptor():
    return S.make_receptor()


def _receptor(seed, n_rec=2000):
    """The receptor shell turned about the pocket's centre, its atom types dealt anew."""
    rng = np.random.default_rng(seed)
    r = _base_receptor()
    c = np.asarray(S.POCKET_CENTER)
    q, t = np.linalg.qr(rng.normal(size=(3, 3)))
    xyz = ((r.xyz - c) @ (q * np.sign(np.diag(t))) + c).astype(np.float32)
    order = rng.permutation(len(r.types))
    return dataclasses.replace(r, xyz=xyz[:n_rec], types=r.types[order][:n_rec], ff_types=r.ff_types[order][:n_rec],
                               charges=r.charges[:n_rec])


@functools.lru_cache(maxsize=None)
def _pool(name, n):
    return (S.config1_ligands if name == "screen" else S.config4_ligands)(n)


@functools.lru_cache(maxsize=None)
def _fixed(seed, natom, ntors):
    return S.make_ligand(seed, natom, ntors)


def _synth(seed, n_lig, lo, hi, pool="screen"):
    """n_lig synthetic ligands of lo to hi heavy atoms, the same ones for every seed, in an order of its own."""
    if lo == hi:
        return [_fixed(1000 + (seed + k) % 8, lo, 5) for k in range(n_lig)]
    got = [s for s in _pool(pool, 1024 if n_lig > 256 else 256) if lo <= s.ligand.natom <= hi]
    chosen = np.random.default_rng(n_lig + 1000 * lo + 7).permutation(max(n_lig, len(got)))[:n_lig]
    return [got[i % len(got)] for i in np.random.default_rng(seed + 17).permutation(chosen)]


def _turned(lig, rng):
    """The ligand with its input conformation turned about its centroid."""
    q, t = np.linalg.qr(rng.normal(size=(3, 3)))
    c = lig.coords.astype(np.float64).mean(axis=0)
    q = q * np.sign(np.diag(t))
    if np.linalg.det(q) < 0:
        q[:, 0] *= -1.0
    return dataclasses.replace(lig, coords=((lig.coords - c) @ q + c).astype(np.float32))


def _ligands(case, seed):
    rng = np.random.default_rng(seed + 29)
    return [_turned(s.ligand, rng) for s in _synth(seed, case["n_lig"], case["lo"], case["hi"],
                                                  case.get("pool", "screen"))]


def _scene(seed, mode):
    receptor, box = _receptor(seed), S.docking_box()
    scene = N.Scene(receptor, box)
    if mode == "grid":
        scene.build_grids(SPACING, DEFAULT_PROBE_TYPES)
    return scene


def _pose_arrays(ligands, nchain, seed):
    """nchain rigid poses of every ligand, in a few basins each as a search leaves them: coordinates,
    centres, rotation vectors and energies of every pose, in the order of the pose buffers."""
    rng = np.random.default_rng(seed + 31)
    xs, cs, rs, es = [], [], [], []
    centre = np.asarray(S.POCKET_CENTER)
    for lig in ligands:
        x0 = lig.coords.astype(np.float64)
        x0 = x0 - x0.mean(axis=0)
        nb = max(1, min(nchain, int(rng.integers(4, 40))))
        basin = np.minimum(rng.geometric(0.12, size=nchain) - 1, nb - 1)
        u = rng.normal(size=(nb, 3))
        u /= np.linalg.norm(u, axis=1, keepdims=True)
        ang = rng.uniform(0.05, 3.0, size=nb)
        v = (u * ang[:, None])[basin] + rng.normal(0.0, 0.06, size=(nchain, 3))
        c = (centre + rng.uniform(-8.0, 8.0, size=(nb, 3)))[basin] + rng.normal(0.0, 0.15, size=(nchain, 3))
        th = np.linalg.norm(v, axis=1)[:, None, None]
        k = np.zeros((nchain, 3, 3))
        k[:, 0, 1], k[:, 0, 2], k[:, 1, 2] = -v[:, 2], v[:, 1], -v[:, 0]
        k[:, 1, 0], k[:, 2, 0], k[:, 2, 1] = v[:, 2], -v[:, 1], v[:, 0]
        rot = np.eye(3) + np.sin(th) / th * k + (1.0 - np.cos(th)) / th ** 2 * (k @ k)
        xs.append((np.einsum("cij,aj->cai", rot, x0) + c[:, None, :]).astype(np.float32).reshape(-1))
        cs.append(c)
        rs.append(v)
        es.append(np.linspace(-9.0, -2.0, nb)[basin] + rng.normal(0.0, 0.3, size=nchain))
    return (np.concatenate(xs), np.concatenate(cs).astype(np.float32), np.concatenate(rs).astype(np.float32),
            np.concatenate(es).astype(np.float32))


def _poses(ligset, nchain, seed):
    pb = N.PoseBuffers(ligset, nchain)
    x, c, r, e = _pose_arrays(ligset.ligands, nchain, seed)
    pb.x.copy_(torch.from_numpy(x))
    pb.c.copy_(torch.from_numpy(c.reshape(-1)))
    pb.rv.copy_(torch.from_numpy(r.reshape(-1)))
    pb.e.copy_(torch.from_numpy(e))
    for lig, at in zip(ligset.ligands, ligset.arrays["tors_off"]):
        if lig.ntors:
            d = torch.from_numpy(np.ascontiguousarray(lig.dihedrals, np.float32)).repeat(nchain)
            pb.dihe[int(at) * nchain:int(at) * nchain + d.numel()].copy_(d)
    return pb


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _score_ligand(case):
    return _fixed(3000, case["natom"], case["ntors"]).ligand


def _pose_vectors(case, seed):
    # centres in the middle of the box, where a search keeps its ligands
    lig = _score_ligand(case)
    return S.random_pose_vectors(case["n_pose"], lig.ntors, Box.from_center_size(S.POCKET_CENTER, (20.0,) * 3), seed=seed)


def _train_data(case, seed):
    """Features and labels of twice the minibatch's groups of 16 candidates, and a shuffled minibatch.
    Counts, pooled energies and move globals as the feature kernel gives them, in bf16."""
    rng = np.random.default_rng(seed + 41)
    n = 2 * case["groups"] * N.MLP_GROUP
    x = np.zeros((n, N.MLP_FEATURES), np.float32)
    x[:, :64] = rng.poisson(2.0, size=(n, 64)) * rng.normal(0.5, 0.6, size=(n, 64))
    x[:, 64 + np.arange(3)] = np.eye(3)[rng.integers(0, 3, size=n)]
    x[:, 67:73] = rng.normal(0.3, 0.4, size=(n, 6))
    bits = (torch.from_numpy(x).to(torch.bfloat16).view(torch.int16)).cuda()
    y = torch.from_numpy(rng.gamma(2.0, 1.5, size=n).astype(np.float32) - 6.0).cuda()
    g = torch.from_numpy(rng.permutation(2 * case["groups"])[:case["groups"]].astype(np.int32)).cuda()
    params = LP.init_params(seed % 1000)
    params[N.MLP_NPARAM:N.MLP_NPARAM + N.MLP_FEATURES] = 0.2
    params[N.MLP_NPARAM + N.MLP_FEATURES:] = 0.7
    return bits, y, g, params


def prepare(case, seed):
    kind = case["kind"]
    if kind == "dock":
        ligands = _ligands(case, seed)
        opt = case["opt_steps"] if case["opt_steps"] >= 0 else heuristic_opt_steps(max(l.natom for l in ligands))
        return dict(kind=kind, scene=_scene(seed, case["mode"]), ligset=N.LigSet(ligands),
                    mlp=N.Mlp(LP.load()) if case["search"] == "learned" else None,
                    args=dict(nchain=case["nchain"], mc_steps=case["mc_steps"], opt_steps=opt, seed=seed,
                              mode=MODES[case["mode"]]))
    if kind == "pipeline":
        out = tempfile.TemporaryDirectory(prefix="ud2_")
        cx, cy, cz = S.POCKET_CENTER
        pipe = DockingPipeline(output_dir=out.name, center_x=cx, center_y=cy, center_z=cz, size_x=S.BOX_SIZE,
                               size_y=S.BOX_SIZE, size_z=S.BOX_SIZE, search_mode=case["preset"], seed=seed % (1 << 31))
        pipe.set_receptor(S.receptor_json(_receptor(seed)))
        pipe.add_ligands({"mol%d" % k: s.json_obj
                          for k, s in enumerate(_synth(seed, case["n_lig"], case["lo"], case["hi"]))})
        return dict(kind=kind, pipe=pipe, out=out, shape=(case["n_lig"], 10, 7 + 3 * case["hi"] + 20))
    if kind == "score":
        lig = _score_ligand(case)
        n = case["n_pose"]
        return dict(kind=kind, scene=_scene(seed, case["mode"]), ligset=N.LigSet([lig]), n=n, mode=MODES[case["mode"]],
                    pv=torch.from_numpy(_pose_vectors(case, seed)).cuda(), e=torch.zeros(n, device="cuda"),
                    g=torch.zeros((n, 6 + lig.ntors), device="cuda"))
    if kind in ("energy_grad", "rescore", "cluster"):
        ligset = N.LigSet(_ligands(case, seed))
        nchain, n = case["nchain"], case["n_lig"] * case["nchain"]
        s = dict(kind=kind, scene=_scene(seed, case.get("mode", "direct")), ligset=ligset, n=n,
                 poses=_poses(ligset, nchain, seed))
        if kind == "cluster":
            s["leaders"] = torch.zeros((case["n_lig"], nchain), dtype=torch.int32, device="cuda")
            s["nlead"] = torch.zeros(case["n_lig"], dtype=torch.int32, device="cuda")
            return s
        s["sel"] = torch.arange(n, dtype=torch.int32, device="cuda")
        if kind == "energy_grad":
            return dict(s, mode=MODES[case["mode"]], e=torch.zeros(n, device="cuda"),
                        g=torch.zeros((n, 64), device="cuda"))
        stride = max(l.natom for l in ligset.ligands)
        return dict(s, stride=stride, out4=torch.zeros((n, 4), device="cuda"),
                    decomp=torch.zeros((n, stride, 5), device="cuda"))
    if kind == "grids":
        box = S.docking_box(size=case["box"])
        return dict(kind=kind, scene=N.Scene(_receptor(seed, case["n_rec"]), box), types=_probe_types(case))
    x, y, g, params = _train_data(case, seed)
    return dict(kind=kind, mlp=N.Mlp(params), x=x, y=y, groups=g, opt=N.Adam(1e-3, 0.9, 0.999, 1e-8),
                loss=torch.zeros(1, device="cuda"))


def _probe_types(case):
    return (list(DEFAULT_PROBE_TYPES) + [9, 8, 7, 12])[:case["n_types"]]


# -------------------------------------------------------------------- run
def run(state):
    kind = state["kind"]
    lib = N.lib()
    if kind == "dock":
        r = N.dock(state["scene"], state["ligset"], mlp=state["mlp"], **state["args"])
        # search_ms and stats are a timer and counters, not results
        return {k: r[k] for k in ("n_out", "chain", "energy", "coords", "dihedrals")}
    if kind == "pipeline":
        pipe = state["pipe"]
        pipe.output_files.clear()
        pipe.run()
        n_pose, values = np.zeros(state["shape"][0], np.int32), np.zeros(state["shape"], np.float32)
        for path in pipe.output_files:
            with open(path) as f:
                for name, poses in json.load(f).items():
                    at = int(name[3:])
                    n_pose[at] = len(poses)
                    for k, p in enumerate(poses):
                        v = p["energy"] + p["coords"] + p["dihedrals"]
                        values[at, k, :len(v)] = v
        return dict(n_pose=n_pose, values=values)
    st = N.stream_ptr()
    if kind == "score":
        N.check(lib.ud2_score_posevecs(state["scene"].h, state["ligset"].h, 0, state["n"], _ptr(state["pv"]),
                                       _ptr(state["e"]), _ptr(state["g"]), state["mode"], 10.0, 1e6, st),
                "ud2_score_posevecs")
        return dict(e=state["e"], g=state["g"])
    if kind == "energy_grad":
        N.check(lib.ud2_energy_grad(state["scene"].h, state["ligset"].h, state["poses"].ref, _ptr(state["sel"]),
                                    state["n"], state["mode"], 10.0, 1e6, _ptr(state["e"]), _ptr(state["g"]), st),
                "ud2_energy_grad")
        return dict(e=state["e"], g=state["g"])
    if kind == "rescore":
        N.check(lib.ud2_final_score(state["scene"].h, state["ligset"].h, state["poses"].ref, _ptr(state["sel"]),
                                    state["n"], _ptr(state["out4"]), st), "ud2_final_score")
        N.check(lib.ud2_score_decomp(state["scene"].h, state["ligset"].h, state["poses"].ref, _ptr(state["sel"]),
                                     state["n"], state["stride"], _ptr(state["decomp"]), st), "ud2_score_decomp")
        return dict(out4=state["out4"], decomp=state["decomp"])
    if kind == "cluster":
        N.check(lib.ud2_cluster(state["ligset"].h, state["poses"].ref, 1.0, _ptr(state["leaders"]),
                                _ptr(state["nlead"]), st), "ud2_cluster")
        return dict(leaders=state["leaders"], n=state["nlead"])
    if kind == "grids":
        state["scene"].build_grids(SPACING, state["types"])
        return state["scene"].download_maps()
    N.check(lib.ud2_mlp_train_step(state["mlp"].h, _ptr(state["x"]), _ptr(state["y"]), _ptr(state["groups"]),
                                   state["groups"].numel(), C.byref(state["opt"]), _ptr(state["loss"]), st),
            "ud2_mlp_train_step")
    return dict(loss=state["loss"], params=state["mlp"].params())


# ------------------------------------------------------------------- work
def work(case):
    """Bytes: inputs and outputs once (the maps and the receptor among the inputs). Operations: an
    evaluation is 40 per scored pair, 60 per atom on maps, 25 per receptor atom in the direct sum's
    reach (about 90) for each ligand atom, and 60 per torsion; a search step is a BFGS run with one
    evaluation per iteration."""
    kind = case["kind"]
    maps = 8 * 4 * 81 ** 3
    reach = 90

    def evaluation(na, nt, mode):
        return 40 * MEAN_PAIRS * na * na + na * (60 if mode == "grid" else 25 * reach) + 60 * nt

    if kind in ("dock", "pipeline"):
        c = dict(dict(nchain=128, mc_steps=20, opt_steps=-1, mode="grid"), **case)
        na = 0.5 * (c["lo"] + c["hi"])
        opt = c["opt_steps"] if c["opt_steps"] > 0 else heuristic_opt_steps(c["hi"])
        evals = c["n_lig"] * c["nchain"] * c["mc_steps"] * (opt + 1)
        return dict(bytes=(maps if c["mode"] == "grid" else 0) + 32000 + c["n_lig"] * na * 12 * 11,
                    flops=evals * evaluation(na, 7, c["mode"]))
    if kind == "score":
        n, na, nt = case["n_pose"], case["natom"], case["ntors"]
        return dict(bytes=n * 4 * (7 + nt + 1 + 6 + nt) + (maps if case["mode"] == "grid" else 32000),
                    flops=n * evaluation(na, nt, case["mode"]))
    if kind in ("energy_grad", "rescore", "cluster"):
        n, na = case["n_lig"] * case["nchain"], 0.5 * (case["lo"] + case["hi"])
        if kind == "energy_grad":
            return dict(bytes=n * (12 * na + 4 * 65) + min(maps, n * na * 32), flops=n * evaluation(na, 7, case["mode"]))
        if kind == "rescore":
            return dict(bytes=n * (12 * na + 16 + 20 * na) + 32000, flops=n * 2 * na * 25 * reach)
        # every pose is compared with the leaders before it: a tenth of the chains on average
        return dict(bytes=n * 12 * na + n * 4, flops=n * 0.1 * case["nchain"] * 8 * na)
    if kind == "grids":
        npt = (round(case["box"] / SPACING) + 1) ** 3
        return dict(bytes=npt * 4 * case["n_types"], flops=npt * 45 * case["n_types"] * 25)
    rows = case["groups"] * N.MLP_GROUP
    return dict(bytes=rows * 164 + 4 * 7 * N.MLP_NPARAM, flops=6 * rows * (80 * 256 + 256 * 256 + 256))


# ------------------------------------------------------------------ exact
# Vina's radii and type flags (1 hydrophobic, 2 acceptor, 4 donor) by XS type, its weights and cutoff
RADII = [1.1, 1.92, 1.9, 1.9, 1.8, 1.8, 1.8, 1.8, 1.7, 1.7, 1.7, 1.7, 1.5, 2.2, 2.1, 2.0, 1.8, 2.0, 2.2, 2.3, 1.2]
FLAGS = [0, 0, 1, 0, 0, 4, 2, 6, 0, 4, 2, 6, 1, 0, 0, 0, 1, 1, 1, 0, 4]


def _terms(d, hyd, hb):
    zero = torch.zeros_like(d)
    return (-0.035579 * torch.exp(-4.0 * d * d), -0.005156 * torch.exp(-((d - 3.0) / 2.0) ** 2),
            0.840245 * torch.clamp(d, max=0.0) ** 2,
            torch.where(hyd, -0.035069 * torch.clamp(1.5 - d, 0.0, 1.0), zero),
            torch.where(hb, -0.587439 * torch.clamp(-d / 0.7, 0.0, 1.0), zero))


def _pair_terms(xi, xj, ti, tj):
    """Vina terms of atoms xi (type ti) with xj, broadcast; zero from 8 A on and for hydrogens."""
    f = torch.tensor(FLAGS, device=xi.device)
    r = torch.tensor(RADII, dtype=torch.float64, device=xi.device)
    rr = ((xi - xj) ** 2).sum(-1)
    near = (rr < 64.0) & (ti > 0) & (tj > 0)
    d = torch.sqrt(torch.where(near, rr, torch.ones_like(rr))) - (r[ti] + r[tj])
    a, b = f[ti], f[tj]
    t = _terms(d, (a & b & 1) > 0, (((a >> 1) & (b >> 2)) | ((a >> 2) & (b >> 1))) % 2 > 0)
    return [torch.where(near, v, torch.zeros_like(v)) for v in t]


def _curl(e, cap):
    return torch.where(e > 0, e * cap / (cap + e.clamp(min=0.0)), e)


def _penalty(x, box):
    lo, hi = (torch.tensor(v, dtype=torch.float64, device=x.device) for v in (box.lo, box.hi))
    return ((lo - x).clamp(min=0.0) + (x - hi).clamp(min=0.0)).sum(-1)


def _rec64(receptor):
    return (torch.tensor(receptor.xyz, dtype=torch.float64, device="cuda"),
            torch.tensor(receptor.types, device="cuda").long())


def _maps64(receptor, box, types):
    rx, rt = _rec64(receptor)
    n = [int(round(float(h - l) / SPACING)) + 1 for l, h in zip(box.lo, box.hi)]
    ax = [np.float32(box.lo[d]) + np.float32(SPACING) * np.arange(n[d], dtype=np.float32) for d in range(3)]
    z, y, x = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    pts = torch.from_numpy(np.stack([x, y, z], -1).reshape(-1, 3)).cuda().double()
    maps = torch.zeros((len(types), pts.shape[0]), dtype=torch.float64, device="cuda")
    for at in range(0, pts.shape[0], 4096):
        p = pts[at:at + 4096]
        lo, hi = p.amin(0) - 8.001, p.amax(0) + 8.001
        keep = ((rx > lo) & (rx < hi)).all(1)
        for k, t in enumerate(types):
            tt = torch.full((1, 1), t, device="cuda")
            maps[k, at:at + 4096] = sum(_pair_terms(p[:, None], rx[None, keep], tt, rt[None, keep])).sum(1)
    return maps.view(len(types), n[2], n[1], n[0])


def _inter64(x, types, receptor, box, maps):
    """Receptor energy of each heavy atom at x [n, natom, 3], before the curl."""
    if maps is None:
        rx, rt = _rec64(receptor)
        return torch.stack([sum(_pair_terms(x[:, a, None], rx[None], types[a], rt[None])).sum(1)
                            for a in range(x.shape[1])], 1)
    slot = torch.tensor([DEFAULT_PROBE_TYPES.index(int(t)) if t > 0 else 0 for t in types.tolist()], device="cuda")
    n = torch.tensor([maps.shape[3], maps.shape[2], maps.shape[1]], device="cuda")
    g = (x - torch.tensor(box.lo, dtype=torch.float64, device="cuda")) / SPACING
    g = torch.minimum(g.clamp(min=0.0), (n - 1).double())
    i = torch.minimum(g.detach().floor().long(), n - 2)
    f = g - i
    e = 0.0
    for c in range(8):
        o = [c & 1, (c >> 1) & 1, c >> 2]
        w = 1.0
        for d in range(3):
            w = w * (f[..., d] if o[d] else 1.0 - f[..., d])
        e = e + w * maps[slot[None, :], i[..., 2] + o[2], i[..., 1] + o[1], i[..., 0] + o[0]]
    return e


def _energy_grad64(lig, x, centre, rv, receptor, box, maps):
    """Energy (curl cap 10, slope 1e6) and pose gradient of coordinates x [n, natom, 3]."""
    types = torch.tensor(lig.types, device="cuda").long()
    heavy = types > 0
    x = x.detach().requires_grad_(True)
    e = _curl(torch.where(heavy, _inter64(x, types, receptor, box, maps), 0.0), 10.0).sum(1)
    e = e + 1e6 * torch.where(heavy, _penalty(x, box), 0.0).sum(1)
    if lig.npair:
        i, j = torch.tensor(lig.pairs, device="cuda").long().T
        e = e + _curl(sum(_pair_terms(x[:, i], x[:, j], types[i], types[j])), 10.0).sum(1)
    (f,) = torch.autograd.grad(e.sum(), x)
    x = x.detach()
    f = torch.where(heavy[None, :, None], f, 0.0)
    tau = torch.linalg.cross(x - centre[:, None], f).sum(1)
    # orientation: J(v)^T tau, J the left Jacobian at the same rotation with its angle in [0, pi]
    ang = rv.norm(dim=1, keepdim=True)
    th = torch.remainder(ang, 2.0 * math.pi)
    sign = torch.where(th > math.pi, -1.0, 1.0)
    th = torch.where(th > math.pi, 2.0 * math.pi - th, th)
    v = rv * (sign * th / ang.clamp(min=1e-30))
    small = th < 1e-3
    t1 = torch.where(small, torch.ones_like(th), th)
    a = torch.where(small, 0.5 - th ** 2 / 24.0, (1.0 - torch.cos(t1)) / t1 ** 2)
    b = torch.where(small, 1.0 / 6.0 - th ** 2 / 120.0, (t1 - torch.sin(t1)) / t1 ** 3)
    vt = torch.linalg.cross(v, tau)
    g = [f.sum(1), tau - a * vt + b * torch.linalg.cross(v, vt)]
    for t in range(lig.ntors):
        frm, to = (int(k) for k in lig.axis[t])
        at = torch.tensor(lig.rot_atoms[lig.rot_start[t]:lig.rot_start[t + 1]], device="cuda").long()
        u = x[:, to] - x[:, frm]
        u = u / u.norm(dim=1, keepdim=True)
        g.append((torch.linalg.cross(x[:, at] - x[:, to, None], f[:, at]).sum(1) * u).sum(1, keepdim=True))
    return e.detach(), torch.cat(g, 1)


def _apply_posevecs64(lig, pv):
    x = torch.tensor(lig.coords, dtype=torch.float64, device="cuda").repeat(pv.shape[0], 1, 1)
    for t in range(lig.ntors):
        frm, to = (int(k) for k in lig.axis[t])
        at = torch.tensor(lig.rot_atoms[lig.rot_start[t]:lig.rot_start[t + 1]], device="cuda").long()
        ang = (pv[:, 7 + t] - float(lig.dihedrals[t]))[:, None, None]
        u = x[:, to] - x[:, frm]
        u = (u / u.norm(dim=1, keepdim=True))[:, None].expand(-1, len(at), -1)
        w = x[:, at] - x[:, to, None]
        x[:, at] = (torch.cos(ang) * w + torch.sin(ang) * torch.linalg.cross(u, w) +
                    (1.0 - torch.cos(ang)) * u * (u * w).sum(-1, keepdim=True) + x[:, to, None])
    q = pv[:, 3:7]
    w, v = q[:, :1, None], q[:, None, 1:].expand(-1, lig.natom, -1)
    x = x - x.mean(1, keepdim=True)
    # rotation by the quaternion as its matrix, whose entries are quadratic in it
    x = (w ** 2 - (v * v).sum(-1, keepdim=True)) * x + 2.0 * v * (v * x).sum(-1, keepdim=True) + \
        2.0 * w * torch.linalg.cross(v, x)
    return x + pv[:, None, :3]


def _exact_score(case, seed):
    lig = _score_ligand(case)
    receptor, box = _receptor(seed), S.docking_box()
    maps = _maps64(receptor, box, DEFAULT_PROBE_TYPES) if case["mode"] == "grid" else None
    pv = torch.from_numpy(_pose_vectors(case, seed)).cuda().double()
    es, gs = [], []
    step = 16384 if maps is not None else 512
    for at in range(0, pv.shape[0], step):
        p = pv[at:at + step]
        th = 2.0 * torch.acos(p[:, 3:4].clamp(-1.0, 1.0))
        s = torch.sqrt((1.0 - p[:, 3:4] ** 2).clamp(min=0.0))
        rv = p[:, 4:7] * torch.where(s > 1e-9, th / s.clamp(min=1e-9), torch.zeros_like(s))
        e, g = _energy_grad64(lig, _apply_posevecs64(lig, p), p[:, :3], rv, receptor, box, maps)
        es.append(e)
        gs.append(g)
    return dict(e=torch.cat(es), g=torch.cat(gs))


def _exact_poses(case, seed):
    ligands = _ligands(case, seed)
    nchain = case["nchain"]
    x, c, r, _ = (torch.from_numpy(v).cuda().double() for v in _pose_arrays(ligands, nchain, seed))
    receptor, box = _receptor(seed), S.docking_box()
    n = len(ligands) * nchain
    if case["kind"] == "energy_grad":
        maps = _maps64(receptor, box, DEFAULT_PROBE_TYPES) if case["mode"] == "grid" else None
        e, g = torch.zeros(n, dtype=torch.float64), torch.zeros((n, 64), dtype=torch.float64)
    else:
        rx, rt = _rec64(receptor)
        stride = max(l.natom for l in ligands)
        out4, decomp = torch.zeros((n, 4), dtype=torch.float64), torch.zeros((n, stride, 5), dtype=torch.float64)
    at = 0
    for k, lig in enumerate(ligands):
        xl = x[at:at + nchain * lig.natom * 3].view(nchain, lig.natom, 3)
        at += xl.numel()
        rows = slice(k * nchain, (k + 1) * nchain)
        if case["kind"] == "energy_grad":
            ek, gk = _energy_grad64(lig, xl, c[rows], r[rows], receptor, box, maps)
            e[rows], g[rows, :gk.shape[1]] = ek.cpu(), gk.cpu()
            continue
        types = torch.tensor(lig.types, device="cuda").long()
        heavy = types > 0
        terms = torch.stack([t.sum(2) for t in _pair_terms(xl[:, :, None], rx, types[:, None], rt)], -1)
        i, j = torch.tensor(lig.pairs, device="cuda").long().T
        intra = sum(_pair_terms(xl[:, i], xl[:, j], types[i], types[j])).sum(1)
        pen = 1e6 * torch.where(heavy, _penalty(xl, box), 0.0).sum(1)
        out4[rows] = torch.stack([intra, terms.sum((1, 2)), pen, torch.zeros_like(pen)], 1).cpu()
        decomp[rows, :lig.natom] = terms.cpu()
    return dict(e=e, g=g) if case["kind"] == "energy_grad" else dict(out4=out4, decomp=decomp)


def _exact_train(case, seed):
    """The step without the network's bf16 roundings."""
    bits, y, g, params = _train_data(case, seed)
    rows = (g.long()[:, None] * N.MLP_GROUP + torch.arange(N.MLP_GROUP, device="cuda")).view(-1)
    x = bits.view(torch.bfloat16)[rows].double()
    p = torch.from_numpy(params).cuda().double()
    w = p[:N.MLP_NPARAM].clone().requires_grad_(True)
    F, H = N.MLP_FEATURES, N.MLP_HIDDEN
    w1, b1, w2, b2, w3, b3 = torch.split(w, [F * H, H, H * H, H, H, 1])
    norm = p[N.MLP_NPARAM:]
    a = torch.relu((x - norm[:F]) * norm[F:] @ w1.view(F, H) + b1)
    out = torch.relu(a @ w2.view(H, H) + b2) @ w3 + b3
    lab = y[rows].double().view(-1, N.MLP_GROUP)
    res = out.view(-1, N.MLP_GROUP) - torch.minimum(lab, lab.amin(1, keepdim=True) + 6.0)
    loss = ((res - res.mean(1, keepdim=True)) ** 2).mean()
    (grad,) = torch.autograd.grad(loss, w)
    new = w.detach() - 1e-3 * grad / (grad.abs() + 1e-8)
    return dict(loss=loss.detach().view(1), params=torch.cat([new, norm]))


def exact(case, seed):
    kind = case["kind"]
    if kind == "score":
        return _exact_score(case, seed)
    if kind in ("energy_grad", "rescore"):
        return _exact_poses(case, seed)
    if kind == "grids":
        return _maps64(_receptor(seed, case["n_rec"]), S.docking_box(size=case["box"]), _probe_types(case))
    if kind == "train":
        return _exact_train(case, seed)
    return None
