"""Drop-in for Uni-Dock2's ``unidock_engine.api.python.pipeline`` module.

``DockingPipeline`` keeps the reference's keyword-only constructor, defaults and
methods (unidock/unidock_engine/api/python/pipeline.cpp:56-217): set_receptor(list),
add_ligands(dict), run(). run() parses the same engine-JSON objects
(src/format/rapidjson_parser.cpp semantics, see ``unidock_engine.topology``),
applies the search-mode and task presets (src/screening/core.cpp:65-209), splits
the ligands into the reference's size groups and memory-bounded batches
(src/screening/screening.cpp:17-219), docks each batch on the GPU through
libud2.so and writes ``<output_dir>/<name_json>_<batch_id>.json`` in the
reference's output format (src/format/json.cpp:88-191). Failures raise
RuntimeError("Core pipeline failed.") as the reference does (pipeline.cpp:141-143).
"""
from __future__ import annotations

import json
import logging
import math
import os
import time

import numpy as np

from ... import _native as N
from ...engine import DockEngine, DockParams, heuristic_opt_steps
from ...topology import Box, XS_H, ligand_from_json, receptor_from_json

log = logging.getLogger("unidock_engine")

# CoreInputDefaults (src/screening/core.h:9-36) with DockParam's values (src/model/model.h:151-168)
DEFAULTS = dict(
    output_dir="./res_ud2", task="screen", search_mode="balance", exhaustiveness=512, randomize=True,
    mc_steps=20, opt_steps=-1, refine_steps=5, num_pose=10, rmsd_limit=1.0, energy_range=10.0, seed=12345,
    bias="no", bias_k=0.1, constraint_docking=False, use_tor_lib=False, energy_decomp=False, gpu_device_id=0,
    name_json="from_python_obj", max_gpu_mem=0,
)

# size groups of run_screening (src/screening/screening.h:19-26): (max atoms, max torsions)
GROUPS = ((40, 8), (80, 16), (120, 24), (160, 32))
MAX_BATCH = 1000  # screening.cpp:183
MAX_SAFE = 1e6    # json.cpp:78-85


def apply_search_mode(p: dict) -> None:
    """apply_search_mode, src/screening/core.cpp:65-84."""
    mode = p["search_mode"]
    if mode in ("", "free"):
        return
    presets = {"fast": (128, 20), "balance": (256, 30), "detail": (512, 40)}
    if mode not in presets:
        raise ValueError(f"Not supported search_mode: {mode} doesn't belong to (fast, balance, detail, free)")
    p["exhaustiveness"], p["mc_steps"] = presets[mode]
    p["opt_steps"] = -1


def apply_task(p: dict) -> None:
    """Task presets of core_pipeline, src/screening/core.cpp:165-209."""
    t = p["task"]
    if t == "screen":
        return
    if t == "score":
        p.update(randomize=False, exhaustiveness=1, mc_steps=0, opt_steps=0, refine_steps=0, num_pose=1,
                 energy_range=999.0, rmsd_limit=999.0)
    elif t == "mc":
        p.update(randomize=True, opt_steps=0, refine_steps=0)
    elif t == "randomize":
        p.update(randomize=True, mc_steps=0, opt_steps=0, refine_steps=0, num_pose=p["exhaustiveness"],
                 energy_range=1e9, rmsd_limit=0.0)
    elif t == "optimize":
        p.update(randomize=False, exhaustiveness=1, mc_steps=0, opt_steps=0, num_pose=1, energy_range=1e9,
                 rmsd_limit=0.0)
    else:
        raise ValueError(f"Not supported task: {t} doesn't belong to (screen, score, mc, randomize, optimize)")


def group_ligands(ligands) -> list:
    """group_flex_mols, src/screening/screening.cpp:17-41: index lists per size group (+ overflow)."""
    groups = [[] for _ in range(len(GROUPS) + 1)]
    for i, l in enumerate(ligands):
        for g, (na, nt) in enumerate(GROUPS):
            if l.natom <= na and l.ntors <= nt:
                groups[g].append(i)
                break
        else:
            groups[-1].append(i)
    return groups


MIB = 1048576


class BatchSize:
    """Device memory of one batch in this library's layout (the counterpart of predict_gpu_flex,
    src/screening/screening.cpp:53-127): pose buffers, topology, clustering / selection arrays."""

    def __init__(self):
        self.n_lig = self.natom = self.ntors = self.npair = self.nbias = self.nstep = 0

    def add(self, lig) -> "BatchSize":
        b = BatchSize()
        b.n_lig, b.natom, b.ntors = self.n_lig + 1, self.natom + lig.natom, self.ntors + lig.ntors
        b.npair = self.npair + lig.npair
        b.nbias = self.nbias + (0 if lig.bias is None else len(lig.bias))
        b.nstep = self.nstep + self.pair_steps(lig)
        return b

    @staticmethod
    def pair_steps(lig) -> int:
        """Steps of the ligand's pair table, 1 KB each: two diagonals a step up to 32 atoms; up to 64 atoms
        about what the pairs and the busiest atom's pairs (four a step) need, which holds what the
        packing takes; none for larger ligands."""
        if lig.npair == 0 or lig.natom > 64:
            return 0
        if lig.natom <= 32:
            return (lig.natom // 2 + 1) // 2
        return max(lig.npair // 50, (int(np.bincount(np.asarray(lig.pairs).reshape(-1)).max()) + 3) // 4) + 3

    def bytes(self, nchain: int) -> int:
        poses = nchain * (3 * self.natom + self.ntors) * 4 + self.n_lig * nchain * 7 * 4
        topo = self.natom * 48 + self.ntors * 64 + self.npair * 8 + self.nbias * 32 + self.n_lig * 128 + self.nstep * 1024
        return poses + topo + self.n_lig * nchain * 4 * 3


def memory_limit_mb(user_mb: int) -> int:
    """decide_memory_limit_mb (src/screening/core.cpp:32-63): 95 % of the device's free memory,
    capped by 95 % of the host's memory and by the caller's limit when that is positive."""
    free, _ = N.device_memory()
    lim = int((free // MIB) * 0.95)
    ram = int((os.sysconf("SC_PHYS_PAGES") * os.sysconf("SC_PAGE_SIZE") // MIB) * 0.95)
    lim = min(lim, ram)
    if user_mb > 0 and user_mb < lim:
        lim = user_mb
    return lim


def scene_bytes(receptor, scene) -> int:
    """The scene's device memory (predict_gpu_fix, screening.cpp:44-51): receptor atoms, grid maps
    and their cell-major copy, reach lists."""
    n, _, _, nt = scene.grid_info()
    n0, n1, n2 = (int(v) for v in n)
    maps = nt * n0 * n1 * n2 * 4 + (nt * (n0 - 1) * (n1 - 1) * (n2 - 1) * 32 if nt else 0)
    return receptor.natom * 16 + maps + scene.reach_bytes()


def memory_batches(ligands, group, nchain: int, limit_mb: int):
    """Batches of one size group: at most 1,000 ligands each, with the estimated device memory
    under the budget (run_screening, screening.cpp:168-196)."""
    done = 0
    while done < len(group):
        batch, est = [], BatchSize()
        while done + len(batch) < len(group):
            i = group[done + len(batch)]
            nxt = est.add(ligands[i])
            if len(batch) >= MAX_BATCH or nxt.bytes(nchain) // MIB >= limit_mb:
                break
            batch.append(i)
            est = nxt
        if not batch:
            raise RuntimeError(f"Not enough GPU Memory to process at least one ligand in a batch of group {group[done]}")
        done += len(batch)
        yield batch


def fmt_float(v: float) -> str:
    """A float as the reference's rapidjson writer prints it: shortest round-trip digits of the
    double value, at most 3 decimals (extra digits dropped, not rounded), at least one."""
    v = float(v)
    if v != v or math.isinf(v):
        v = MAX_SAFE
    v = min(max(v, -MAX_SAFE), MAX_SAFE)
    r = repr(v)
    if "e" in r or "E" in r:
        r = f"{v:.20f}".rstrip("0")
    if "." not in r:
        r += ".0"
    ip, fp = r.split(".")
    fp = fp[:3].rstrip("0") or "0"
    return f"{ip}.{fp}"


def dumps_poses(results) -> str:
    """write_poses_to_json, src/format/json.cpp:88-191 (compact, no whitespace); a pose
    with a per-atom energy decomposition gets its "decomp" member (json.cpp:134-147)."""
    parts = []
    for r in results:
        poses = []
        for k in range(len(r.energies)):
            e = ",".join(fmt_float(x) for x in r.energies[k])
            c = ",".join(fmt_float(x) for x in np.asarray(r.coords[k], np.float32))
            d = ",".join(fmt_float(x) for x in np.asarray(r.dihedrals[k], np.float32))
            extra = ""
            if k < len(getattr(r, "decomp", ())):
                extra = ',"decomp":[' + ",".join(
                    "[" + ",".join(fmt_float(x) for x in row) + "]" for row in np.asarray(r.decomp[k], np.float32)) + "]"
            poses.append('{"energy":[' + e + '],"coords":[' + c + '],"dihedrals":[' + d + "]" + extra + "}")
        parts.append(json.dumps(r.name, ensure_ascii=False) + ":[" + ",".join(poses) + "]")
    return "{" + ",".join(parts) + "}"


def write_json_with_retry(path: str, text: str, retries: int = 5, wait: float = 5.0) -> None:
    """dump_poses, src/task/DockTask.cpp:285-334: write, fsync, check the last byte is '}',
    retry with doubling back-off."""
    for attempt in range(1, retries + 1):
        try:
            with open(path, "w") as f:
                f.write(text)
                f.flush()
                os.fsync(f.fileno())
            with open(path, "rb") as f:
                f.seek(-1, os.SEEK_END)
                if f.read(1) != b"}":
                    raise IOError("JSON file is incomplete.")
            return
        except Exception as e:  # noqa: BLE001 - any I/O failure is retried
            if attempt == retries:
                raise
            log.warning("attempt %d to write %s failed: %s; retrying in %.0f s", attempt, path, e, wait)
            time.sleep(wait)
            wait *= 2


class DockingPipeline:
    """Uni-Dock2 molecular docking pipeline on an MI355X."""

    def __init__(self, *, output_dir=DEFAULTS["output_dir"], center_x, center_y, center_z, size_x, size_y, size_z,
                 task=DEFAULTS["task"], search_mode=DEFAULTS["search_mode"],
                 exhaustiveness=DEFAULTS["exhaustiveness"], randomize=DEFAULTS["randomize"],
                 mc_steps=DEFAULTS["mc_steps"], opt_steps=DEFAULTS["opt_steps"],
                 refine_steps=DEFAULTS["refine_steps"], num_pose=DEFAULTS["num_pose"],
                 rmsd_limit=DEFAULTS["rmsd_limit"], energy_range=DEFAULTS["energy_range"], seed=DEFAULTS["seed"],
                 bias=DEFAULTS["bias"], bias_k=DEFAULTS["bias_k"], constraint_docking=DEFAULTS["constraint_docking"],
                 use_tor_lib=DEFAULTS["use_tor_lib"], energy_decomp=DEFAULTS["energy_decomp"],
                 gpu_device_id=DEFAULTS["gpu_device_id"], name_json=DEFAULTS["name_json"],
                 max_gpu_mem=DEFAULTS["max_gpu_mem"]):
        self.box = Box.from_center_size((center_x, center_y, center_z), (size_x, size_y, size_z))
        self.center_size = dict(center_x=float(center_x), center_y=float(center_y), center_z=float(center_z),
                                size_x=float(size_x), size_y=float(size_y), size_z=float(size_z))
        self.params = dict(output_dir=str(output_dir), task=task, search_mode=search_mode,
                           exhaustiveness=int(exhaustiveness), randomize=bool(randomize), mc_steps=int(mc_steps),
                           opt_steps=int(opt_steps), refine_steps=int(refine_steps), num_pose=int(num_pose),
                           rmsd_limit=float(rmsd_limit), energy_range=float(energy_range), seed=int(seed),
                           bias=bias, bias_k=float(bias_k), constraint_docking=bool(constraint_docking),
                           use_tor_lib=bool(use_tor_lib), energy_decomp=bool(energy_decomp),
                           gpu_device_id=int(gpu_device_id), name_json=str(name_json), max_gpu_mem=int(max_gpu_mem))
        self.json_data: dict = {}
        self.output_files: list = []
        self.inter_mode = N.MODE_GRID
        # "native": the whole run in libud2.so (ud2_run_json); "python": the same pipeline driven
        # from Python over the kernel-level entry points (core_pipeline below)
        self.host = "native"
        # search method, not one of the reference's arguments: "plain" (the reference's MC) or
        # "learned" (the learned-proposal search with the network in proposal_weights, default the
        # packaged one, and its knobs: n_cand, top_k, n_start, sel_temp; 0 = the library's defaults)
        self.search = "plain"
        self.proposal_weights = None
        self.learned = dict(n_cand=0, top_k=0, n_start=0, sel_temp=0.0)

    def set_receptor(self, receptor_info: list) -> None:
        self.json_data["receptor"] = receptor_info

    def add_ligands(self, ligands_info: dict) -> None:
        for k, v in ligands_info.items():
            self.json_data[k] = v

    def run(self) -> None:
        try:
            self._run()
        except Exception as e:  # the reference logs and returns 1 from core_pipeline (core.cpp:218-222)
            log.critical("Core pipeline failed: %s", e)
            raise RuntimeError("Core pipeline failed.") from e

    # ------------------------------------------------------------------
    def _run(self) -> None:
        # the reference serialises the cached objects to JSON text and hands the text to its C++
        # core_pipeline (pipeline.cpp:120-145)
        text = json.dumps(self.json_data, ensure_ascii=False)
        if self.search not in ("plain", "learned"):
            raise ValueError(f"unknown search {self.search!r} (plain, learned)")
        if self.host == "python":
            if self.search != "plain":
                raise ValueError("the Python-driven pipeline runs the plain search only")
            self.output_files.extend(core_pipeline(dict(self.params), self.box, json.loads(text), self.inter_mode))
            return
        if self.host != "native":
            raise ValueError(f"unknown host {self.host!r} (native, python)")
        proposal = None
        if self.search == "learned":
            from ... import proposal as LP
            proposal = LP.load(self.proposal_weights or LP.WEIGHTS)
        self.output_files.extend(run_native(dict(self.params, **self.center_size), text, self.inter_mode, proposal,
                                            self.learned))


def output_path(p: dict, batch_id: int) -> str:
    """<output_dir>/<name_json>_<batch_id>.json; an empty directory is the working directory
    (gen_filepath, src/myutils/myio.cpp:7-13)."""
    name = f"{p['name_json']}_{batch_id}.json"
    return os.path.join(p["output_dir"], name) if p["output_dir"] else name


def run_native(p: dict, text: str, inter_mode: int = N.MODE_GRID, proposal=None, learned=None) -> list:
    """core_pipeline in libud2.so (ud2_run_json) over an engine-JSON text; ``p`` holds
    DockingPipeline's keyword arguments with the box centre and size; ``proposal`` (network
    parameters) selects the learned search. Returns the files written."""
    t0 = time.time()
    n = N.run_json(p, text, inter_mode, proposal, learned)
    log.info("%d batch(es) docked in %.1f ms", n, (time.time() - t0) * 1e3)
    return [output_path(p, k) for k in range(1, n + 1)]


def core_pipeline(p: dict, box: Box, doc: dict, inter_mode: int = N.MODE_GRID) -> list:
    """core_pipeline, src/screening/core.cpp:100-223, over an engine-JSON document (receptor under
    "receptor", one member per ligand, optional "score"): bias check, search-mode and task presets,
    size groups and batches of at most 1,000 ligands within the device-memory budget, one docking
    run and one output file per batch.
    ``p`` holds DockingPipeline's keyword arguments. Returns the files written; raises on failure.
    This is the Python-driven twin of ud2_run_json (DockingPipeline.host = "python"); both make
    the same kernel calls with the same arguments and write the same bytes."""
    p = dict(p)
    if p["bias"] not in ("no", "pos", "align"):  # apply_bias, core.cpp:86-97
        raise ValueError(f"Not supported bias: {p['bias']} doesn't belong to (no, pos, align)")
    apply_search_mode(p)
    if p["opt_steps"] < 0:
        p["opt_steps"] = -1
    if p["constraint_docking"]:  # prepare_context_by_input, core.cpp:142-146
        p["randomize"] = False
    apply_task(p)
    if p["output_dir"]:
        os.makedirs(p["output_dir"], exist_ok=True)
    N.check(N.lib().ud2_set_device(p["gpu_device_id"]), "ud2_set_device")
    receptor = receptor_from_json(doc.get("receptor", []), box)
    ligands = [ligand_from_json(k, v, p["use_tor_lib"]) for k, v in doc.items()
               if k not in ("score", "receptor")]
    if not ligands:
        log.error("No flexible molecules are found")
        return []
    eng = DockEngine(receptor, box, mode=inter_mode)
    eng.ensure_types(ligands)
    limit_mb = memory_limit_mb(p["max_gpu_mem"])
    # the reach lists are given up where the batches would otherwise not hold every ligand
    largest = max(BatchSize().add(lig).bytes(p["exhaustiveness"]) for lig in ligands)
    if largest // MIB >= limit_mb - scene_bytes(receptor, eng.scene) // MIB:
        eng.scene.reach_bytes(keep=False)
    fix_mb = scene_bytes(receptor, eng.scene) // MIB
    if limit_mb < fix_mb:
        raise RuntimeError(f"GPU memory ({limit_mb} MB) is not enough for the receptor ({fix_mb} MB)")
    files = []
    batch_id = 0
    opt_steps = p["opt_steps"]
    for group in group_ligands(ligands):
        for idx in memory_batches(ligands, group, p["exhaustiveness"], limit_mb - fix_mb):
            batch = [ligands[i] for i in idx]
            batch_id += 1
            if opt_steps == -1:  # heuristic of the first batch persists (screening.cpp:206-208)
                opt_steps = heuristic_opt_steps(max(l.natom for l in batch))
            prm = DockParams(nchain=p["exhaustiveness"], mc_steps=p["mc_steps"], opt_steps=opt_steps,
                             refine_steps=p["refine_steps"], num_pose=p["num_pose"],
                             rmsd_limit=p["rmsd_limit"], energy_range=p["energy_range"], seed=p["seed"],
                             randomize=p["randomize"], mode=inter_mode, energy_decomp=p["energy_decomp"])
            t0 = time.time()
            ls = N.LigSet(batch, bias=p["bias"], bias_k=p["bias_k"], constraint=p["constraint_docking"])
            results, _ = eng.dock(ls, prm)
            path = output_path(p, batch_id)
            write_json_with_retry(path, dumps_poses(results))
            files.append(path)
            log.info("Batch %d (%d ligands) running time: %.1f ms", batch_id, len(batch),
                     (time.time() - t0) * 1e3)
    return files
