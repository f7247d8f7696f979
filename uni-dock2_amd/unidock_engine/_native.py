"""ctypes binding of libud2.so, the HIP engine (C ABI in include/ud2.h).

The library is built in-tree (``unidock_engine/lib/libud2.so``) by
``__graft_entry__.build()`` / ``python -m unidock_engine.build``. Loading fails
loudly when it is missing: the engine has no CPU fallback.
"""
from __future__ import annotations

import ctypes as C
import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "lib", "libud2.so")

UD2_OK = 0
MODE_DIRECT = 0
MODE_GRID = 1
MAX_ATOMS = 256
MAX_TORSIONS = 57
MLP_FEATURES = 80
MLP_HIDDEN = 256
MLP_GROUP = 16
MLP_NPARAM = 86785
MLP_NNORM = 160
POLICY_PLAIN, POLICY_EXACT, POLICY_LEARNED, POLICY_COLLECT = 0, 1, 2, 3
SEARCH_PLAIN, SEARCH_LEARNED = 0, 1


class Ud2Error(RuntimeError):
    pass


class LigandBatch(C.Structure):
    _fields_ = [("n_lig", C.c_int32)] + [(n, C.c_void_p) for n in (
        "atom_off_h", "tors_off_h", "pair_off_h", "types_h", "xyz_h", "axis_h", "dihe0_h", "rot_off_h",
        "rot_atoms_h", "range_off_h", "ranges_h", "pairs_h")]


class Poses(C.Structure):
    _fields_ = [("x_d", C.c_void_p), ("c_d", C.c_void_p), ("rv_d", C.c_void_p), ("dihe_d", C.c_void_p),
                ("e_d", C.c_void_p), ("nchain", C.c_int32)]


class McParams(C.Structure):
    _fields_ = [("mc_steps", C.c_int32), ("opt_steps", C.c_int32), ("randomize", C.c_int32),
                ("seed", C.c_uint32), ("mode", C.c_int32), ("lig_index_base", C.c_int32),
                ("stats_d", C.c_void_p)]


class Adam(C.Structure):
    _fields_ = [("lr", C.c_float), ("beta1", C.c_float), ("beta2", C.c_float), ("eps", C.c_float)]


class LmcParams(C.Structure):
    _fields_ = [("mc", McParams), ("policy", C.c_int32), ("n_cand", C.c_int32), ("top_k", C.c_int32),
                ("sel_temp", C.c_float), ("n_start", C.c_int32), ("collect_x_d", C.c_void_p), ("collect_y_d", C.c_void_p), ("collect_e0_d", C.c_void_p)]


class RunParams(C.Structure):
    """ud2_run_params: the run options of ud2_create (CoreInput / DockingPipeline's arguments)."""
    _fields_ = [("center", C.c_float * 3), ("size", C.c_float * 3), ("task", C.c_char_p),
                ("search_mode", C.c_char_p), ("exhaustiveness", C.c_int32), ("randomize", C.c_int32),
                ("mc_steps", C.c_int32), ("opt_steps", C.c_int32), ("refine_steps", C.c_int32),
                ("num_pose", C.c_int32), ("rmsd_limit", C.c_float), ("energy_range", C.c_float),
                ("seed", C.c_int64), ("bias", C.c_char_p), ("bias_k", C.c_float), ("constraint_docking", C.c_int32),
                ("use_tor_lib", C.c_int32), ("energy_decomp", C.c_int32), ("gpu_device_id", C.c_int32),
                ("max_gpu_mem", C.c_int32), ("inter_mode", C.c_int32), ("search", C.c_int32),
                ("proposal_h", C.c_void_p), ("n_cand", C.c_int32), ("top_k", C.c_int32), ("n_start", C.c_int32),
                ("sel_temp", C.c_float)]


class DockParams(C.Structure):
    """ud2_dock_params: one batch of DockTask::run over a resident ligand set."""
    _fields_ = [("nchain", C.c_int32), ("mc_steps", C.c_int32), ("opt_steps", C.c_int32),
                ("refine_steps", C.c_int32), ("num_pose", C.c_int32), ("rmsd_limit", C.c_float),
                ("energy_range", C.c_float), ("seed", C.c_uint32), ("randomize", C.c_int32), ("mode", C.c_int32),
                ("energy_decomp", C.c_int32), ("search", C.c_int32), ("n_cand", C.c_int32), ("top_k", C.c_int32),
                ("n_start", C.c_int32), ("sel_temp", C.c_float)]


class DockOut(C.Structure):
    """ud2_dock_out: caller-owned host arrays for num_pose poses per ligand."""
    _fields_ = [(n, C.c_void_p) for n in ("n_out_h", "chain_h", "energy_h", "coords_h", "dihedrals_h", "decomp_h",
                                          "search_ms_h", "stats_h")]


_lib = None
_torch_first = None  # whether torch's HIP runtime was already loaded when the library was


def lib():
    """The loaded library; raises if it has not been built.

    The library needs only the HIP runtime, and loads without torch. torch's wheel ships its own
    copy of that runtime under the same soname, and whichever copy loads first serves the whole
    process: when torch is already imported the library binds to torch's copy, so torch tensors and
    streams work with it; otherwise it binds to ROCm's, and torch (whose copy would then be shadowed)
    must not be used for device memory in the same process (``stream_ptr`` and ``PoseBuffers``
    check this)."""
    global _lib, _torch_first
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise Ud2Error(f"libud2.so not built ({LIB_PATH}); run __graft_entry__.build()")
    _torch_first = "torch" in sys.modules
    L = C.CDLL(LIB_PATH)
    vp, i32, i64, f32 = C.c_void_p, C.c_int32, C.c_int64, C.c_float
    sig = {
        "ud2_version": (C.c_char_p, []),
        "ud2_last_error": (C.c_char_p, []),
        "ud2_device_count": (C.c_int, [vp]),
        "ud2_set_device": (C.c_int, [i32]),
        "ud2_synchronize": (C.c_int, []),
        "ud2_device_memory": (C.c_int, [vp, vp]),
        "ud2_scene_create": (C.c_int, [vp, vp, i32, vp, vp, vp]),
        "ud2_scene_build_grids": (C.c_int, [vp, f32, vp, i32]),
        "ud2_scene_set_grids": (C.c_int, [vp, vp, vp, f32, vp, i32, vp]),
        "ud2_scene_grid_info": (C.c_int, [vp, vp, vp, vp, vp]),
        "ud2_scene_download_maps": (C.c_int, [vp, vp]),
        "ud2_scene_gather_probe": (C.c_int, [vp, i64, i64, C.c_uint32, vp, vp]),
        "ud2_scene_reach": (C.c_int, [vp, C.c_int32, vp]),
        "ud2_scene_destroy": (C.c_int, [vp]),
        "ud2_valu_probe": (C.c_int, [i64, i32, vp, vp]),
        "ud2_ligset_create": (C.c_int, [vp, vp]),
        "ud2_ligset_destroy": (C.c_int, [vp]),
        "ud2_ligset_set_bias": (C.c_int, [vp, i32, f32, vp, vp]),
        "ud2_ligset_set_constraint": (C.c_int, [vp, i32]),
        "ud2_ligset_pose_layout": (C.c_int, [vp, i32, vp, vp, vp]),
        "ud2_ligset_sizes": (C.c_int, [vp, vp, vp, vp]),
        "ud2_dock": (C.c_int, [vp, vp, vp, vp, vp, vp]),
        "ud2_init_poses": (C.c_int, [vp, vp, vp]),
        "ud2_score_posevecs": (C.c_int, [vp, vp, i32, i64, vp, vp, vp, i32, f32, f32, vp]),
        "ud2_energy_grad": (C.c_int, [vp, vp, vp, vp, i32, i32, f32, f32, vp, vp, vp]),
        "ud2_pose_update": (C.c_int, [vp, vp, vp, i32, vp, f32, vp]),
        "ud2_line_search": (C.c_int, [vp, vp, vp, vp, i32, i32, f32, f32, vp, vp, vp]),
        "ud2_optimize": (C.c_int, [vp, vp, vp, vp, i32, i32, i32, f32, f32, vp, vp]),
        "ud2_mc": (C.c_int, [vp, vp, vp, vp, vp]),
        "ud2_mc_noalloc": (C.c_int, [vp, vp, vp, vp, vp]),
        "ud2_set_tile_policy": (C.c_int, [i32, i32]),
        "ud2_tune_info": (C.c_int, [vp, vp, vp, vp]),
        "ud2_autotune": (C.c_int, [vp, vp, vp, i32, C.c_char_p, vp]),
        "ud2_cluster": (C.c_int, [vp, vp, f32, vp, vp, vp]),
        "ud2_final_score": (C.c_int, [vp, vp, vp, vp, i32, vp, vp]),
        "ud2_score_decomp": (C.c_int, [vp, vp, vp, vp, i32, i32, vp, vp]),
        "ud2_mlp_create": (C.c_int, [vp, vp]),
        "ud2_mlp_set_params": (C.c_int, [vp, vp]),
        "ud2_mlp_get_params": (C.c_int, [vp, vp]),
        "ud2_mlp_destroy": (C.c_int, [vp]),
        "ud2_mlp_forward": (C.c_int, [vp, vp, vp, i32, vp, vp]),
        "ud2_mlp_backward": (C.c_int, [vp, vp, vp, i32, vp, vp, vp]),
        "ud2_mlp_train_step": (C.c_int, [vp, vp, vp, vp, i32, vp, vp, vp]),
        "ud2_features": (C.c_int, [vp, vp, vp, vp, i32, vp, vp]),
        "ud2_lmc": (C.c_int, [vp, vp, vp, vp, vp, vp]),
        "ud2_create": (C.c_int, [vp, vp]),
        "ud2_run_json": (C.c_int, [vp, C.c_char_p, C.c_size_t, C.c_char_p, C.c_char_p, vp]),
        "ud2_destroy": (C.c_int, [vp]),
    }
    for name, (res, args) in sig.items():
        fn = getattr(L, name)
        fn.restype = res
        fn.argtypes = args
    _lib = L
    return L


EXPORTED = (
    "ud2_version", "ud2_last_error", "ud2_device_count", "ud2_set_device", "ud2_synchronize", "ud2_device_memory",
    "ud2_scene_create",
    "ud2_scene_build_grids", "ud2_scene_set_grids", "ud2_scene_grid_info", "ud2_scene_download_maps",
    "ud2_scene_gather_probe", "ud2_valu_probe", "ud2_scene_reach", "ud2_scene_destroy", "ud2_ligset_create", "ud2_ligset_destroy", "ud2_ligset_set_bias",
    "ud2_ligset_set_constraint", "ud2_ligset_pose_layout", "ud2_ligset_sizes", "ud2_dock", "ud2_init_poses",
    "ud2_score_posevecs", "ud2_energy_grad", "ud2_pose_update", "ud2_line_search", "ud2_optimize", "ud2_mc", "ud2_mc_noalloc",
    "ud2_set_tile_policy", "ud2_tune_info", "ud2_autotune",
    "ud2_cluster", "ud2_final_score", "ud2_score_decomp", "ud2_mlp_create", "ud2_mlp_set_params", "ud2_mlp_get_params",
    "ud2_mlp_destroy", "ud2_mlp_forward", "ud2_mlp_backward", "ud2_mlp_train_step", "ud2_features", "ud2_lmc",
    "ud2_create", "ud2_run_json", "ud2_destroy",
)


def check(rc: int, what: str = "") -> None:
    if rc != UD2_OK:
        msg = lib().ud2_last_error().decode(errors="replace")
        raise Ud2Error(f"{what or 'ud2 call'} failed (code {rc}): {msg}")


def _ptr(a: np.ndarray):
    return C.c_void_p(a.ctypes.data)


class Scene:
    """Receptor + box (+ grid maps) on the device."""

    def __init__(self, receptor, box):
        xyz = np.ascontiguousarray(receptor.xyz, dtype=np.float32).reshape(-1)
        ty = np.ascontiguousarray(receptor.types, dtype=np.int32)
        lo = np.ascontiguousarray(box.lo, dtype=np.float32)
        hi = np.ascontiguousarray(box.hi, dtype=np.float32)
        self.box = box
        self.h = C.c_void_p()
        check(lib().ud2_scene_create(_ptr(xyz), _ptr(ty), int(ty.size), _ptr(lo), _ptr(hi), C.byref(self.h)),
              "ud2_scene_create")

    def build_grids(self, spacing: float, probe_types) -> None:
        pt = np.ascontiguousarray(probe_types, dtype=np.int32)
        check(lib().ud2_scene_build_grids(self.h, float(spacing), _ptr(pt), int(pt.size)), "ud2_scene_build_grids")

    def set_grids(self, n, origin, spacing, probe_types, maps) -> None:
        nn = np.ascontiguousarray(n, dtype=np.int32)
        org = np.ascontiguousarray(origin, dtype=np.float32)
        pt = np.ascontiguousarray(probe_types, dtype=np.int32)
        m = np.ascontiguousarray(maps, dtype=np.float32)
        check(lib().ud2_scene_set_grids(self.h, _ptr(nn), _ptr(org), float(spacing), _ptr(pt), int(pt.size), _ptr(m)),
              "ud2_scene_set_grids")

    def grid_info(self):
        n = np.zeros(3, dtype=np.int32)
        org = np.zeros(3, dtype=np.float32)
        sp = C.c_float()
        nt = C.c_int32()
        check(lib().ud2_scene_grid_info(self.h, _ptr(n), _ptr(org), C.byref(sp), C.byref(nt)), "ud2_scene_grid_info")
        return n, org, sp.value, nt.value

    def download_maps(self) -> np.ndarray:
        n, _, _, nt = self.grid_info()
        out = np.zeros((nt, n[2], n[1], n[0]), dtype=np.float32)
        check(lib().ud2_scene_download_maps(self.h, _ptr(out)), "ud2_scene_download_maps")
        return out

    def reach_bytes(self, keep: bool = True) -> int:
        """Device memory of the reach lists; keep=False frees them (the same results without them)."""
        n = C.c_int64()
        check(lib().ud2_scene_reach(self.h, int(keep), C.byref(n)), "ud2_scene_reach")
        return n.value

    def close(self):
        if self.h:
            lib().ud2_scene_destroy(self.h)
            self.h = C.c_void_p()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def pack_ligands(ligands) -> dict:
    """CSR arrays of a ligand list in the layout of ud2_ligand_batch."""
    n = len(ligands)
    atom_off = np.zeros(n + 1, dtype=np.int32)
    tors_off = np.zeros(n + 1, dtype=np.int32)
    pair_off = np.zeros(n + 1, dtype=np.int32)
    for i, l in enumerate(ligands):
        atom_off[i + 1] = atom_off[i] + l.natom
        tors_off[i + 1] = tors_off[i] + l.ntors
        pair_off[i + 1] = pair_off[i] + l.npair
    types = np.concatenate([l.types for l in ligands]).astype(np.int32)
    xyz = np.concatenate([l.coords.reshape(-1) for l in ligands]).astype(np.float32)
    axis = np.concatenate([l.axis.reshape(-1) for l in ligands] + [np.zeros(0, np.int32)]).astype(np.int32)
    dihe0 = np.concatenate([l.dihedrals for l in ligands] + [np.zeros(0, np.float32)]).astype(np.float32)
    rot_off = [0]
    rot_atoms = []
    range_off = [0]
    ranges = []
    for l in ligands:
        for t in range(l.ntors):
            r = l.rot_atoms[l.rot_start[t]:l.rot_start[t + 1]]
            rot_atoms.append(r)
            rot_off.append(rot_off[-1] + len(r))
            q = l.ranges[l.range_start[t]:l.range_start[t + 1]]
            ranges.append(q.reshape(-1))
            range_off.append(range_off[-1] + q.shape[0])
    pairs = np.concatenate([l.pairs.reshape(-1) for l in ligands] + [np.zeros(0, np.int32)]).astype(np.int32)
    return dict(
        atom_off=atom_off, tors_off=tors_off, pair_off=pair_off, types=types, xyz=xyz, axis=axis, dihe0=dihe0,
        rot_off=np.asarray(rot_off, dtype=np.int32),
        rot_atoms=(np.concatenate(rot_atoms) if rot_atoms else np.zeros(0)).astype(np.int32),
        range_off=np.asarray(range_off, dtype=np.int32),
        ranges=(np.concatenate(ranges) if ranges else np.zeros(0)).astype(np.float32),
        pairs=pairs,
    )


BIAS_TYPES = {"no": 0, "pos": 1, "align": 2}  # UD2_BIAS_NO / POS / ALIGN


class LigSet:
    """A batch of ligand topologies on the device.

    ``bias`` ("no", "pos", "align") and ``bias_k`` select the bias term over the
    ligands' bias sites (``Ligand.bias_start`` / ``Ligand.bias``);
    ``constraint`` turns on constraint docking (no rigid degrees of freedom).
    """

    def __init__(self, ligands, bias: str = "no", bias_k: float = 0.1, constraint: bool = False):
        self.ligands = list(ligands)
        self.arrays = pack_ligands(self.ligands)
        a = {k: (v if v.size else np.zeros(1, v.dtype)) for k, v in self.arrays.items()}
        self._keep = a
        b = LigandBatch(len(self.ligands), *[C.c_void_p(a[k].ctypes.data) for k in (
            "atom_off", "tors_off", "pair_off", "types", "xyz", "axis", "dihe0", "rot_off", "rot_atoms",
            "range_off", "ranges", "pairs")])
        self.h = C.c_void_p()
        check(lib().ud2_ligset_create(C.byref(b), C.byref(self.h)), "ud2_ligset_create")
        if bias not in BIAS_TYPES:
            raise ValueError(f"Not supported bias: {bias} doesn't belong to (no, pos, align)")
        if BIAS_TYPES[bias] != 0:
            off, sites = bias_arrays(self.ligands)
            self._bias = (off, sites)
            check(lib().ud2_ligset_set_bias(self.h, BIAS_TYPES[bias], float(bias_k), _ptr(off), _ptr(sites)),
                  "ud2_ligset_set_bias")
        if constraint:
            check(lib().ud2_ligset_set_constraint(self.h, 1), "ud2_ligset_set_constraint")

    @property
    def n_lig(self) -> int:
        return len(self.ligands)

    def layout(self, nchain: int):
        xf, df, npz = C.c_int64(), C.c_int64(), C.c_int64()
        check(lib().ud2_ligset_pose_layout(self.h, int(nchain), C.byref(xf), C.byref(df), C.byref(npz)),
              "ud2_ligset_pose_layout")
        return xf.value, df.value, npz.value

    def x_offset(self, lig: int, nchain: int, chain: int) -> int:
        """Float offset of pose (lig, chain) in the x buffer."""
        return (int(self.arrays["atom_off"][lig]) * nchain + chain * self.ligands[lig].natom) * 3

    def dihe_offset(self, lig: int, nchain: int, chain: int) -> int:
        return int(self.arrays["tors_off"][lig]) * nchain + chain * self.ligands[lig].ntors

    def close(self):
        if self.h:
            lib().ud2_ligset_destroy(self.h)
            self.h = C.c_void_p()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def bias_arrays(ligands):
    """CSR of bias sites over the atoms of a ligand batch: offsets [atoms+1] (int32)
    and sites [n, 5] (float32: x, y, z, V, r2)."""
    counts, sites = [], []
    for lig in ligands:
        bs = getattr(lig, "bias_start", None)
        if bs is None:
            counts.append(np.zeros(lig.natom, np.int64))
            continue
        counts.append(np.diff(np.asarray(bs, np.int64)))
        if np.size(lig.bias):
            sites.append(np.asarray(lig.bias, np.float32).reshape(-1, 5))
    off = np.zeros(sum(len(c) for c in counts) + 1, np.int32)
    off[1:] = np.cumsum(np.concatenate(counts))
    sites = np.concatenate(sites) if sites else np.zeros((1, 5), np.float32)
    return off, np.ascontiguousarray(sites, np.float32)


def _require_torch():
    """torch for device buffers and streams; only valid when torch's HIP runtime serves the library."""
    import torch
    if lib() is not None and not _torch_first:
        raise Ud2Error("libud2.so was loaded before torch: import torch first to use torch tensors or streams "
                       "with the library")
    return torch


def stream_ptr(stream=None):
    """hipStream_t of a torch stream (None: torch's current stream)."""
    torch = _require_torch()
    s = torch.cuda.current_stream() if stream is None else stream
    return C.c_void_p(s.cuda_stream)


class PoseBuffers:
    """Device pose buffers (torch tensors) for nchain poses per ligand of a LigSet."""

    def __init__(self, ligset: LigSet, nchain: int, device="cuda"):
        torch = _require_torch()
        self.ligset = ligset
        self.nchain = int(nchain)
        xf, df, npz = ligset.layout(nchain)
        self.n_pose = npz
        f32 = torch.float32
        self.x = torch.zeros(max(xf, 1), dtype=f32, device=device)
        self.c = torch.zeros(max(3 * npz, 1), dtype=f32, device=device)
        self.rv = torch.zeros(max(3 * npz, 1), dtype=f32, device=device)
        self.dihe = torch.zeros(max(df, 1), dtype=f32, device=device)
        self.e = torch.zeros(max(npz, 1), dtype=f32, device=device)
        self.s = Poses(self.x.data_ptr(), self.c.data_ptr(), self.rv.data_ptr(), self.dihe.data_ptr(),
                       self.e.data_ptr(), self.nchain)

    @property
    def ref(self):
        return C.byref(self.s)

    def init(self, stream=None):
        check(lib().ud2_init_poses(self.ligset.h, self.ref, stream_ptr(stream)), "ud2_init_poses")

    def pose(self, lig: int, chain: int) -> dict:
        """Host copy of one pose."""
        L = self.ligset.ligands[lig]
        xo = self.ligset.x_offset(lig, self.nchain, chain)
        do = self.ligset.dihe_offset(lig, self.nchain, chain)
        pid = lig * self.nchain + chain
        return dict(
            x=self.x[xo:xo + 3 * L.natom].cpu().numpy().copy(),
            c=self.c[3 * pid:3 * pid + 3].cpu().numpy().copy(),
            rv=self.rv[3 * pid:3 * pid + 3].cpu().numpy().copy(),
            dihe=self.dihe[do:do + L.ntors].cpu().numpy().copy(),
            e=float(self.e[pid].cpu()),
        )

    def set_pose(self, lig: int, chain: int, x, c, rv, dihe, e=999.0):
        import torch
        L = self.ligset.ligands[lig]
        xo = self.ligset.x_offset(lig, self.nchain, chain)
        do = self.ligset.dihe_offset(lig, self.nchain, chain)
        pid = lig * self.nchain + chain
        dev = self.x.device
        self.x[xo:xo + 3 * L.natom] = torch.as_tensor(np.asarray(x, np.float32).reshape(-1), device=dev)
        self.c[3 * pid:3 * pid + 3] = torch.as_tensor(np.asarray(c, np.float32), device=dev)
        self.rv[3 * pid:3 * pid + 3] = torch.as_tensor(np.asarray(rv, np.float32), device=dev)
        if L.ntors:
            self.dihe[do:do + L.ntors] = torch.as_tensor(np.asarray(dihe, np.float32), device=dev)
        self.e[pid] = float(e)


def run_json(p: dict, text: str, inter_mode: int = MODE_GRID, proposal=None, learned: dict | None = None) -> int:
    """One whole docking run in the library (ud2_create + ud2_run_json): ``p`` holds
    DockingPipeline's keyword arguments (box centre and size included), ``text`` the engine-JSON
    document. ``proposal`` (network parameters) selects the learned search, with the knobs in
    ``learned`` (n_cand, top_k, n_start, sel_temp). Writes <output_dir>/<name_json>_<batch>.json;
    returns the number of batches."""
    rp = RunParams()
    rp.center[:] = [float(p["center_x"]), float(p["center_y"]), float(p["center_z"])]
    rp.size[:] = [float(p["size_x"]), float(p["size_y"]), float(p["size_z"])]
    rp.task, rp.search_mode, rp.bias = (str(p[k]).encode() for k in ("task", "search_mode", "bias"))
    for k in ("exhaustiveness", "mc_steps", "opt_steps", "refine_steps", "num_pose", "gpu_device_id", "max_gpu_mem"):
        setattr(rp, k, int(p[k]))
    for k in ("randomize", "constraint_docking", "use_tor_lib", "energy_decomp"):
        setattr(rp, k, 1 if p[k] else 0)
    rp.rmsd_limit, rp.energy_range, rp.bias_k = float(p["rmsd_limit"]), float(p["energy_range"]), float(p["bias_k"])
    rp.seed = int(p["seed"])
    rp.inter_mode = int(inter_mode)
    if proposal is not None:
        prop = np.ascontiguousarray(proposal, dtype=np.float32).reshape(-1)
        if prop.size != MLP_NPARAM + MLP_NNORM:
            raise ValueError(f"expected {MLP_NPARAM + MLP_NNORM} network parameters, got {prop.size}")
        rp.search, rp.proposal_h = SEARCH_LEARNED, prop.ctypes.data
        for k, v in (learned or {}).items():
            setattr(rp, k, v)
    L = lib()
    h = C.c_void_p()
    check(L.ud2_create(C.byref(rp), C.byref(h)), "ud2_create")
    try:
        raw = text.encode("utf-8")
        n = C.c_int32(0)
        check(L.ud2_run_json(h, raw, len(raw), str(p["output_dir"]).encode(), str(p["name_json"]).encode(),
                             C.byref(n)), "ud2_run_json")
        return n.value
    finally:
        L.ud2_destroy(h)


def dock(scene: Scene, ligset: LigSet, nchain: int, mc_steps: int, opt_steps: int, refine_steps: int = 5,
         num_pose: int = 10, rmsd_limit: float = 1.0, energy_range: float = 10.0, seed: int = 12345,
         randomize: bool = True, mode: int = MODE_GRID, energy_decomp: bool = False, mlp: "Mlp | None" = None,
         n_cand: int = 0, top_k: int = 0, n_start: int = 0, sel_temp: float = 0.0, stream=None) -> dict:
    """One batch of DockTask::run in the library (ud2_dock) over a resident ligand set: the plain
    search, or the learned one when ``mlp`` is given. Host arrays only (numpy). Returns n_out[n_lig],
    chain / energy [n_lig, num_pose(, 7)], coords [atoms * num_pose * 3] and dihedrals
    [torsions * num_pose] in ud2_dock_out's layout (``pose_coords`` picks one pose), decomp when asked,
    the search launches' milliseconds and the search kernels' counters."""
    n_lig = ligset.n_lig
    a = ligset.arrays
    n_atoms, n_tors = int(a["atom_off"][-1]), int(a["tors_off"][-1])
    res = dict(n_out=np.zeros(n_lig, np.int32), chain=np.zeros((n_lig, num_pose), np.int32),
               energy=np.zeros((n_lig, num_pose, 7), np.float32), coords=np.zeros(n_atoms * num_pose * 3, np.float32),
               dihedrals=np.zeros(max(n_tors * num_pose, 1), np.float32),
               decomp=np.zeros(n_atoms * num_pose * 5, np.float32) if energy_decomp else None,
               search_ms=np.zeros(1, np.float32), stats=np.zeros(4, np.uint64), num_pose=num_pose)
    prm = DockParams(nchain=nchain, mc_steps=mc_steps, opt_steps=opt_steps, refine_steps=refine_steps,
                     num_pose=num_pose, rmsd_limit=rmsd_limit, energy_range=energy_range, seed=seed & 0xFFFFFFFF,
                     randomize=int(bool(randomize)), mode=mode, energy_decomp=int(bool(energy_decomp)),
                     search=SEARCH_LEARNED if mlp is not None else SEARCH_PLAIN, n_cand=n_cand, top_k=top_k,
                     n_start=n_start, sel_temp=sel_temp)
    out = DockOut(*[_ptr(res[k]) if res[k] is not None else None for k in (
        "n_out", "chain", "energy", "coords", "dihedrals", "decomp", "search_ms", "stats")])
    check(lib().ud2_dock(scene.h, ligset.h, C.byref(prm), mlp.h if mlp is not None else None, C.byref(out),
                         stream), "ud2_dock")
    return res


TILE_AUTO, TILE_NEVER, TILE_ALWAYS = 0, 1, 2
MC_WHOLE, MC_HALF4, MC_HALF3, MC_HALF2 = 0, 1, 2, 3
MC_VARIANTS = ("whole wave", "half wave, 4 waves/SIMD", "half wave, 3 waves/SIMD", "half wave, 2 waves/SIMD")
TUNE_BUCKETS = 16


def set_tile_policy(policy: int, variant: int = 0) -> None:
    """Which MC kernel runs ligands of up to 32 atoms and 14 torsions: TILE_AUTO (per (natom, ntors)
    bucket, from the tuning table), TILE_NEVER (one chain per wave) or TILE_ALWAYS (two chains per
    wave with the half-wave variant `variant`, 0 = MC_HALF4). Process-wide."""
    check(lib().ud2_set_tile_policy(int(policy), int(variant)), "ud2_set_tile_policy")


def tune_info() -> dict:
    """The tile policy and, per bucket, the chosen variant, the probe times in ms per variant (-1
    unmeasured) and the bucket's natom / ntors ranges (lo, hi, lo, hi)."""
    pol = C.c_int32(0)
    var = np.zeros(TUNE_BUCKETS, np.int32)
    ms = np.zeros((TUNE_BUCKETS, len(MC_VARIANTS)), np.float32)
    rng = np.zeros((TUNE_BUCKETS, 4), np.int32)
    check(lib().ud2_tune_info(C.byref(pol), _ptr(var), _ptr(ms), _ptr(rng)), "ud2_tune_info")
    return {"policy": pol.value, "variant": var, "ms": ms, "range": rng}


def autotune(scene: Scene, ligset: LigSet, opt_steps: int, mc_steps: int = 40, mode: int = MODE_GRID,
             nchain: int = 8, cache_path: str | None = None, seed: int = 12345) -> dict:
    """Times a probe search of the set's small ligands with every MC kernel variant per (natom,
    ntors) bucket and keeps a half-wave variant where it beats whole waves by 2% (ud2_autotune);
    returns tune_info()."""
    prm = McParams(mc_steps=int(mc_steps), opt_steps=int(opt_steps), randomize=1, seed=int(seed), mode=int(mode),
                   lig_index_base=0, stats_d=None)
    path = cache_path.encode() if cache_path else None
    check(lib().ud2_autotune(scene.h, ligset.h, C.byref(prm), int(nchain), path, None), "ud2_autotune")
    return tune_info()


def pose_coords(ligset: LigSet, res: dict, lig: int, k: int) -> np.ndarray:
    """Coordinates [natom * 3] of kept pose k of ligand lig in a ``dock`` result."""
    L = ligset.ligands[lig]
    o = (int(ligset.arrays["atom_off"][lig]) * res["num_pose"] + k * L.natom) * 3
    return res["coords"][o:o + 3 * L.natom]


def device_memory() -> tuple:
    """(free, total) bytes of the current device (ud2_device_memory)."""
    free, total = C.c_int64(), C.c_int64()
    check(lib().ud2_device_memory(C.byref(free), C.byref(total)), "ud2_device_memory")
    return free.value, total.value


def version() -> str:
    return lib().ud2_version().decode()


class Mlp:
    """The learned proposal network on the device (canonical FP32 parameters)."""

    def __init__(self, params):
        p = np.ascontiguousarray(params, dtype=np.float32).reshape(-1)
        if p.size != MLP_NPARAM + MLP_NNORM:
            raise ValueError(f"expected {MLP_NPARAM + MLP_NNORM} parameters, got {p.size}")
        self.h = C.c_void_p()
        check(lib().ud2_mlp_create(_ptr(p), C.byref(self.h)), "ud2_mlp_create")

    def set_params(self, params) -> None:
        p = np.ascontiguousarray(params, dtype=np.float32).reshape(-1)
        check(lib().ud2_mlp_set_params(self.h, _ptr(p)), "ud2_mlp_set_params")

    def params(self) -> np.ndarray:
        out = np.zeros(MLP_NPARAM + MLP_NNORM, dtype=np.float32)
        check(lib().ud2_mlp_get_params(self.h, _ptr(out)), "ud2_mlp_get_params")
        return out

    def close(self):
        if self.h:
            lib().ud2_mlp_destroy(self.h)
            self.h = C.c_void_p()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass
