/*
 * ud2.h: C ABI of the MI355X (gfx950) docking engine library, libud2.so.
 *
 * Plain C types only: host pointers are marked _h, device pointers _d (HIP
 * device memory, e.g. allocated by the caller with hipMalloc or torch). Every
 * function returns UD2_OK (0) or an error code; ud2_last_error() returns the
 * calling thread's message for the last failure. Streams are hipStream_t
 * passed as void* (NULL = default stream). No exception crosses the ABI.
 *
 * Reference citations use E/ = unidock/unidock_engine/ of Uni-Dock2.
 */
#ifndef UD2_H
#define UD2_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define UD2_OK 0
#define UD2_ERR_ARG 1      /* invalid argument or input topology */
#define UD2_ERR_HIP 2      /* a HIP runtime call failed */
#define UD2_ERR_NODEV 3    /* no GPU / device id out of range */
#define UD2_ERR_LIMIT 4    /* input beyond a compiled limit (atoms, torsions, types) */
#define UD2_ERR_STATE 5    /* object in the wrong state (e.g. grid mode without maps) */

#define UD2_MODE_DIRECT 0  /* inter-molecular term as the direct receptor sum (reference semantics) */
#define UD2_MODE_GRID 1    /* inter-molecular term from trilinear grid maps */

#define UD2_MAX_ATOMS 256
#define UD2_MAX_TORSIONS 57

typedef struct ud2_scene ud2_scene;   /* receptor, docking box, grid maps (device) */
typedef struct ud2_ligset ud2_ligset; /* a batch of ligand topologies (device) */
typedef struct ud2_mlp ud2_mlp;       /* the learned proposal's network (device) */

/* Ligand batch in CSR form. Atom, torsion and pair indices inside one ligand
 * are local (0-based within that ligand). Field meaning follows FlexTopo and
 * FlexParamVina (E/src/model/model.h:95-108, E/src/score/vina.h:17-25). */
typedef struct {
    int32_t n_lig;
    const int32_t* atom_off_h;   /* [n_lig+1] */
    const int32_t* tors_off_h;   /* [n_lig+1] */
    const int32_t* pair_off_h;   /* [n_lig+1] */
    const int32_t* types_h;      /* [atoms] XS type (E/src/constants/constants.h:48-68) */
    const float* xyz_h;          /* [atoms*3] input conformation */
    const int32_t* axis_h;       /* [tors*2] (from, to) */
    const float* dihe0_h;        /* [tors] input dihedrals, radians */
    const int32_t* rot_off_h;    /* [tors+1] CSR into rot_atoms_h */
    const int32_t* rot_atoms_h;  /* atoms rotated by each torsion, its "to" atom included */
    const int32_t* range_off_h;  /* [tors+1] CSR into ranges_h, in (lo, hi) pairs */
    const float* ranges_h;       /* allowed dihedral intervals (lo, hi), radians */
    const int32_t* pairs_h;      /* [pairs*2] intra-molecular pairs (i, j) */
} ud2_ligand_batch;

/* Pose buffers for nchain poses per ligand of a ligand set (device memory).
 * Layout (atom_off / tors_off are the batch's CSR offsets):
 *   x    [(atom_off[l]*nchain + c*natom_l)*3 + 3*a + k]
 *   dihe [tors_off[l]*nchain + c*ntors_l + t]
 *   c, rv [(l*nchain + c)*3 + k]   centre, rotation vector of the last rotation increment
 *   e    [l*nchain + c]            energy
 * Pose id of (ligand l, chain c) = l*nchain + c. */
typedef struct {
    float* x_d;
    float* c_d;
    float* rv_d;
    float* dihe_d;
    float* e_d;
    int32_t nchain;
} ud2_poses;

typedef struct {
    int32_t mc_steps;        /* DockParam::mc_steps (E/src/model/model.h:156) */
    int32_t opt_steps;       /* BFGS iterations per MC step; 0 = no local optimisation */
    int32_t randomize;       /* randomise the input pose first (E/src/cuda/mc.cu:109-134) */
    uint32_t seed;           /* key of each chain's Philox stream, with the ligand index */
    int32_t mode;            /* UD2_MODE_DIRECT or UD2_MODE_GRID */
    int32_t lig_index_base;  /* added to the ligand index in the random-stream key */
    uint64_t* stats_d;       /* optional device counters, accumulated: [0] energy evaluations,
                                [1] grid-gather bytes (evals * 32 * heavy atoms), [2] intra-pair
                                evaluations, [3] chains done */
} ud2_mc_params;

/* ------------------------------------------------------------- library */
const char* ud2_version(void);
const char* ud2_last_error(void);
int ud2_device_count(int32_t* n_h);
int ud2_set_device(int32_t device_id);  /* cudaSetDevice in decide_memory_limit_mb, E/src/screening/core.cpp:39 */
int ud2_synchronize(void);
/* Free and total bytes of the current device (cudaMemGetInfo in decide_memory_limit_mb,
 * E/src/screening/core.cpp:32-63). */
int ud2_device_memory(int64_t* free_h, int64_t* total_h);

/* ------------------------------------------------------------- receptor
 * Replaces the receptor half of DockTask::alloc_gpu (E/src/cuda/task.cu:304-402):
 * heavy receptor atoms (hydrogens are dropped here, as the reference's parser
 * does, E/src/format/rapidjson_parser.cpp:34) and the docking box. */
int ud2_scene_create(const float* rec_xyz_h, const int32_t* rec_types_h, int32_t n_rec, const float box_lo_h[3],
                     const float box_hi_h[3], ud2_scene** out);
/* Grid maps over the box (no reference counterpart): map_t(p) = sum over heavy
 * receptor atoms within 8 A of the uncurled pair energy Vina::eval_ef
 * (E/src/score/vina.h:216-245) of a probe of type t. Points at box_lo +
 * spacing*(i, j, k), n = round(size/spacing) + 1 per axis. */
int ud2_scene_build_grids(ud2_scene* sc, float spacing, const int32_t* probe_types_h, int32_t n_types);
/* Prebuilt maps, [n_types][nz][ny][nx] at origin + spacing*(i, j, k). */
int ud2_scene_set_grids(ud2_scene* sc, const int32_t n_h[3], const float origin_h[3], float spacing,
                        const int32_t* probe_types_h, int32_t n_types, const float* maps_h);
int ud2_scene_grid_info(const ud2_scene* sc, int32_t n_h[3], float origin_h[3], float* spacing_h, int32_t* n_types_h);
int ud2_scene_download_maps(const ud2_scene* sc, float* maps_h);
/* Random-gather probe (no reference counterpart; a measurement aid): ceil(n_gathers / 16)
 * threads each read 16 cells of the cell-major map copy the search kernels gather from (two
 * float4, one 32-byte sector per cell), drawn by a hash of (thread, seed) from the first
 * span_cells cells (<= 0: all of them, 8 maps x 80^3 cells = 131 MB for the default grids),
 * and write the sum of what they read to out_d[thread]. Its achieved bandwidth is the ceiling
 * for scattered map gathers over that footprint. */
int ud2_scene_gather_probe(const ud2_scene* sc, int64_t n_gathers, int64_t span_cells, uint32_t seed, float* out_d,
                           void* stream);
/* VALU probe (no reference counterpart; a measurement aid): n_threads threads each run 8 independent
 * FP32 FMA chains of iters steps (8 * iters unpacked v_fma_f32 per thread) and write their sum to
 * out_d[thread]. Its instruction rate is the ceiling for the search kernels' plain FP32 VALU work. */
int ud2_valu_probe(int64_t n_threads, int32_t iters, float* out_d, void* stream);
/* Device memory of the scene's reach lists (no reference counterpart): per cell of the space around the
 * box the receptor atoms that a point in it can have within the cutoff, built with the scene. The
 * direct sums (direct mode, final score, decomposition) read them, and without them go over the whole
 * receptor, with the same results. *bytes_h (optional) = their bytes, 0 without; keep 0 frees them (no
 * call on the scene may run meanwhile). */
int ud2_scene_reach(ud2_scene* sc, int32_t keep, int64_t* bytes_h);
int ud2_scene_destroy(ud2_scene* sc);

/* ------------------------------------------------------------- ligands
 * Replaces the ligand half of DockTask::alloc_gpu (E/src/cuda/task.cu:16-284). */
int ud2_ligset_create(const ud2_ligand_batch* batch, ud2_ligset** out);
int ud2_ligset_destroy(ud2_ligset* ls);

/* Bias sites and the bias option of the task: apply_bias (E/src/screening/core.cpp:86-97)
 * plus the bias half of DockTask's ligand upload (FlexParamVina::inds_bias /
 * params_bias, E/src/cuda/task.cu:157-168) and the BIAS_TYPE / BIAS_K constants
 * (E/src/cuda/common.cu:25-26). bias_off_h [atoms+1] is a CSR over the set's
 * atoms (atom_off order) into bias_h, 5 floats per site as in the input JSON
 * (E/src/format/rapidjson_parser.cpp:114-124): x, y, z, V, r2. pos adds
 * V k exp(-|site - atom|^2 / r2) per site (Vina::eval_ef_pos, E/src/score/vina.h:277-289);
 * align adds the Z-align attraction with affinity V k (Vina::eval_ef_zalign,
 * vina.h:306-324). The bias enters every search energy, uncurled, and is reported
 * separately by ud2_final_score. NULL bias_off_h clears the sites. */
#define UD2_BIAS_NO 0
#define UD2_BIAS_POS 1
#define UD2_BIAS_ALIGN 2
int ud2_ligset_set_bias(ud2_ligset* ls, int32_t bias_type, float bias_k, const int32_t* bias_off_h,
                        const float* bias_h);
/* Constraint docking (DockParam::constraint_docking, FLAG_CONSTRAINT_DOCK of
 * E/src/cuda/common.cu:27): the centre and orientation stay fixed in every
 * search entry point, mutations draw torsions only (E/src/cuda/mc.cu:159-166),
 * randomisation keeps the rigid pose (mc.cu:27-35), the rigid gradient
 * components are zero (E/src/cuda/bfgs.cuh:176) and the pose update has no
 * rigid step (bfgs.cuh:571). */
int ud2_ligset_set_constraint(ud2_ligset* ls, int32_t constraint);
/* Sizes of the pose buffers (floats) for nchain poses per ligand. */
int ud2_ligset_pose_layout(const ud2_ligset* ls, int32_t nchain, int64_t* x_floats_h, int64_t* dihe_floats_h,
                           int64_t* n_pose_h);
/* Every pose set to the input conformation: centre = centroid, rot_vec = 0,
 * energy 999 (E/src/cuda/task.cu:94-108). */
int ud2_init_poses(const ud2_ligset* ls, const ud2_poses* P, void* stream);

/* ------------------------------------------------------------- hot path
 * E + gradient of pose vectors [centre(3), quaternion w,x,y,z (4), torsions]
 * of ligand `lig`: the torsions are set on its input conformation in index
 * order, the conformer is rotated by q about its centroid and moved to the
 * centre, rot_vec = rotvec(q). Batched form of cal_e_grad_one_gpu
 * (E/src/cuda/bfgs_wrapper.cu:63-98). e_d[n], g_d[n][6+ntors]. */
int ud2_score_posevecs(const ud2_scene* sc, const ud2_ligset* ls, int32_t lig, int64_t n, const float* pv_d,
                       float* e_d, float* g_d, int32_t mode, float v_cap, float slope, void* stream);
/* E + gradient (cal_e_grad_tile, E/src/cuda/bfgs.cuh:397-410) of the selected
 * poses (pose ids sel_d[n_sel]); g_d is [n_sel][64], components 0..5+ntors. */
int ud2_energy_grad(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d,
                    int32_t n_sel, int32_t mode, float v_cap, float slope, float* e_d, float* g_d, void* stream);
/* One pose update x <- x (+) alpha * dir (apply_grad_update_pose_tile,
 * E/src/cuda/bfgs.cuh:560-618); dir_d is [n_sel][64]. */
int ud2_pose_update(const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d, int32_t n_sel,
                    const float* dir_d, float alpha, void* stream);
/* One backtracking line search from H = I (line_search_one_gpu,
 * E/src/cuda/bfgs_wrapper.cu:104-159), in place; alpha_d[n_sel], g_d[n_sel][64]. */
int ud2_line_search(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d,
                    int32_t n_sel, int32_t mode, float v_cap, float slope, float* alpha_d, float* g_d, void* stream);
/* In-place BFGS of the selected poses (optimize_cu, E/src/cuda/optimize.cu:197-212). */
int ud2_optimize(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d,
                 int32_t n_sel, int32_t mode, int32_t max_steps, float v_cap, float slope, float* e_d, void* stream);
/* Monte Carlo search, nchain chains per ligand, best pose per chain written to
 * P (mc_cu, E/src/cuda/mc.cu:408-448). One persistent launch per atoms-per-lane
 * class over a size-sorted work queue. */
int ud2_mc(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const ud2_mc_params* params,
           void* stream);
/* ud2_mc without allocation (no reference counterpart): for callers that cannot allocate device
 * memory (HIP graph capture, tight serving loops). The same kernels, launches and results as ud2_mc;
 * the work-queue heads of the persistent launches live in a static device array of the library
 * (64 int32 per GPU, of which one per launch, at most 7, is used) instead of the ligand set's
 * memory. No hipMalloc / hipFree, no host copy, no synchronisation. Every call on one GPU shares
 * that GPU's array: calls that overlap on one GPU (other streams or host threads) race. */
int ud2_mc_noalloc(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const ud2_mc_params* params,
                   void* stream);
/* Two chains per wave (no reference counterpart; the reference runs one chain per fixed-size
 * thread tile). ud2_mc runs a ligand of at most 32 atoms and 14 torsions with one of four kernel
 * variants, all with the same results bit for bit: one chain per 64-lane wave
 * (UD2_MC_WHOLE), or two chains of the ligand per wave, one per 32-lane half, with the register
 * allocation held to 4, 3 or 2 waves per SIMD (UD2_MC_HALF4 / 3 / 2). The variant is chosen per
 * (natom, ntors) bucket: natom 1-8, 9-16, 17-24, 25-32 by ntors 0-3, 4-7, 8-11, 12-14
 * (bucket = natom index * 4 + ntors index). Larger ligands, and every ligand in direct mode, run one
 * chain per wave whatever is chosen; a search of few chains runs each chain on four waves, unless
 * UD2_TILE_ALWAYS asks for a half-wave variant. The choice is process-wide and applies to the
 * searches launched after it is set; a ligand set's first search after a change copies its new work
 * split to the device and synchronises. */
#define UD2_MC_WHOLE 0
#define UD2_MC_HALF4 1
#define UD2_MC_HALF3 2
#define UD2_MC_HALF2 3
#define UD2_MC_VARIANTS 4
#define UD2_TUNE_BUCKETS 16
#define UD2_TILE_AUTO 0    /* per bucket, from the table (UD2_MC_WHOLE everywhere until tuned) */
#define UD2_TILE_NEVER 1   /* UD2_MC_WHOLE for every ligand */
#define UD2_TILE_ALWAYS 2  /* the half-wave variant `variant` (0: UD2_MC_HALF4) for every ligand that fits (grid mode) */
int ud2_set_tile_policy(int32_t policy, int32_t variant);
/* The policy, and per bucket the variant (variant_h), the probe times in ms per variant
 * (ms_h[b][v]; -1 unmeasured) and the bucket's ranges natom lo, hi, ntors lo, hi (range_h[b][4]);
 * arrays of UD2_TUNE_BUCKETS rows, any pointer may be null. */
int ud2_tune_info(int32_t* policy_h, int32_t* variant_h, float* ms_h, int32_t* range_h);
/* Autotuner: for every bucket that the ligand set's ligands fall in, times a probe search of those
 * ligands with each variant (params' mode, mc_steps and opt_steps, nchain chains each (0: 8), the
 * ligands repeated to fill the GPU twice over) and keeps a half-wave variant in the table only
 * where it is at least 2% faster than whole waves. With cache_path, buckets found in that file for
 * this GPU model, CU count, mode and version of the search kernels are taken from it instead, and
 * the file is rewritten with every bucket known. Allocates its probe buffers; synchronises the stream. */
int ud2_autotune(const ud2_scene* sc, const ud2_ligset* ls, const ud2_mc_params* params, int32_t nchain,
                 const char* cache_path, void* stream);
/* Greedy leader clustering per ligand by heavy-atom RMSD (cluster_cu,
 * E/src/cuda/cluster.cu:74-135): leaders_d[n_lig][nchain] in selection order
 * (chain indices), nleaders_d[n_lig]. */
int ud2_cluster(const ud2_ligset* ls, const ud2_poses* P, float rmsd_limit, int32_t* leaders_d,
                int32_t* nleaders_d, void* stream);
/* Final re-score (score(), E/src/score/score.cpp:12-108): out4_d[n_sel][4] =
 * intra (pairs once, no curl), inter (direct sum, no curl), box penalty, bias. */
int ud2_final_score(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d,
                    int32_t n_sel, float* out4_d, void* stream);
/* Energy decomposition (score_decomp, E/src/score/score.cpp:115-147): the
 * inter-molecular direct sum of each selected pose split per ligand atom into
 * its weighted Vina terms, decomp_d[n_sel][atom_stride][5] = gauss1, gauss2,
 * repulsion, hydrophobic, hbond (zero for hydrogens); atom_stride >= the
 * largest natom among the selected poses. */
int ud2_score_decomp(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d,
                     int32_t n_sel, int32_t atom_stride, float* decomp_d, void* stream);

/* ------------------------------------------------------------- one batch, device-resident
 * DockTask::run (E/src/task/DockTask.cpp:39-123) over a ligand set already on the device: the
 * search (ud2_mc, or ud2_lmc for the learned search), clustering (ud2_cluster), refinement with the
 * penalty-slope ramp (run_refine, DockTask.cpp:155-186: refine_steps rounds of 2 BFGS iterations
 * at cap 1000, slope 100 * 10^(2p) capped at 1e6), filtering by energy_range and num_pose
 * (run_filter, DockTask.cpp:188-220), the final score and the affinity (run_score,
 * DockTask.cpp:224-282). Pose buffers and selections are allocated by the library for the call
 * and freed before it returns; the results land in caller-owned host arrays; the call returns
 * when they are written. ud2_run_json docks each of its batches with this call. */
#define UD2_SEARCH_PLAIN 0    /* the reference's Monte Carlo search (ud2_mc) */
#define UD2_SEARCH_LEARNED 1  /* the learned-proposal search (ud2_lmc, UD2_POLICY_LEARNED); needs a network */

typedef struct {
    int32_t nchain;           /* MC chains per ligand (exhaustiveness) */
    int32_t mc_steps;
    int32_t opt_steps;        /* BFGS iterations per MC step (>= 0) */
    int32_t refine_steps;
    int32_t num_pose;         /* poses kept per ligand, >= 1 */
    float rmsd_limit;
    float energy_range;
    uint32_t seed;
    int32_t randomize;
    int32_t mode;             /* UD2_MODE_GRID or UD2_MODE_DIRECT for the search and refinement */
    int32_t energy_decomp;    /* also write decomp_h */
    int32_t search;           /* UD2_SEARCH_PLAIN or UD2_SEARCH_LEARNED */
    int32_t n_cand, top_k, n_start;  /* learned search: as ud2_lmc_params (0: 8, 1, 6) */
    float sel_temp;           /* learned search: > 0 sampling temperature as ud2_lmc_params; 0: 1.0;
                                 < 0: the network's top_k rescored exactly instead of sampling */
} ud2_dock_params;

/* Results of ud2_dock, caller-owned host arrays sized for num_pose poses per ligand. Pose k
 * (k < n_out_h[l]) of ligand l, with atom_off / tors_off the set's CSR offsets: */
typedef struct {
    int32_t* n_out_h;      /* [n_lig] poses kept (0 .. num_pose), in ascending search energy */
    int32_t* chain_h;      /* [n_lig * num_pose] MC chain of each pose (optional) */
    float* energy_h;       /* [(l * num_pose + k) * 7]: affinity, total, intra, inter, penalty,
                              conf-independent, bias (E/src/task/DockTask.cpp:248-276) */
    float* coords_h;       /* [(atom_off[l] * num_pose + k * natom_l) * 3 + 3 a + d] */
    float* dihedrals_h;    /* [tors_off[l] * num_pose + k * ntors_l + t], radians (optional) */
    float* decomp_h;       /* [(atom_off[l] * num_pose + k * natom_l) * 5 + q] (energy_decomp only) */
    float* search_ms_h;    /* optional: milliseconds of the search launches, HIP events on the stream */
    uint64_t* stats_h;     /* optional [4]: the search kernels' counters, as ud2_mc_params::stats_d */
} ud2_dock_out;

/* Atom and torsion counts of the set's ligands (natom_h / ntors_h [n_lig], each optional). */
int ud2_ligset_sizes(const ud2_ligset* ls, int32_t* n_lig_h, int32_t* natom_h, int32_t* ntors_h);
int ud2_dock(const ud2_scene* sc, const ud2_ligset* ls, const ud2_dock_params* params, const ud2_mlp* mlp,
             const ud2_dock_out* out, void* stream);

/* ------------------------------------------------------------- whole docking run
 * The reference's core_pipeline (E/src/screening/core.cpp:100-223) behind a
 * handle: ud2_create takes the run options of CoreInput (E/src/screening/core.h:70-100;
 * the keyword arguments of DockingPipeline, E/api/python/pipeline.cpp:167-189),
 * ud2_run_json parses an engine-JSON document (receptor under "receptor", one
 * member per ligand, optional "score"; E/src/format/json.cpp:34-76 and
 * E/src/format/rapidjson_parser.cpp:25-296), applies the search-mode and task
 * presets, docks the ligands in size groups and batches of at most 1,000 within
 * the device-memory budget (E/src/screening/screening.cpp:140-219,
 * E/src/screening/core.cpp:32-63) and writes
 * <out_dir>/<name_json>_<batch>.json (out_dir "" = working directory) in the
 * reference's output format (E/src/format/json.cpp:88-191). *n_files_h (optional)
 * = batches written. Host memory only crosses the ABI; the device work runs on
 * the device gpu_device_id on the default stream. One run per handle at a time. */
typedef struct ud2_handle ud2_handle;

typedef struct {
    float center[3], size[3];   /* docking box: lo = center - size/2, hi = center + size/2 */
    const char* task;           /* screen | score | mc | randomize | optimize (NULL = screen) */
    const char* search_mode;    /* fast | balance | detail | free (NULL = balance) */
    int32_t exhaustiveness;     /* MC chains per ligand */
    int32_t randomize;
    int32_t mc_steps;
    int32_t opt_steps;          /* < 0: (25 + natom_max of the first batch) / 3 */
    int32_t refine_steps;
    int32_t num_pose;
    float rmsd_limit;
    float energy_range;
    int64_t seed;               /* its low 32 bits key the random streams */
    const char* bias;           /* no | pos | align (NULL = no) */
    float bias_k;
    int32_t constraint_docking;
    int32_t use_tor_lib;
    int32_t energy_decomp;
    int32_t gpu_device_id;
    int32_t max_gpu_mem;        /* MB (<= 0: none): with 95 % of the free device memory and of the host's
                                   memory, the budget that bounds each batch's estimated device memory */
    int32_t inter_mode;         /* UD2_MODE_GRID or UD2_MODE_DIRECT for the search and refinement */
    /* Search method (no CoreInput counterpart): UD2_SEARCH_PLAIN, or UD2_SEARCH_LEARNED with the
     * network's parameters proposal_h[UD2_MLP_NPARAM + UD2_MLP_NNORM] (copied by ud2_create) and
     * the knobs of ud2_dock_params (0 / negative: defaults). Zero-initialised = the plain search. */
    int32_t search;
    const float* proposal_h;
    int32_t n_cand, top_k, n_start;
    float sel_temp;
} ud2_run_params;

/* DockingPipeline's constructor / CoreInput set-up (E/api/python/pipeline.cpp:56-100). */
int ud2_create(const ud2_run_params* params, ud2_handle** out);
/* core_pipeline over a JSON text (E/src/screening/core.cpp:100-223; the pybind
 * run() serialises its objects to this text, E/api/python/pipeline.cpp:120-145). */
int ud2_run_json(ud2_handle* h, const char* json, size_t len, const char* out_dir, const char* name_json,
                 int32_t* n_files_h);
int ud2_destroy(ud2_handle* h);

/* ------------------------------------------------------------- learned proposal
 * No reference counterpart: the reference's MC tries one random mutation per
 * step (E/src/cuda/mc.cu:146-256). The learned search draws n_cand mutations
 * per step, scores them with a small network on the GPU (BF16 MFMA, FP32
 * accumulation), rescores the top_k with the exact search energy and refines
 * the best with BFGS; the Metropolis test and the best-pose bookkeeping are
 * the reference's (mc.cu:340-392). Every kept pose is exact Vina.
 *
 * Network: 80 inputs per candidate (pooled per-atom grid-map statistics by
 * feature class, and move globals), two ReLU layers of 256, one output. The
 * parameters are FP32 in the canonical order W1[80][256], b1[256],
 * W2[256][256], b2[256], w3[256], b3, followed by the fixed input
 * normalisation mu[80], inv_sigma[80]. Inputs are bf16 bit patterns,
 * [rows][80], rows in groups of 16 candidates of one MC state. */
#define UD2_MLP_FEATURES 80
#define UD2_MLP_HIDDEN 256
#define UD2_MLP_GROUP 16
#define UD2_MLP_NPARAM 86785
#define UD2_MLP_NNORM 160

#define UD2_POLICY_PLAIN 0    /* one random mutation per step, no network (the reference's step) */
#define UD2_POLICY_EXACT 1    /* n_cand mutations, all scored with the exact energy, no network */
#define UD2_POLICY_LEARNED 2  /* n_cand mutations, the network's top_k scored exactly */
#define UD2_POLICY_COLLECT 3  /* n_cand mutations, all BFGS-refined: features and labels for training */

typedef struct {
    float lr, beta1, beta2, eps;
} ud2_adam;

typedef struct {
    ud2_mc_params mc;     /* as for ud2_mc; mc_steps >= 1 */
    int32_t policy;       /* UD2_POLICY_* */
    int32_t n_cand;       /* mutations per step, 1..16 (ignored by the plain policy) */
    int32_t top_k;        /* learned policy: candidates rescored exactly, 1..n_cand */
    float sel_temp;       /* learned policy: > 0 instead draws one candidate with p ~ exp(-score / sel_temp) */
    int32_t n_start;      /* > 1: randomised starts drawn per chain (orientations spread over n_start * nchain);
                             the chain starts from the best by the network (learned) or the exact energy */
    uint16_t* collect_x_d;  /* collect: [mc_steps][n_pose][16][80] features (bf16) */
    float* collect_y_d;     /* collect: [mc_steps][n_pose][16] energies after BFGS */
    float* collect_e0_d;    /* collect, optional: [mc_steps][n_pose][16] energies before BFGS */
} ud2_lmc_params;

/* Network on the current device from params_h[UD2_MLP_NPARAM + UD2_MLP_NNORM]. */
int ud2_mlp_create(const float* params_h, ud2_mlp** out);
int ud2_mlp_set_params(ud2_mlp* m, const float* params_h);  /* also resets the Adam state */
int ud2_mlp_get_params(const ud2_mlp* m, float* params_h);
int ud2_mlp_destroy(ud2_mlp* m);
/* y_d[16 n_groups]: scores of the rows of groups groups_d[i] (NULL: 0..n_groups-1) of x_d. */
int ud2_mlp_forward(const ud2_mlp* m, const uint16_t* x_d, const int32_t* groups_d, int32_t n_groups, float* y_d,
                    void* stream);
/* grad_d[UD2_MLP_NPARAM] = gradient of sum_r dy_d[r] * y[r] over the same rows. */
int ud2_mlp_backward(ud2_mlp* m, const uint16_t* x_d, const int32_t* groups_d, int32_t n_groups, const float* dy_d,
                     float* grad_d, void* stream);
/* One Adam step on the minibatch of groups groups_d: group-centred squared
 * error against labels clipped at (group minimum + 6); loss_d (optional, device) = the loss. */
int ud2_mlp_train_step(ud2_mlp* m, const uint16_t* x_d, const float* label_d, const int32_t* groups_d,
                       int32_t n_groups, const ud2_adam* opt, float* loss_d, void* stream);
/* Network inputs of the selected poses (as if reached by no move from an
 * accepted energy of 0); needs grid maps for every ligand atom type. */
int ud2_features(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d, int32_t n_sel,
                 uint16_t* x_d, void* stream);
/* Learned-proposal Monte Carlo search; best pose per chain written to P as
 * ud2_mc does (one persistent launch per atoms-per-lane class over a
 * size-sorted work queue). mlp may be NULL except for the learned policy. */
int ud2_lmc(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const ud2_lmc_params* params,
            const ud2_mlp* mlp, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* UD2_H */
